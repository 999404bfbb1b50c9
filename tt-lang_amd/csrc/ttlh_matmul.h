// Register-direct GEMM kernels (matmul_direct.hip), chosen and launched for
// the entry points in matmul.hip.
#pragma once

#include "ttlh_common.h"

namespace ttlh {

struct DirectArgs {
  const void* A;  // bf16 or f32, row-major
  const void* B;  // bf16 or f32 row-major [K, N], or the packed block-float tiles
  void* C;
  int64_t lda, ldb, ldc;
  int32_t M, N, K;
  int32_t c_dtype, accumulate, c_vec;  // c_vec: four results are one aligned store
  int32_t grid_m, grid_n;
  int32_t splits;    // workgroups per output block, each a part of K
  float* partial;    // splits > 1: fp32 blocks of the parts
  int32_t* arrived;  // ... and a counter per output block, 0 between launches
};

// Each launches the product (M, N, K multiples of 32) and returns true with
// the launch's status in *status, or returns false, having launched nothing,
// where the caller's other kernels take the problem.  `scratch`: null, or
// TTLH_MATMUL_SCRATCH_BYTES of device memory (see ttlh_matmul_scratch).
// other_us: the modelled time of the caller's best kernel.
bool launch_direct_bf16(DirectArgs a, double other_us, void* scratch, hipStream_t s, int* status);
bool launch_direct_f32(DirectArgs a, void* scratch, hipStream_t s, int* status);
bool launch_direct_block(DirectArgs a, int bits, void* scratch, hipStream_t s, int* status);
// false: none of them divides K in a product of these sizes
bool may_divide_k(int a_dtype, int b_dtype, int64_t M, int64_t N, int64_t K);

}  // namespace ttlh
