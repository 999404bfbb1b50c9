// GEMM kernels that read their operands from global memory straight into the
// MFMA registers, without LDS staging, for the problems that the 256x256 LDS
// kernels (matmul.hip) leave most of the chip idle on: few rows of A (decode
// steps, small batches), outputs of few tiles, block-float weights, and fp32.
//
// A workgroup owns one BM x BN output block and its WK waves split K between
// them (wave w takes k stages w, w + WK, ...), so that a small output still
// puts WK waves per block on the chip, each with its own loads in flight and
// no barrier in the loop.  At the end the waves' partial blocks meet in LDS
// and are summed in wave order: results repeat exactly.
#include <algorithm>

#include "ttlh_common.h"
#include "ttlh_matmul.h"

namespace ttlh {
namespace {

// Scratch: the arrival counters of at most 256 output blocks, then their parts
// (at most 256 workgroups' blocks of 32 x 128).
constexpr int kArrivedBytes = 1024;
static_assert(TTLH_MATMUL_SCRATCH_BYTES >= kArrivedBytes + 256 * 32 * 128 * 4, "scratch size");

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4a8 __attribute__((aligned(8)));  // packed tiles may be 8-byte aligned

template <int N>
struct WordVec;
template <>
struct WordVec<2> { typedef u32x2 type; };
template <>
struct WordVec<4> { typedef u32x4 type; };

// A uniform base plus a 32-bit byte offset of the lane (one load instruction,
// no 64-bit vector address arithmetic).
template <typename T>
__device__ __forceinline__ T gload(const void* base, uint32_t off) {
  typedef const __attribute__((address_space(1))) T gT;
  typedef const __attribute__((address_space(1))) char gchar;
  return *reinterpret_cast<gT*>(reinterpret_cast<gchar*>(reinterpret_cast<uintptr_t>(base)) + off);
}

// A copy of a lane's byte offset that the compiler cannot widen to 64 bits
// outside the loop (it would then add it with vector instructions instead of
// using the load's scalar base).
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Output block of this workgroup.  Workgroup i runs on XCD i % 8: each XCD
// takes a contiguous run of the block order, in which the row blocks of one
// column of blocks follow each other (they share B through that XCD's L2).
__device__ __forceinline__ void direct_block(const DirectArgs& p, int& bm, int& bn, int& split) {
  const int n = gridDim.x, id = blockIdx.x;
  const int per = n >> 3, rem = n & 7, x = id & 7;
  const int i = x * per + min(x, rem) + (id >> 3);
  const int j = i / p.grid_m;
  bm = i - j * p.grid_m;
  split = j / p.grid_n;
  bn = j - split * p.grid_n;
}

// Four consecutive results of one row.  vec: the row pitch and the base allow
// one store of all four.
__device__ __forceinline__ void store4(const DirectArgs& p, int row, int col, f32x4 v) {
  const int64_t off = static_cast<int64_t>(row) * p.ldc + col;
  if (p.c_dtype == TTLH_BF16) {
    uint16_t* c = static_cast<uint16_t*>(p.C) + off;
    if (p.accumulate) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += bf16_to_f32(c[i]);
    }
    const u32x2 w = {cvt_pk_bf16x2(v[0], v[1]), cvt_pk_bf16x2(v[2], v[3])};
    if (p.c_vec) {
      *reinterpret_cast<u32x2*>(c) = w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = static_cast<uint16_t>(w[i >> 1] >> (16 * (i & 1)));
    }
  } else {
    float* c = static_cast<float*>(p.C) + off;
    if (p.accumulate) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += c[i];
    }
    if (p.c_vec) {
      *reinterpret_cast<f32x4*>(c) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = v[i];
    }
  }
}

// Four values of a part, to and from memory past the caches that other
// workgroups' XCDs do not see: relaxed device-scope atomics, which write
// through and read at the device's coherence point.
__device__ __forceinline__ void put_part(float* d, f32x4 v) {
  typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
  const u64x2 w = __builtin_bit_cast(u64x2, v);
  unsigned long long* q = reinterpret_cast<unsigned long long*>(d);
  __hip_atomic_store(q, w[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(q + 1, w[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x4 get_part(const float* d) {
  typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
  const unsigned long long* q = reinterpret_cast<const unsigned long long*>(d);
  const u64x2 w = {__hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                   __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
  return __builtin_bit_cast(f32x4, w);
}

// Chunk c (four results of a row) of the sum over the waves' blocks in LDS (rows
// at a pitch of PITCH floats), in wave order.
template <int BM, int BN, int PITCH, int WK>
__device__ __forceinline__ f32x4 wave_sum(const float* part, int c) {
  const float* q = part + c / (BN / 4) * PITCH + (c % (BN / 4)) * 4;
  f32x4 s = *reinterpret_cast<const f32x4*>(q);
#pragma unroll
  for (int w = 1; w < WK; ++w) s += *reinterpret_cast<const f32x4*>(q + w * BM * PITCH);
  return s;
}

// The block's result: of each of the p.splits parts of K, part_of(split) leaves
// the waves' blocks in LDS, behind a barrier; their sums are added in split order.
// WHOLE: this workgroup takes all parts, one after the other (where there is no
// scratch to meet in); the results are the same bits.
template <int BM, int BN, int PITCH, int WK, int THREADS, bool WHOLE, typename F>
__device__ __forceinline__ void reduce_store(const DirectArgs& p, const float* part, int bm, int bn,
                                             int split, F part_of) {
  constexpr int kChunks = BM * BN / 4;
  const int m0 = bm * BM, n0 = bn * BN;
  const auto store = [&](int c, f32x4 v) {
    const int row = m0 + c / (BN / 4), col = n0 + (c % (BN / 4)) * 4;
    if (row < p.M && col < p.N) store4(p, row, col, v);
  };
  if constexpr (WHOLE) {
    constexpr int kPer = (kChunks + THREADS - 1) / THREADS;
    const int t = threadIdx.x;
    f32x4 sum[kPer];
    for (int s = 0; s < p.splits; ++s) {
      part_of(s);
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        if (t + i * THREADS < kChunks) {
          const f32x4 v = wave_sum<BM, BN, PITCH, WK>(part, t + i * THREADS);
          sum[i] = s == 0 ? v : sum[i] + v;
        }
      __syncthreads();  // the next part writes over these
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      if (t + i * THREADS < kChunks) store(t + i * THREADS, sum[i]);
    return;
  }
  part_of(split);
  const int block = bn * p.grid_m + bm;
  float* mine = p.partial + static_cast<int64_t>(block * p.splits + split) * (BM * BN);
  for (int c = threadIdx.x; c < kChunks; c += THREADS) {
    const f32x4 s = wave_sum<BM, BN, PITCH, WK>(part, c);
    if (p.splits > 1)
      put_part(mine + 4 * c, s);
    else
      store(c, s);
  }
  if (p.splits == 1) return;
  // The workgroup that arrives last at this block's counter adds the parts,
  // in split order; nobody waits for anybody.  That the parts come before the
  // counter is an assumption about the hardware, not a rule of the memory model:
  // both are relaxed device-scope accesses, and a wave counts in only after
  // vmcnt(0) and a barrier.  A device-scope store is written through, and its
  // acknowledgement is taken to mean that it has reached the device's coherence
  // point, where the last workgroup's loads read.  A release fence would say the
  // same in the model's terms, by writing back the whole L2 (measured: 20 us a
  // launch).
  __shared__ int last;
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  if (threadIdx.x == 0) {
    last = __hip_atomic_fetch_add(p.arrived + block, 1, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT) == p.splits - 1;
    if (last) __hip_atomic_store(p.arrived + block, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last) return;
  const float* parts = p.partial + static_cast<int64_t>(block) * p.splits * (BM * BN);
  for (int c = threadIdx.x; c < kChunks; c += THREADS) {
    f32x4 s = get_part(parts + 4 * c);
    for (int w = 1; w < p.splits; ++w)
      s += get_part(parts + static_cast<int64_t>(w) * (BM * BN) + 4 * c);
    store(c, s);
  }
}

__device__ __forceinline__ uint32_t perm_lo(uint32_t x, uint32_t y) {
  return __builtin_amdgcn_perm(y, x, 0x05040100u);  // lo16(x) | lo16(y) << 16
}
__device__ __forceinline__ uint32_t perm_hi(uint32_t x, uint32_t y) {
  return __builtin_amdgcn_perm(y, x, 0x07060302u);
}

// ---------------------------------------------------------------------------
// bf16 A and B.  Block of 16 MT rows x 16 NPL columns; a stage is 32 k.
// v_mfma_f32_16x16x32_bf16 takes from lane l row / column l % 16 and k
// 8 (l / 16) .. + 7.  A: one 16-byte load per lane and 16 rows.  B is stored
// with n contiguous: the lane loads NPL adjacent columns of its eight k rows
// (16 lanes cover the block's 32 NPL bytes of a row) and transposes them in
// registers with v_perm_b32, column c of every lane feeding MFMA c, whose
// columns are therefore NPL apart.  D stages are in flight per wave.
template <int MT, int NPL, int D>
struct BfStage {
  typedef typename WordVec<NPL / 2>::type vec;
  u32x4 a[MT];
  vec b[8];
};

template <int MT, int NPL, int WK, int D, int OCC, bool WHOLE = false>
__global__ __launch_bounds__(64 * WK, OCC) void mm_direct_kernel(const DirectArgs p) {
  constexpr int BM = 16 * MT, BN = 16 * NPL, PITCH = BN + 4;
  __shared__ __attribute__((aligned(16))) float part[WK * BM * PITCH];
  int bm, bn, split;
  direct_block(p, bm, bn, split);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kg = lane >> 4;
  const int m0 = bm * BM, n0 = bn * BN;
  const uint16_t* A = static_cast<const uint16_t*>(p.A) + static_cast<int64_t>(m0) * p.lda;
  const uint16_t* B = static_cast<const uint16_t*>(p.B);

  // lane offsets (bytes); rows past M and columns past N re-read the last
  // ones, for results that are not stored
  uint32_t a_off[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    a_off[i] = 2 * (static_cast<uint32_t>(min(16 * i + l16, p.M - 1 - m0)) *
                        static_cast<uint32_t>(p.lda) + 8 * kg);
  const uint32_t b_off = 2 * (static_cast<uint32_t>(8 * kg) * static_cast<uint32_t>(p.ldb) +
                              min(n0 + NPL * l16, p.N - NPL));

  const auto part_of = [&](int part_id) {
    f32x4 acc[MT][NPL];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NPL; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const int stages = p.K / 32, first = part_id * WK + wave, step = p.splits * WK;
    typedef BfStage<MT, NPL, D> Stage;
    auto load = [&](Stage& s, int i) {  // the wave's i-th stage
      const int64_t k0 = static_cast<int64_t>(min(first + i * step, stages - 1)) * 32;
      const uint32_t bo = opaque(b_off);
      const uint16_t* ak = A + k0;
      const uint16_t* bk = B + k0 * p.ldb;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        s.b[j] = gload<typename Stage::vec>(bk + static_cast<int64_t>(j) * p.ldb, bo);
#pragma unroll
      for (int m = 0; m < MT; ++m) s.a[m] = gload<u32x4>(ak, opaque(a_off[m]));
    };
    auto compute = [&](const Stage& s) {
#pragma unroll
      for (int c = 0; c < NPL; ++c) {
        u32x4 f;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const uint32_t x = s.b[2 * d][c >> 1], y = s.b[2 * d + 1][c >> 1];
          f[d] = (c & 1) ? perm_hi(x, y) : perm_lo(x, y);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, s.a[m]), __builtin_bit_cast(bf16x8, f), acc[m][c], 0, 0, 0);
      }
    };

    const int n = stages > first ? (stages - first + step - 1) / step : 0;
    Stage st[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(st[d], d);
      __builtin_amdgcn_sched_barrier(0);
    }
    int i = 0;
    for (; i + 2 * D <= n; i += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        compute(st[d]);
        __builtin_amdgcn_sched_barrier(0);
        load(st[d], i + D + d);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (i + d < n) compute(st[d]);
      if (i + D + d < n) load(st[d], i + D + d);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (i + D + d < n) compute(st[d]);

    // lane holds of MFMA (m, c): column NPL l16 + c, rows 16 m + 4 kg + r
    float* mine = part + wave * BM * PITCH + (4 * kg) * PITCH + NPL * l16;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float* d = mine + (16 * m + r) * PITCH;
#pragma unroll
        for (int c = 0; c < NPL; c += 4)
          *reinterpret_cast<f32x4*>(d + c) =
              f32x4{acc[m][c][r], acc[m][c + 1][r], acc[m][c + 2][r], acc[m][c + 3][r]};
      }
    __syncthreads();
  };
  reduce_store<BM, BN, PITCH, WK, 64 * WK, WHOLE>(p, part, bm, bn, split, part_of);
}

// ---------------------------------------------------------------------------
// bf16 A, block-float B (BITS 8: bfloat8_b, 4: bfloat4_b).  Block of 16 MT
// rows x 32 NT columns; a stage is one tile row (32 k).  Lane l loads face row
// l of each tile (16 or 8 bytes, contiguous over the wave) and its exponent
// byte l, so the 16 elements that it decodes share one shift; it writes them
// as bf16 to the wave's own LDS, from where ds_read_b64_tr_b16 gives the
// MFMA's B operand (lane l of 16: column l of four 32-byte row pieces).
// Decoding takes most of the time (3.6 VALU instructions an element; VALU on 57%
// of a SIMD's cycles at 32 x 4096 x 11008, MFMA on 13%), not the packed bytes' 8 to
// 9 us.
template <int MT, int NT, int BITS>
struct BqStage {
  u32x4 a[MT];
  u32x4 q[NT];     // element bytes of face row `lane` (bfloat4_b: 8 bytes)
  uint32_t e[NT];  // its exponent
};

// two elements (bytes 0, 1 or 2, 3 of w; m: their magnitudes) as bf16 bits.
// v_cvt_f32_ubyte is written out: from shifts and masks the compiler extracts
// every byte first.
__device__ __forceinline__ uint32_t decode_pair(uint32_t w, uint32_t m, int shift, bool high) {
  float x, y;
  if (high) {
    asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(x) : "v"(m));
    asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(y) : "v"(m));
  } else {
    asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(x) : "v"(m));
    asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(y) : "v"(m));
  }
  // exact: at most 7 significant bits, the low half of the pattern is zero
  x = __builtin_amdgcn_ldexpf(x, shift);
  y = __builtin_amdgcn_ldexpf(y, shift);
  const uint32_t v = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
  const uint32_t sign = __builtin_amdgcn_perm(w, w, high ? 0x030C020Cu : 0x010C000Cu);
  return (sign & 0x80008000u) | v;
}

// eight nibbles (column order) -> eight bytes: sign in bit 7, magnitude below
__device__ __forceinline__ u32x2 spread_nibbles(uint32_t w) {
  const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;  // even, odd columns
  const uint32_t x = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
  const uint32_t y = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
  return u32x2{(x | (x << 4)) & 0x87878787u, (y | (y << 4)) & 0x87878787u};
}

template <int MT, int NT, int BITS, int WK, int D, int OCC, bool WHOLE = false>
__global__ __launch_bounds__(64 * WK, OCC) void mm_direct_bq_kernel(const DirectArgs p) {
  constexpr int BM = 16 * MT, BN = 32 * NT, PITCH = BN + 4;
  constexpr int kTile = BITS == 8 ? TTLH_BFP8_TILE_BYTES : TTLH_BFP4_TILE_BYTES;
  constexpr int kBias = BITS == 8 ? 133 : 129;
  // decoded stage: k row r at position (r & 3) + 4 (r >> 3) + 16 ((r >> 2) & 1),
  // which puts the rows of one transpose read on consecutive positions; the
  // pitch is an odd number of 32-byte pieces, so 32 lanes' pieces of a read fall
  // in different banks (in a write two lanes of 16 share theirs; the LDS is busy
  // 15% of the time)
  constexpr int kRow = 64 * NT + 32, kStageLds = 32 * kRow;
  constexpr int kPart = BM * PITCH * 4;
  __shared__ __attribute__((aligned(16))) uint8_t lds[WK * (kPart > kStageLds ? kPart : kStageLds)];
  int bm, bn, split;
  direct_block(p, bm, bn, split);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kg = lane >> 4;
  const int m0 = bm * BM;
  const uint16_t* A = static_cast<const uint16_t*>(p.A) + static_cast<int64_t>(m0) * p.lda;
  const uint8_t* Q = static_cast<const uint8_t*>(p.B);

  uint32_t a_off[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    a_off[i] = 2 * (static_cast<uint32_t>(min(16 * i + l16, p.M - 1 - m0)) *
                        static_cast<uint32_t>(p.lda) + 8 * kg);
  const int tiles_n = p.N / 32;
  // tiles past the last column re-read the last one
  uint32_t q_off[NT], e_off[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    e_off[t] = static_cast<uint32_t>(min(bn * NT + t, tiles_n - 1)) * kTile + lane;
    q_off[t] = e_off[t] + 64 + (BITS == 8 ? 15 : 7) * lane;
  }
  // face row `lane`: k row 16 (face / 2) + lane % 16, columns 16 (face % 2) ..
  const int kr = 16 * (lane >> 5) + l16;
  uint8_t* const put = lds + wave * kStageLds +
                       ((kr & 3) + 4 * (kr >> 3) + 16 * ((kr >> 2) & 1)) * kRow +
                       32 * ((lane >> 4) & 1);
  // transpose read of k rows 8 kg + 4 half .. + 3: lane addresses row l16 / 4,
  // columns 4 (l16 % 4) ..
  uint8_t* const get = lds + wave * kStageLds + (4 * kg + (l16 >> 2)) * kRow + 8 * (l16 & 3);
  float* const part = reinterpret_cast<float*>(lds);

  const auto part_of = [&](int part_id) {
    f32x4 acc[MT][2 * NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 2 * NT; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const int stages = p.K / 32, first = part_id * WK + wave, step = p.splits * WK;
    typedef BqStage<MT, NT, BITS> Stage;
    auto load = [&](Stage& s, int i) {
      const int64_t st = min(first + i * step, stages - 1);
      const uint16_t* ak = A + st * 32;
      const uint8_t* qk = Q + st * (static_cast<int64_t>(tiles_n) * kTile);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if constexpr (BITS == 8) {
          s.q[t] = gload<u32x4a8>(qk, opaque(q_off[t]));
        } else {
          const u32x2 v = gload<u32x2>(qk, opaque(q_off[t]));
          s.q[t].x = v.x;
          s.q[t].y = v.y;
        }
        s.e[t] = gload<uint8_t>(qk, opaque(e_off[t]));
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) s.a[m] = gload<u32x4>(ak, opaque(a_off[m]));
    };
    typedef short i16x4 __attribute__((ext_vector_type(4)));
    typedef short i16x8 __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
    auto compute = [&](const Stage& s) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        u32x4 v = s.q[t];
        if constexpr (BITS == 4) {
          const u32x2 x = spread_nibbles(v.x), y = spread_nibbles(v.y);
          v = u32x4{x.x, x.y, y.x, y.y};
        }
        const int shift = static_cast<int>(s.e[t]) - kBias;
        uint32_t o[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t m = v[i] & 0x7f7f7f7fu;
          o[2 * i] = decode_pair(v[i], m, shift, false);
          o[2 * i + 1] = decode_pair(v[i], m, shift, true);
        }
        *reinterpret_cast<u32x4*>(put + 64 * t) = u32x4{o[0], o[1], o[2], o[3]};
        *reinterpret_cast<u32x4*>(put + 64 * t + 16) = u32x4{o[4], o[5], o[6], o[7]};
      }
      // (the wave reads what it wrote itself: LDS operations of one wave
      // complete in order, so no barrier)
      asm volatile("" ::: "memory");
#pragma unroll
      for (int j = 0; j < 2 * NT; ++j) {
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(get + 32 * j));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(get + 16 * kRow + 32 * j));
        const i16x8 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, s.a[m]), __builtin_bit_cast(bf16x8, w), acc[m][j], 0, 0, 0);
      }
      asm volatile("" ::: "memory");
    };

    const int n = stages > first ? (stages - first + step - 1) / step : 0;
    Stage st[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(st[d], d);
      __builtin_amdgcn_sched_barrier(0);
    }
    int i = 0;
    for (; i + 2 * D <= n; i += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        compute(st[d]);
        __builtin_amdgcn_sched_barrier(0);
        load(st[d], i + D + d);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (i + d < n) compute(st[d]);
      if (i + D + d < n) load(st[d], i + D + d);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (i + D + d < n) compute(st[d]);

    __syncthreads();  // the stage buffers become the partial blocks
    float* d = part + wave * BM * PITCH + (4 * kg) * PITCH + l16;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < 2 * NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) d[(16 * m + r) * PITCH + 16 * j] = acc[m][j][r];
    __syncthreads();
  };
  reduce_store<BM, BN, PITCH, WK, 64 * WK, WHOLE>(p, part, bm, bn, split, part_of);
}

// ---------------------------------------------------------------------------
// fp32.  A wave owns 32 MT x 32 NT outputs and runs v_mfma_f32_32x32x2f32,
// whose operands are one element a lane (row / column lane % 32, k lane / 32):
// the k order inside a group of eight is free, so MFMA s of the group takes
// k = 4 (lane / 32) + s and a lane's A elements are one 16-byte load; B needs
// no transpose, the lane loads NT adjacent columns of a k row.
template <int MT, int NT>
struct FStage {
  f32x4 a[2][MT];       // two groups of eight k
  float b[2][4][NT];
};

template <int MT, int NT, int WM, int WN, int WK, int OCC, bool WHOLE = false>
__global__ __launch_bounds__(64 * WM * WN * WK, OCC) void mm_direct_f32_kernel(const DirectArgs p) {
  constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, PITCH = BN + 4, D = 2;
  constexpr int kWaves = WM * WN * WK;
  __shared__ __attribute__((aligned(16))) float part[WK * BM * PITCH];
  int bm, bn, split;
  direct_block(p, bm, bn, split);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave % WK, wn = (wave / WK) % WN, wm = wave / (WK * WN);
  const int l32 = lane & 31, h = lane >> 5;
  const int m0 = bm * BM, n0 = bn * BN;
  const float* A = static_cast<const float*>(p.A) + static_cast<int64_t>(m0) * p.lda;
  const float* B = static_cast<const float*>(p.B);
  uint32_t a_off[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    a_off[i] = 4 * (static_cast<uint32_t>(min(32 * (wm * MT + i) + l32, p.M - 1 - m0)) *
                        static_cast<uint32_t>(p.lda) + 4 * h);
  const uint32_t b_off = 4 * (static_cast<uint32_t>(4 * h) * static_cast<uint32_t>(p.ldb) +
                              min(n0 + 32 * NT * wn + NT * l32, p.N - NT));

  const auto part_of = [&](int part_id) {
    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    const int stages = p.K / 16, first = part_id * WK + wk, step = p.splits * WK;
    typedef FStage<MT, NT> Stage;
    auto load = [&](Stage& s, int i) {  // stage of 16 k
      const int64_t k0 = static_cast<int64_t>(min(first + i * step, stages - 1)) * 16;
      const uint32_t bo = opaque(b_off);
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const float* bk = B + (k0 + 8 * g) * p.ldb;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float* src = bk + static_cast<int64_t>(j) * p.ldb;
          if constexpr (NT == 2) {
            const f32x2 v = gload<f32x2>(src, bo);
            s.b[g][j][0] = v[0];
            s.b[g][j][1] = v[1];
          } else {
            s.b[g][j][0] = gload<float>(src, bo);
          }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) s.a[g][m] = gload<f32x4>(A + k0 + 8 * g, opaque(a_off[m]));
      }
    };
    auto compute = [&](const Stage& s) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < NT; ++c)
              acc[m][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(s.a[g][m][j], s.b[g][j][c], acc[m][c],
                                                               0, 0, 0);
    };

    const int n = stages > first ? (stages - first + step - 1) / step : 0;
    Stage st[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(st[d], d);
      __builtin_amdgcn_sched_barrier(0);
    }
    int i = 0;
    for (; i + 2 * D <= n; i += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        compute(st[d]);
        __builtin_amdgcn_sched_barrier(0);
        load(st[d], i + D + d);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (i + d < n) compute(st[d]);
      if (i + D + d < n) load(st[d], i + D + d);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (i + D + d < n) compute(st[d]);

    // lane holds of MFMA (m, c): column NT l32 + c, rows 8 (r / 4) + 4 h + r % 4
    float* d = part + wk * BM * PITCH + (32 * MT * wm + 4 * h) * PITCH + 32 * NT * wn + NT * l32;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float* dst = d + (32 * m + 8 * (r >> 2) + (r & 3)) * PITCH;
        if constexpr (NT == 2)
          *reinterpret_cast<f32x2*>(dst) = f32x2{acc[m][0][r], acc[m][1][r]};
        else
          *dst = acc[m][0][r];
      }
    __syncthreads();
  };
  reduce_store<BM, BN, PITCH, WK, 64 * kWaves, WHOLE>(p, part, bm, bn, split, part_of);
}

// ---------------------------------------------------------------------------
// Choice of the kernel.

// Parts of K for `blocks` output blocks of which the chip holds 256 at once
// (one per CU): as many as fill it, at most four, while every wave keeps
// `min_k` of K.  Where the parts are not each a workgroup's (below), one
// workgroup takes them in turn: a product's bits depend on its sizes alone.
int k_parts(int64_t blocks, int K, int min_k) {
  int parts = 1;
  while (parts < 4 && blocks * parts * 2 <= 256 && K >= min_k * parts * 2) parts *= 2;
  return parts;
}

// Whether the launch may use the scratch.  Not while the stream is being
// captured: a replay may run beside other launches that use it.
bool usable(void* scratch, hipStream_t s) {
  if (!scratch) return false;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();  // not this launch's error
    return false;
  }
  return st == hipStreamCaptureStatusNone;
}

void set_blocks(DirectArgs& a, int bm, int bn, int splits, void* scratch) {
  a.grid_m = (a.M + bm - 1) / bm;
  a.grid_n = (a.N + bn - 1) / bn;
  a.splits = splits;
  a.arrived = static_cast<int32_t*>(scratch);
  a.partial = scratch ? reinterpret_cast<float*>(static_cast<char*>(scratch) + kArrivedBytes) : nullptr;
}

void set_c_vec(DirectArgs& a) {
  const uintptr_t c = reinterpret_cast<uintptr_t>(a.C);
  a.c_vec = a.ldc % 4 == 0 && c % (a.c_dtype == TTLH_BF16 ? 8 : 16) == 0;
}

int64_t blocks_of(const DirectArgs& a, int bm, int bn) {
  return static_cast<int64_t>((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
}

// lane offsets, inside a row block of A and a stage of B, are 32-bit bytes
bool offsets_fit(const DirectArgs& a, int elem) {
  return 128 * a.lda * elem < (int64_t(1) << 32) && (24 * a.ldb + a.N) * elem < (int64_t(1) << 32);
}

#define TTLH_DIRECT_GRID(kernel, blocks, waves, name)                                          \
  do {                                                                                         \
    hipLaunchKernelGGL(HIP_KERNEL_NAME kernel, dim3(blocks), dim3(64 * (waves)), 0, s, a);     \
    *status = check_launch(name);                                                              \
  } while (0)
// a workgroup for each part of each block, and (kernels with WHOLE) one a block
#define TTLH_DIRECT(kernel, waves, name) \
  TTLH_DIRECT_GRID(kernel, a.grid_m * a.grid_n * a.splits, waves, name)
#define TTLH_DIRECT_WHOLE(kernel, waves, name) \
  TTLH_DIRECT_GRID(kernel, a.grid_m * a.grid_n, waves, name)

}  // namespace

bool may_divide_k(int a_dtype, int b_dtype, int64_t M, int64_t N, int64_t K) {
  DirectArgs a = {};
  a.M = static_cast<int32_t>(M);
  a.N = static_cast<int32_t>(N);
  const int k = static_cast<int>(K);
  if (a_dtype == TTLH_F32) return k_parts(blocks_of(a, 32, 32), k, 256) > 1;
  if (b_dtype == TTLH_BFP8 || b_dtype == TTLH_BFP4) return k_parts(blocks_of(a, 32, 64), k, 1024) > 1;
  return k_parts(blocks_of(a, 32, 128), k, 1024) > 1;  // few enough 32x64 blocks are few of these
}

bool launch_direct_bf16(DirectArgs a, double other_us, void* scratch, hipStream_t s, int* status) {
  if (!offsets_fit(a, 2)) return false;
  set_c_vec(a);
  // Modelled time of each block shape, us: per round of 256 workgroups a fixed
  // part and one per 32-k stage of a wave's share, fitted to measurements of 50
  // problems from 32x32x32 to 4096x512x2048 (the choice was the fastest of the
  // shapes or within 10% of it, but for a few at 20%).  There is no term for
  // memory: where B's bytes bound all shapes alike the times are too short (32 x
  // 11008 x 4096 13.7 us, measured 21.8), and a choice against another kernel near
  // a tie is not borne out by them.
  const double k = a.K / 32.0;
  const auto rounds = [](int64_t blocks) { return static_cast<double>((blocks + 255) / 256); };
  const int64_t b64 = blocks_of(a, 32, 64), b128 = blocks_of(a, 32, 128), m64 = blocks_of(a, 64, 128);
  const int p64 = k_parts(b64, a.K, 1024);
  const int p128 = b128 >= 80 ? std::min(2, k_parts(b128, a.K, 1024)) : 1;
  const double t[3] = {
      1 + (1.2 + 0.11 * k / p64) * rounds(b64 * p64) + (p64 > 1 ? 2 : 0),
      1 + (1.5 + 0.153 * k / p128) * rounds(b128 * p128) + (p128 > 1 ? 2 : 0),
      1 + (2 + 0.237 * k) * rounds(m64),
  };
  const int best = static_cast<int>(std::min_element(t, t + 3) - t);
  if (t[best] >= other_us) return false;
  const int parts = best == 0 ? p64 : best == 1 ? p128 : 1;
  if (parts > 1 && !usable(scratch, s)) {
    // (also where the parts would be of 32x128 blocks, which use half as many
    // CUs here: the bits are those of the parts, not of the blocks' width)
    set_blocks(a, 32, 64, parts, nullptr);
    TTLH_DIRECT_WHOLE((mm_direct_kernel<2, 4, 8, 3, 3, true>), 8, "mm_direct_kernel");
  } else if (best == 0) {
    set_blocks(a, 32, 64, p64, scratch);
    TTLH_DIRECT((mm_direct_kernel<2, 4, 8, 3, 3>), 8, "mm_direct_kernel");
  } else if (best == 1) {
    set_blocks(a, 32, 128, p128, scratch);
    TTLH_DIRECT((mm_direct_kernel<2, 8, 8, 2, 2>), 8, "mm_direct_kernel");
  } else {
    set_blocks(a, 64, 128, 1, nullptr);
    TTLH_DIRECT((mm_direct_kernel<4, 8, 4, 2, 2>), 4, "mm_direct_kernel");
  }
  return true;
}

bool launch_direct_block(DirectArgs a, int bits, void* scratch, hipStream_t s, int* status) {
  const int64_t row = static_cast<int64_t>(a.N / 32) *
                      (bits == 8 ? TTLH_BFP8_TILE_BYTES : TTLH_BFP4_TILE_BYTES);
  if (128 * a.lda * 2 >= (int64_t(1) << 32) || row >= (int64_t(1) << 32)) return false;
  set_c_vec(a);
  // A wave decodes the weights of its columns once for all its rows, so 64
  // rows are taken as soon as such blocks fill most of the CUs: 64 x 4096 x
  // 11008 20.6 us against 25.0, 1024^3 8.4 against 10.2; fewer blocks are
  // faster in 32 rows: 512^3 4.8 against 5.6.
  if (blocks_of(a, 64, 64) >= 160 && a.M > 32) {
    set_blocks(a, 64, 64, 1, nullptr);
    if (bits == 8) TTLH_DIRECT((mm_direct_bq_kernel<4, 2, 8, 4, 2, 2>), 4, "mm_direct_bq_kernel");
    else TTLH_DIRECT((mm_direct_bq_kernel<4, 2, 4, 4, 2, 2>), 4, "mm_direct_bq_kernel");
    return true;
  }
  set_blocks(a, 32, 64, k_parts(blocks_of(a, 32, 64), a.K, 1024), scratch);
  if (a.splits > 1 && !usable(scratch, s)) {
    if (bits == 8)
      TTLH_DIRECT_WHOLE((mm_direct_bq_kernel<2, 2, 8, 8, 3, 3, true>), 8, "mm_direct_bq_kernel");
    else
      TTLH_DIRECT_WHOLE((mm_direct_bq_kernel<2, 2, 4, 8, 3, 3, true>), 8, "mm_direct_bq_kernel");
    return true;
  }
  if (bits == 8) TTLH_DIRECT((mm_direct_bq_kernel<2, 2, 8, 8, 3, 3>), 8, "mm_direct_bq_kernel");
  else TTLH_DIRECT((mm_direct_bq_kernel<2, 2, 4, 8, 3, 3>), 8, "mm_direct_bq_kernel");
  return true;
}

bool launch_direct_f32(DirectArgs a, void* scratch, hipStream_t s, int* status) {
  // 16-byte loads of A, 8-byte loads of B
  if ((reinterpret_cast<uintptr_t>(a.A) & 15) || a.lda % 4 || (reinterpret_cast<uintptr_t>(a.B) & 7) ||
      a.ldb % 2 || !offsets_fit(a, 4))
    return false;
  set_c_vec(a);
  // 128x128 blocks where they fill whole rounds of the CUs: 2048^3 126 us
  // against 142 to 145 in smaller blocks, but 1504^3 (144 blocks) 93 against
  // 68.  Few outputs go in 32x32 blocks with K over eight (and more) waves:
  // 256 x 2048 x 256 8.3 us, 12.9 without the parts.
  const int64_t big = blocks_of(a, 128, 128), small = blocks_of(a, 32, 32);
  if (4 * big >= 3 * 256 * ((big + 255) / 256)) {
    set_blocks(a, 128, 128, 1, nullptr);
    TTLH_DIRECT((mm_direct_f32_kernel<2, 2, 2, 2, 2, 2>), 8, "mm_direct_f32_kernel");
  } else if (small <= 128) {
    set_blocks(a, 32, 32, k_parts(small, a.K, 256), scratch);
    if (a.splits > 1 && !usable(scratch, s))
      TTLH_DIRECT_WHOLE((mm_direct_f32_kernel<1, 1, 1, 1, 8, 4, true>), 8, "mm_direct_f32_kernel");
    else
      TTLH_DIRECT((mm_direct_f32_kernel<1, 1, 1, 1, 8, 4>), 8, "mm_direct_f32_kernel");
  } else if (small <= 512) {
    set_blocks(a, 32, 32, 1, nullptr);
    TTLH_DIRECT((mm_direct_f32_kernel<1, 1, 1, 1, 4, 4>), 4, "mm_direct_f32_kernel");
  } else {
    set_blocks(a, 32, 64, 1, nullptr);
    TTLH_DIRECT((mm_direct_f32_kernel<1, 2, 1, 1, 8, 3>), 8, "mm_direct_f32_kernel");
  }
  return true;
}

}  // namespace ttlh
