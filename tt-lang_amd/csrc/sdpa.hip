// Fused scaled-dot-product attention forward for gfx950:
//   O[b, h] = softmax(Q[b, h] K[b, h]^T * scale) V[b, h],  bf16 in / out,
//   fp32 scores and online softmax.
//
// The reference has no attention kernel; this composes the spec's tile ops
// (@, exp, reduce_max, reduce_sum, recip, broadcast:
// docs/sphinx/specs/TTLangSpecification.md:693-761) into one flash-style pass.
//
// Per wave, 32 query rows and per KV block (64 rows):
//     S^T = K Q^T   (16 x v_mfma_f32_32x32x16_bf16, Q^T operands kept in VGPRs)
//     O^T += V^T P^T (16 more MFMAs)
// Computing the transposes puts one query row in each lane's accumulator
// column for both products, so the softmax statistics (running max m and sum
// l) and the O rescale are per-lane scalars; the two lane halves that share a
// query combine with one exchange.  P goes from the S accumulators to the
// second MFMA without touching LDS: the accumulator layout hands each lane kv
// rows {16c + 4h + 8u + i}, so the V^T operand is read in the same kv order
// (the contraction is invariant under a common permutation of kv), with two
// ds_read_b64_tr_b16 transpose loads from row-major V: within a group of 16
// lanes, output lane i, element k is element i % 4 of the 8 bytes that lane
// 4k + i / 4 addresses, so lanes addressing 4 kv rows x 16 d columns receive
// 4 consecutive kv of one d column each.
//
// Two kernels share that per-wave math:
//  * sdpa_w8_kernel (D = 128, non-causal, S a multiple of 256): 8 waves of
//    32 queries, two per SIMD, each interleaving the MFMAs of a KV block with
//    the softmax of the previous one, the second wave's VALU issuing under
//    the first one's MFMAs; Q pre-scaled and the S accumulation started from
//    -m, so the softmax is one exp2 per score; a persistent grid of one
//    workgroup per CU (details at its definition);
//  * sdpa_fwd_kernel (everything else): 128 queries per workgroup, K and V
//    blocks of 64 rows, in two forms.  One group of four waves, two workgroups
//    per CU, drifts apart so that one's softmax runs under the other's MFMAs;
//    it is the faster one wherever the blocks fill the chip's 512 places.  With
//    fewer, a CU would hold one group with nothing to hide its latencies, so
//    two groups share the workgroup's queries, taking the even and the odd KV
//    blocks, and their results meet in LDS: 1 x 8 x 4000 x 128 causal 107 ->
//    66 us, 1 x 16 x 992 x 128 31 -> 22.5.  Either is bound by the latencies of
//    its chain S -> softmax -> O.  K and V come by direct-to-LDS loads: through
//    registers and LDS stores they took a quarter of the time (1 x 32 x 2048 x 128
//    causal, with nothing to load or store 39 of 50 us); 4 x 32 x 4096 x 128 causal
//    663 -> 615 us, 4 x 32 x 4096 x 64 647 -> 614.
//    A third kernel, which ran the two groups in ping-pong over 256 queries, was
//    slower than these in every case it took (1 x 32 x 2048 x 128 causal 71 us
//    against 58, 4 x 32 x 4096 x 64 682 against 646).
//
// K and V lie in LDS row-major and unpadded (a direct-to-LDS load writes 64 x 16
// consecutive bytes), the 16-byte chunks of a row permuted.  gfx950's LDS serves
// 256 bytes (64 banks) per cycle: a ds_read_b128 is conflict-free when each 16
// lanes hit 16 distinct 16-byte bank groups, a ds_read_b64 when each 32 lanes do.
// K (16 rows, one chunk each): chunk c of row r at c ^ (r & 15), for D = 64, where
// two rows share the banks, at c ^ ((r >> 1) & 7); V (4 rows x 4 chunks per 32
// lanes of a transpose read): at c ^ 4 (r & 3), for D = 64 at c ^ 4 ((r >> 1) & 1).
// (No bank conflict is counted in any form.)
// The next block's loads run while the current block computes.
// Softmax runs in the log2 domain: exp2(fma(s, scale log2 e, -m)) in
// sdpa_fwd_kernel, with the block max taken on the raw scores (sign of the
// scale handled by taking the min instead); the causal mask touches only the blocks
// that straddle the diagonal.  P is rounded to bf16 for the MFMA; O is
// divided by l at the end.  Workgroup ids are regrouped so the query blocks
// of one (batch, head) land on the same XCD and share K/V in its L2.

#include <cmath>
#include <type_traits>

#include "ttlh_common.h"

namespace ttlh {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

constexpr int BQ = 128;   // query rows per workgroup
constexpr int BKV = 64;   // kv rows per block
constexpr int kThreads = 256;

struct SdpaArgs {
  const uint16_t* Q;
  const uint16_t* K;
  const uint16_t* V;
  uint16_t* O;
  int32_t S;
  int32_t nqb;        // query blocks per (b, h)
  int32_t nbh;        // B * H
  int32_t heads_together;  // causal: heads whose blocks are dispatched longest first
  float scale_log2;   // scale * log2(e)
};

__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) { return cvt_pk_bf16x2(lo, hi); }

// x combined with the value of lane l ^ 32, without LDS: v_permlane32_swap
// exchanges the upper half of its first operand with the lower half of its
// second, so with both operands = x the two results hold, per lane, x and
// x of lane l ^ 32 (in some order)
__device__ __forceinline__ float xor32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_min(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fminf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_add(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// s_waitcnt immediate (gfx9 encoding): at most n global loads outstanding
constexpr int vmcnt_imm_sdpa(int n) { return 0x0F70 | (n & 0xF) | ((n >> 4) << 14); }

typedef __attribute__((address_space(3))) void lds_void;

// One direct-to-LDS load per lane: its 16 bytes at byte `off` from the uniform
// `src` land at the uniform `lds` + 16 lane.  Inline asm, waited for explicitly:
// the compiler would wait for every LDS read while one it knows of is in flight.
__device__ __forceinline__ void dma16(uint64_t src, uint32_t off, uint32_t lds) {
  const uint64_t g =
      (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(src >> 32)))) << 32) |
      uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(src))));
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(off), "s"(g)
      : "memory", "m0");
}

// the block's queries: q blocks of one (b, h) are kept on one XCD
__device__ __forceinline__ void block_coords(const SdpaArgs& p, int& bh, int& qb) {
  const int nblk = p.nbh * p.nqb;
  int id = blockIdx.x;
  constexpr int kXcd = 8;
  if (nblk % kXcd == 0) {
    const int per = nblk / kXcd;
    id = (id % kXcd) * per + id / kXcd;
  }
  bh = id / p.nqb;
  qb = id - bh * p.nqb;
}

// Causal: block qb has qb + 1 units of work, and the workgroups are dispatched
// in order as CUs fall free, so the longest go first: of `heads_together` heads
// (as many as share an XCD's L2 with their K and V), all last blocks, then all
// last but one, and so on.
template <bool CAUSAL>
__device__ __forceinline__ void ordered_block(const SdpaArgs& p, int& bh, int& qb) {
  block_coords(p, bh, qb);
  if constexpr (CAUSAL) {
    const int id = bh * p.nqb + qb, span = p.heads_together * p.nqb;
    const int g = id / span, r = id - g * span;
    const int heads = min(p.heads_together, p.nbh - g * p.heads_together);
    qb = p.nqb - 1 - r / heads;
    bh = g * p.heads_together + r % heads;
  }
}

template <int D, bool CAUSAL, bool RAGGED = false>
struct Sdpa {
  static constexpr int ND = D / 32;   // d tiles of O^T
  static constexpr int NDC = D / 16;  // 16-wide d chunks of the S^T contraction

  const SdpaArgs& p;
  uint16_t (*Ks)[BKV * D];
  uint16_t (*Vs)[BKV * D];
  int64_t base;
  int qb, wave, lane, l32, h, q, nkv;
  float sc;
  bf16x8 qop[NDC];
  f32x16 o[ND];
  float m, l;
  int row0, k_src, v_src;   // DMA: the thread's first row; its chunks' elements in a row
  int k_frag, v_frag[ND];   // LDS elements of the K and V fragment reads

  static constexpr int kChunks = D / 8;                // 16-byte chunks in a row
  static constexpr int kRowsPer = kThreads / kChunks;  // rows that one DMA of the group covers
  // position of chunk c of row r: c ^ k_swz(r) in K, c ^ v_swz(r) in V
  static __device__ __forceinline__ int k_swz(int r) { return D == 128 ? r & 15 : (r >> 1) & 7; }
  static __device__ __forceinline__ int v_swz(int r) {
    return D == 128 ? (r & 3) << 2 : ((r >> 1) & 1) << 2;
  }

  __device__ __forceinline__ void setup() {
    const int t = threadIdx.x & (kThreads - 1);
    row0 = t / kChunks;
    k_src = ((t % kChunks) ^ k_swz(row0)) * 8;
    v_src = ((t % kChunks) ^ v_swz(row0)) * 8;
    k_frag = l32 * D + ((h ^ k_swz(l32)) << 3);
    const int vr = (lane & 15) >> 2;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      const int chunk = 4 * j + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
      v_frag[j] = (4 * h + vr) * D + ((chunk ^ v_swz(vr)) << 3) + 4 * (lane & 1);
    }
  }

  // rows kb * 64 .. + 63 of X into an LDS buffer; with RAGGED, rows past the
  // sequence are its last row again.  Without, the loads share one offset a lane
  // that stays the same for the whole loop, their rows in the uniform address
  // (causal: 1 x 8 x 4096 x 128 65.9 us -> 64.8, 1 x 8 x 2048 x 128 36.5 -> 36.0, 2
  // x 32 x 2048 x 64 51.3 -> 50.4; no change without the mask.  The same for all
  // but the last block of a ragged sequence, behind a branch, was slower: 1 x 8 x
  // 4000 x 128 65.5 -> 66.7).
  __device__ __forceinline__ void dma(const uint16_t* X, int chunk, int kb, const uint16_t* buf) {
    const uint64_t src = reinterpret_cast<uint64_t>(X + base + static_cast<int64_t>(kb) * BKV * D);
    const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)buf));
#pragma unroll
    for (int i = 0; i < BKV / kRowsPer; ++i) {
      const uint32_t at = lds + i * kThreads * 16 + wave * 1024;
      if constexpr (RAGGED) {
        const int row = min(row0 + i * kRowsPer, p.S - 1 - kb * BKV);
        dma16(src, static_cast<uint32_t>(row * D + chunk) * 2u, at);
      } else {
        dma16(src + i * kRowsPer * D * 2, static_cast<uint32_t>(row0 * D + chunk) * 2u, at);
      }
    }
  }

  // The loads of block kb have landed; with RAGGED, the V rows past the sequence
  // become zeros (each thread's own chunks), so that 0 * V is 0 there.  (The
  // scores of such K rows are masked.)
  __device__ __forceinline__ void landed(int kb, uint16_t* Vb) {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm_sdpa(0));
    asm volatile("" ::: "memory");
    if (RAGGED && kb * BKV + BKV > p.S) {
      const int t = threadIdx.x & (kThreads - 1);
#pragma unroll
      for (int i = 0; i < BKV / kRowsPer; ++i)
        if (kb * BKV + row0 + i * kRowsPer >= p.S)
          *reinterpret_cast<u32x4*>(Vb + (i * kThreads + t) * 8) = u32x4{0u, 0u, 0u, 0u};
    }
  }

  // 4 consecutive kv rows of one d column each of V's tile j (see the
  // transpose-load rule above), from row kv + 4 h
  __device__ __forceinline__ i16x4 read_v4(const uint16_t* Vb, int kv, int j) const {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(Vb + v_frag[j] + kv * D));
  }

  // S^T = K Q^T for the K block at K_ (raw scores).  The K fragments are read
  // kAhead before the MFMA that takes them, into the registers that hold the
  // exponentials later; the scheduling fences keep the compiler from sinking the
  // reads to their uses, where each pair waits for the LDS (2% under the mask;
  // eight ahead no faster).
  __device__ __forceinline__ void scores(const uint16_t* K_, f32x16 (&sv)[2]) {
    constexpr int kAhead = 4;
    const auto frag = [&](int i) {
      return *reinterpret_cast<const bf16x8*>(K_ + (k_frag ^ ((i % NDC) * 16)) + (i / NDC) * 32 * D);
    };
    bf16x8 f[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) f[i] = frag(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sv[t][r] = 0.0f;
#pragma unroll
      for (int dc = 0; dc < NDC; ++dc) {
        const int i = t * NDC + dc;
        sv[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[i % kAhead], qop[dc], sv[t], 0, 0, 0);
        if (i + kAhead < 2 * NDC) f[i % kAhead] = frag(i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  __device__ __forceinline__ float expo(float v, float mx) const {
    return __builtin_amdgcn_exp2f(__builtin_fmaf(v, sc, -mx));
  }

  // One KV block kb = it * GROUPS + group, if there is one: the group's next
  // block's K and V are on their way to the other LDS buffer (last read before
  // the previous barrier) while this one computes S, the softmax and
  // O += V(kb)^T P^T from buffer it & 1.
  template <int GROUPS>
  __device__ __forceinline__ void step(int it, int group) {
    const int kb = it * GROUPS + group, next = kb + GROUPS;
    if (next < nkv) {
      dma(p.K, k_src, next, Ks[(it + 1) & 1]);
      dma(p.V, v_src, next, Vs[(it + 1) & 1]);
    }
    // (causal: the last KV block of a workgroup lies wholly past the queries of
    // its waves 0 and 1)
    if ((GROUPS == 1 || kb < nkv) && (!CAUSAL || kb * BKV <= qb * BQ + wave * 32 + 31))
      block(kb, Ks[it & 1], Vs[it & 1]);
    if (next < nkv) landed(next, Vs[(it + 1) & 1]);
    __syncthreads();
  }

  __device__ __forceinline__ void block(int kb, const uint16_t* Kc, const uint16_t* Vc) {
    f32x16 cur[2];
    // (the wave with MFMAs goes first where the other wave of its SIMD is in its
    // softmax: 1 x 32 x 2016 x 128 84.0 -> 81.7 us; no gain under the mask)
    if constexpr (!CAUSAL && D == 128) __builtin_amdgcn_s_setprio(1);
    scores(Kc, cur);
    if constexpr (!CAUSAL && D == 128) __builtin_amdgcn_s_setprio(0);

    // causal: only blocks that reach past this wave's first query need a
    // mask; ragged: the block that runs past the sequence end masks the kv
    // beyond it (masked scores drop out of the block extreme and get exp 0)
    // the V^T operand i of lane (d = 32j + l32, h), j = i % ND, holds kv
    // {16c + 4h + i, 16c + 4h + 8 + i}, c = i / ND; the first ones are read here,
    // under the softmax
    const auto vfrag = [&](int i) {
      const i16x4 lo = read_v4(Vc, 16 * (i / ND), i % ND);
      const i16x4 hi = read_v4(Vc, 16 * (i / ND) + 8, i % ND);
      const i16x8 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      return __builtin_bit_cast(bf16x8, w);
    };
    constexpr int kAhead = 4;
    bf16x8 vf[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) vf[i] = vfrag(i);
    __builtin_amdgcn_sched_barrier(0);

    const bool diag = (CAUSAL && kb * BKV + BKV - 1 > qb * BQ + wave * 32) ||
                      (RAGGED && kb * BKV + BKV > p.S);
    auto masked = [&](int kv) { return (CAUSAL && kv > q) || (RAGGED && kv >= p.S); };
    if (diag) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kv = kb * BKV + 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
          if (masked(kv)) cur[t][r] = sc >= 0.0f ? -INFINITY : INFINITY;
        }
    }
    // block extreme of the raw scores: max if the scale is positive, else min
    float ex = cur[0][0];
    if (sc >= 0.0f) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) ex = fmaxf(ex, cur[t][r]);
      ex = xor32_max(ex);
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) ex = fminf(ex, cur[t][r]);
      ex = xor32_min(ex);
    }
    // O is rescaled only when some lane's running max moves.  (Letting it lag
    // by up to 2^8 saves 2 to 5% of the time, but the largest probability is
    // then no longer 1, exact in bf16: 2 to 5% more error.)
    const float m_blk = ex * sc;
    if (__any(m_blk > m)) {
      const float m_new = fmaxf(m, m_blk);
      const float alpha = m_new == m ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);  // 0 at first
      l *= alpha;
#pragma unroll
      for (int j = 0; j < ND; ++j) o[j] *= alpha;
      m = m_new;
    }
    // (a lane that has seen only masked or -inf scores keeps m = -inf: its
    // exponentials are 0)
    const float mm = m == -INFINITY ? 0.0f : m;
    float rs = 0.0f;
    if (diag) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kv = kb * BKV + 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
          const float e = masked(kv) ? 0.0f : expo(cur[t][r], mm);
          cur[t][r] = e;
          rs += e;
        }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = expo(cur[t][r], mm);
          cur[t][r] = e;
          rs += e;
        }
    }
    l += rs;  // of this lane's kv: the two halves, whose m is one, meet at the end

    // P^T operands: chunk c (16 kv) = tile c/2, accumulators 8(c%2) .. +8
    bf16x8 pb[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int t = c >> 1, r0 = 8 * (c & 1);
      u32x4 w;
      w.x = pk_bf16(cur[t][r0 + 0], cur[t][r0 + 1]);
      w.y = pk_bf16(cur[t][r0 + 2], cur[t][r0 + 3]);
      w.z = pk_bf16(cur[t][r0 + 4], cur[t][r0 + 5]);
      w.w = pk_bf16(cur[t][r0 + 6], cur[t][r0 + 7]);
      pb[c] = __builtin_bit_cast(bf16x8, w);
    }
    if constexpr (!CAUSAL) __builtin_amdgcn_s_setprio(1);
    // O^T += V^T P^T, one chunk of 16 kv after the other, so that consecutive
    // MFMAs are independent
#pragma unroll
    for (int i = 0; i < 4 * ND; ++i) {
      o[i % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i % kAhead], pb[i / ND], o[i % ND], 0,
                                                          0, 0);
      if (i + kAhead < 4 * ND) vf[i % kAhead] = vfrag(i + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!CAUSAL) __builtin_amdgcn_s_setprio(0);
  }
};

// RAGGED: S a multiple of 32 only.  The last query block holds waves past
// the sequence (S % 32 == 0 keeps each wave wholly in or out): they read a
// clamped Q row, take part in the K / V staging and barriers, store nothing.
// The last KV block reads rows past S as zeros and masks their scores.
template <int D, bool CAUSAL, bool RAGGED, int GROUPS>
__global__ __launch_bounds__(kThreads * GROUPS, 2 / GROUPS) void sdpa_fwd_kernel(const SdpaArgs p) {
  // K, then V, of each group, two buffers each
  __shared__ __attribute__((aligned(256))) uint16_t KV[2 * GROUPS][2][BKV * D];
  const int group = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  Sdpa<D, CAUSAL, RAGGED> w{p, KV[group], KV[GROUPS + group]};
  int bh;
  ordered_block<CAUSAL>(p, bh, w.qb);
  w.lane = threadIdx.x & 63;
  w.wave = (threadIdx.x >> 6) & 3;
  w.l32 = w.lane & 31;
  w.h = w.lane >> 5;
  w.base = static_cast<int64_t>(bh) * p.S * D;
  w.q = w.qb * BQ + w.wave * 32 + w.l32;  // this lane's query row
  w.sc = p.scale_log2;
  w.m = -INFINITY;  // running max of s * scale * log2 e
  w.l = 0.0f;
  if constexpr (RAGGED) {
    const int nall = (p.S + BKV - 1) / BKV;
    w.nkv = CAUSAL ? min(nall, (w.qb * BQ + BQ) / BKV) : nall;
  } else {
    w.nkv = CAUSAL ? (w.qb * BQ + BQ) / BKV : p.S / BKV;
  }
  const int qload = RAGGED ? min(w.q, p.S - 1) : w.q;  // a wave past S reads a valid row

  w.setup();
  // prologue: the group's first K and V block into LDS; Q^T into VGPRs
  if (group < w.nkv) {
    w.dma(p.K, w.k_src, group, w.Ks[0]);
    w.dma(p.V, w.v_src, group, w.Vs[0]);
  }
#pragma unroll
  for (int dc = 0; dc < D / 16; ++dc)
    w.qop[dc] = *reinterpret_cast<const bf16x8*>(p.Q + w.base + static_cast<int64_t>(qload) * D +
                                                 dc * 16 + 8 * w.h);
#pragma unroll
  for (int j = 0; j < D / 32; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) w.o[j][r] = 0.0f;
  // (the wait for K and V is one for Q^T too: Q^T must have landed before the
  // loop, or its MFMAs would wait for the next block's K and V every time)
  __builtin_amdgcn_s_waitcnt(vmcnt_imm_sdpa(0));
  if (group < w.nkv) w.landed(group, w.Vs[0]);
  __syncthreads();

  const int steps = (w.nkv + GROUPS - 1) / GROUPS;
  for (int it = 0; it < steps; ++it) w.template step<GROUPS>(it, group);

  if constexpr (GROUPS == 2) {
    // Group 1 leaves its max, sum and O in LDS (every group is past its last
    // read of K and V); group 0's wave w, which holds the same queries in the
    // same lanes as wave w + 4, adds them.
    float* part = reinterpret_cast<float*>(&KV[0][0][0]) + (w.wave * (16 * (D / 32) + 2)) * 64 + w.lane;
    static_assert(sizeof(KV) >= 4 * 64 * (16 * (D / 32) + 2) * sizeof(float), "partial O fits");
    if (group == 1) {
      part[0] = w.m;
      part[64] = w.l;
#pragma unroll
      for (int j = 0; j < D / 32; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) part[(2 + 16 * j + r) * 64] = w.o[j][r];
    }
    __syncthreads();
    if (group == 1) return;
    const float m1 = part[0], mt = fmaxf(w.m, m1);
    const float a0 = w.m == mt ? 1.0f : __builtin_amdgcn_exp2f(w.m - mt);
    const float a1 = m1 == mt ? 1.0f : __builtin_amdgcn_exp2f(m1 - mt);
    w.l = w.l * a0 + part[64] * a1;
#pragma unroll
    for (int j = 0; j < D / 32; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        w.o[j][r] = w.o[j][r] * a0 + part[(2 + 16 * j + r) * 64] * a1;
  }
  if (RAGGED && w.q >= p.S) return;  // wave-uniform (S % 32 == 0); no barrier follows

  // O[q][d], d = 32j + 8u + 4h + i: four contiguous bf16 per (j, u)
  const float inv = 1.0f / xor32_add(w.l);
  uint16_t* orow = p.O + w.base + static_cast<int64_t>(w.q) * D;
#pragma unroll
  for (int j = 0; j < D / 32; ++j)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int d = 32 * j + 8 * u + 4 * w.h;
      const u32x2 v = {pk_bf16(w.o[j][4 * u] * inv, w.o[j][4 * u + 1] * inv),
                       pk_bf16(w.o[j][4 * u + 2] * inv, w.o[j][4 * u + 3] * inv)};
      *reinterpret_cast<u32x2*>(orow + d) = v;
    }
}

template <int N, typename F>
__device__ __forceinline__ void sd_static_for(F&& f) {
  if constexpr (N > 0) {
    sd_static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>());
  }
}

// ---------------------------------------------------------------------------
// 32 queries per wave, eight waves (two per SIMD) per block of 256 queries
// (D = 128, non-causal: C5).  KV blocks of 32 rows; step i of a block is one
// straight-line piece of code:
//     MFMAs: S(i) = K(i) Q^T and O += V(i-2)^T P(i-2)^T (16)
//     VALU:  the softmax of S(i-1) -> P(i-1) and its row sum (the running
//            max moves only on a rare path, see below)
// in eight sections, one per K / V fragment: the section's two MFMAs, a
// share of the softmax VALU, and the LDS reads of the fragments two sections
// ahead.  Two waves per SIMD because a wave alone cannot hide its VALU work:
// on gfx950 an MFMA holds its own wave's issue for about half of its 32
// cycles, so VALU placed between one wave's MFMAs mostly adds to them, while
// a second wave's VALU issues under them (measured: MFMA + 16 FMAs takes 80
// cycles for one wave, 62 for two).  The cost is LDS traffic: each K / V
// fragment feeds one MFMA (128 KB per step per CU; gfx950's LDS serves 256
// bytes per clock to ds_read_b128 and ~186 to ds_read_b64_tr_b16, measured,
// so the reads take ~600 of the step's 1024 MFMA cycles).  The accumulators
// fit in the architectural VGPRs (239, no AGPRs), so the softmax reads S
// without copies.  The waves raise their priority (s_setprio 1) over the first six
// sections, where MFMAs and LDS reads are densest, so a SIMD's matrix core
// is fed first and the other wave's VALU fills the gaps.
// K and V reach LDS by direct-to-LDS DMA (global_load_lds_dwordx4, lane l's
// 16 bytes at the wave's base + 16 l) into rings of four K and four V
// buffers (64 KB): step t reads K(t) from K buffer t % 4 and V(t - 2) from V
// buffer (t - 2) % 4, and loads K(t + 3) and V(t + 1); one workgroup barrier
// per step, and each step's first two K / V fragments are read before the
// previous step's barrier (their blocks were published one barrier earlier).
// Rows are unpadded with XOR-swizzled 16-byte chunks: K chunk c of row r at
// c ^ (r & 15) (the S operand reads 16 rows of one chunk per 16 lanes), V at
// c ^ 4 (r & 3) (a transpose read covers 4 rows x 4 chunks per 32 lanes).
// The grid is persistent: one workgroup per CU walks a sequence of query
// blocks, and the step pipeline runs across block boundaries (t counts steps
// over the sequence; a block is n steps, a multiple of 4, so the ring phases
// repeat).  A block's steps 0 and 1 also carry the previous block's last
// softmax and O products, its first K / V blocks are the loads that follow
// the previous block's, its Q is staged into LDS four steps ahead (64 KB, per
// wave) and loaded into registers at the end of the previous block, and a
// finished block's O is stored after the step holding its last product: per
// block there is no pipeline fill or drain, no Q load latency and no
// workgroup launch (3% faster than one workgroup per block).
constexpr int W8_BQ = 256;
constexpr int W8_THREADS = 512;
constexpr int W8_D = 128;
constexpr int W8_KV = 32;

// one array per ring, so a buffer is a constant offset from the others (an
// immediate in the LDS instructions, not another address register)
__shared__ __attribute__((aligned(16))) uint16_t w8K[4][W8_KV * W8_D];
__shared__ __attribute__((aligned(16))) uint16_t w8V[4][W8_KV * W8_D];
// per wave, the next block's 32 Q rows (staged four steps ahead)
__shared__ __attribute__((aligned(16))) uint16_t w8Q[8][32 * W8_D];

template <int B>
__device__ __forceinline__ uint16_t* w8_kbuf() {
  return w8K[B];
}
template <int B>
__device__ __forceinline__ uint16_t* w8_vbuf() {
  return w8V[B];
}

struct SdpaW8 {
  static constexpr int D = W8_D, ND = D / 32, NDC = D / 16;

  const SdpaArgs& p;
  int wave, lane, l32, h, n;
  bf16x8 qop[NDC];          // Q^T operands, scaled by scale * log2(e)
  f32x16 o[ND];             // O^T accumulators
  f32x16 s;                 // S(i) - m accumulating
  f32x16 sv;                // S(i - 1) - m (renamed, not copied: both live in VGPRs)
  f32x16 negm;              // -m in every element: where each S accumulation starts
  u32x4 pw[2][2];           // [parity][kv chunk]: P(i - 1), P(i - 2) as bf16 pairs
  float m, l;               // running max (log2 units), this lane's share of the row sum
  float limit;              // block sum above which the wave goes to rescale() (uniform)
  int k_src, v_src;         // per-lane DMA source offsets (elements)
  int v_frag[ND];           // LDS offsets of the V transpose reads
  uint32_t lds_wave;        // the wave's byte offset in a K / V buffer (uniform)
  bf16x8 kpf[2], vpf[2];    // the next step's first K / V fragments, read before the barrier

  __device__ __forceinline__ void setup() {
    lds_wave = __builtin_amdgcn_readfirstlane(wave * 1024);
    const int pos = wave * 64 + lane;  // 16-byte chunk position in the buffer
    const int r = pos >> 4, c = pos & 15;
    k_src = r * D + ((c ^ (r & 15)) << 3);
    v_src = r * D + ((c ^ ((r & 3) << 2)) << 3);
    // V transpose reads: row kv0 + (lane & 15) / 4, logical column d0 + 4 (lane & 3),
    // d0 = 32 j + 16 ((lane >> 4) & 1), i.e. chunk 4 j + 2 ((lane >> 4) & 1) + (lane & 3) / 2
    const int vr = (lane & 15) >> 2;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      const int chunk = 4 * j + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
      v_frag[j] = vr * D + ((chunk ^ (vr << 2)) << 3) + 4 * (lane & 1);
    }
  }

  // 32 K or V rows from kv0 into an LDS buffer: one DMA instruction per thread,
  // issued as inline asm: with a compiler-visible LDS DMA outstanding, the
  // compiler's wait-count model treats LDS reads as completing out of order
  // and waits for every LDS read (lgkmcnt(0)) before each use, which defeats
  // the fragment prefetch.  The DMA counts only on vmcnt, waited explicitly
  // at the end of every step, before any wave reads the buffer (the loop has
  // no other vector-memory loads, so vmcnt counts exactly these).  M0 carries the wave's LDS base (one wait
  // state before use).  The address is the uniform row base in an SGPR pair
  // plus the lane's 32-bit byte offset: no 64-bit VGPR address, which would
  // need an even-aligned register pair the asm constraint cannot request.
  // Both uniform operands pass through readfirstlane, so they are SGPRs
  // whatever the register allocator made of them (free when they already
  // are); readfirstlane returns int, so each pointer half widens unsigned.
  __device__ __forceinline__ void dma(const uint16_t* X, int64_t base, int src, int kv0,
                                      const uint16_t* lds) {
    const uint64_t g = reinterpret_cast<uint64_t>(X + base + static_cast<int64_t>(kv0) * D);
    const uint64_t gs =
        (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(g >> 32)))) << 32) |
        uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(g))));
    const uint32_t buf = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)lds));
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2"
        :
        : "s"(__builtin_amdgcn_readfirstlane(buf + lds_wave)),
          "v"(static_cast<uint32_t>(src) * 2u), "s"(gs)
        : "memory", "m0");
  }

  // K fragment (d chunk dc): row l32, 8 elements at 16 dc + 8 h (chunk 2 dc + h)
  __device__ __forceinline__ bf16x8 kfrag(const uint16_t* Kc, int dc) const {
    const int chunk = (2 * dc + h) ^ (l32 & 15);
    return *reinterpret_cast<const bf16x8*>(Kc + l32 * D + chunk * 8);
  }
  // V^T fragment (d tile j, kv chunk c): rows {16c + 4h + i, 16c + 4h + 8 + i}
  __device__ __forceinline__ bf16x8 vfrag(const uint16_t* Vc, int j, int c) const {
    const uint16_t* a0 = Vc + (16 * c + 4 * h) * D + v_frag[j];
    const uint16_t* a1 = a0 + 8 * D;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)a0);
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)a1);
    const i16x8 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, w);
  }

  // The softmax of S(i - 1) - m (sv) into pw[PAR]: one pair of scores per
  // section (two exponentials, one bf16 pair, their sum).  Q is pre-scaled
  // by scale * log2(e) and every S accumulation starts from -m (negm), so the
  // exponent argument comes out of the MFMAs.  The running max m does not
  // move on the common path: a lane's block sum above kSumLimit (some P above
  // 2^8) sends the wave to rescale(), which moves m by the block max where
  // that exceeds kLazy.  Otherwise every P = exp2(s - m) <= 2^12, which fp32
  // O and l absorb.  Row maxima use v_maximum3 (NaN-propagating).
  // A query whose scores have all been -inf has no maximum yet: its m stays 0, its
  // P and l are 0, and as long as a wave holds one, limit is below every sum, so
  // that rescale() sees each block and takes the first finite maximum as it is,
  // downwards too.
  static constexpr float kLazy = 8.0f;
  static constexpr float kSumLimit = 4096.0f;
  float rsum_;

  __device__ __forceinline__ static float max16(const f32x16& c) {
    const float a = __builtin_elementwise_maximum(__builtin_elementwise_maximum(c[0], c[1]), c[2]);
    const float b = __builtin_elementwise_maximum(__builtin_elementwise_maximum(c[3], c[4]), c[5]);
    const float d = __builtin_elementwise_maximum(__builtin_elementwise_maximum(c[6], c[7]), c[8]);
    const float e = __builtin_elementwise_maximum(__builtin_elementwise_maximum(c[9], c[10]), c[11]);
    const float f = __builtin_elementwise_maximum(__builtin_elementwise_maximum(c[12], c[13]), c[14]);
    const float g = __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), d);
    const float hh = __builtin_elementwise_maximum(__builtin_elementwise_maximum(e, f), c[15]);
    return __builtin_elementwise_maximum(g, hh);
  }

  // exponentials of S values 2g, 2g + 1 into one P dword.  The empty asm
  // keeps the bf16 packing in this section: left alone the compiler sinks it
  // into the next step, in front of that step's first LDS reads.  (Summing
  // the bf16 pair with v_dot2c_f32_bf16 instead of two adds measured 4%
  // slower.)
  template <int PAR, int g>
  __device__ __forceinline__ void expo2() {
    const float e0 = __builtin_amdgcn_exp2f(sv[2 * g]);
    const float e1 = __builtin_amdgcn_exp2f(sv[2 * g + 1]);
    uint32_t c = pk_bf16(e0, e1);
    asm volatile("" : "+v"(c));
    pw[PAR][g >> 2][g & 3] = c;
    rsum_ = g == 0 ? e0 + e1 : rsum_ + (e0 + e1);
  }

  // (readfirstlane: in a scalar register, which the check's compare takes for free)
  __device__ __forceinline__ void set_limit(bool every_block) {
    limit = __int_as_float(__builtin_amdgcn_readfirstlane(
        __float_as_int(every_block ? -1.0f : kSumLimit)));
  }

  // The rare path for P(i - 1) (its scores in sp): move m by the block max d
  // where that exceeds kLazy, recompute P(i - 1), scale O (blocks <= i - 2)
  // and l by 2^-d, shift S(i) (accumulated from the old -m, now in sv) and
  // the start value of the next accumulation.  The updates of O, S and -m
  // are inline asm with tied operands: written as C++, they made the compiler
  // keep a second copy of those registers across the branch (256 VGPRs and
  // spills in the main loop, against 214).  The asm is invisible to the
  // compiler's hazard tracking, so the wait states are explicit: the MFMA
  // results it reads were written before the ~40 VALU instructions above it,
  // and the s_nop after it precedes any MFMA that reads what it wrote.
  template <int PAR, bool SHIFT_S>
  __device__ __forceinline__ void rescale(const f32x16& sp) {
    // SHIFT_S: S(i) was accumulated from the old -m (main steps); otherwise
    // S(i) is a new block's raw first block or absent, and -m is reset
    const float bm = xor32_max(max16(sp));
    const bool unset = xor32_add(l) == 0.0f;  // no score above -inf so far: O is 0 too
    const bool none = bm == -INFINITY;
    const float d = unset ? (none ? 0.0f : bm) : bm > kLazy ? bm : 0.0f;
    const float alpha = unset ? 1.0f : __builtin_amdgcn_exp2f(-d);
    set_limit(__any(unset && none));
    m += d;
    float rs = 0.0f;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const float e0 = __builtin_amdgcn_exp2f(sp[2 * g] - d);
      const float e1 = __builtin_amdgcn_exp2f(sp[2 * g + 1] - d);
      pw[PAR][g >> 2][g & 3] = pk_bf16(e0, e1);
      rs += e0 + e1;
    }
    rsum_ = rs;
    l *= alpha;
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7");
#pragma unroll
    for (int j = 0; j < ND; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) asm volatile("v_mul_f32 %0, %1, %0" : "+v"(o[j][r]) : "v"(alpha));
    if constexpr (SHIFT_S) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        asm volatile("v_sub_f32 %0, %0, %1" : "+v"(sv[r]) : "v"(d));
        asm volatile("v_mov_b32 %0, %1" : "+v"(negm[r]) : "v"(-m));
      }
    }
    asm volatile("s_nop 7");
  }

  // VALU slots of a section (for the interleave below)
  static constexpr int kSectionValu[8] = {5, 4, 4, 4, 4, 4, 4, 4};

  // ---- the workgroup's sequence of query blocks (persistent grid) ----
  int G, g, nblk, nqb;
  float l_prev;
  __device__ __forceinline__ int perm() const {
    return G % 8 == 0 ? (g % 8) * (G / 8) + g / 8 : g;
  }
  __device__ __forceinline__ void block(int jb, int64_t& base, int& qb) const {
    const int L = jb * G + perm();
    const int bh = L / nqb;
    qb = L - bh * nqb;
    base = static_cast<int64_t>(bh) * p.S * D;
  }

  // Q rows of a block into the wave's staging buffer (swizzled like K),
  // 8 DMA instructions per wave; read back by the same wave only
  __device__ __forceinline__ void stage_q(int64_t base, int qb) {
    if (qb < 0) return;  // no next block
    const int64_t row0 = static_cast<int64_t>(qb) * W8_BQ + 32 * wave;
#pragma unroll
    for (int ins = 0; ins < 8; ++ins) {
      const int r = 4 * ins + (lane >> 4), pc = lane & 15;
      const int src = r * D + ((pc ^ (r & 15)) << 3);
      const uint64_t gq = reinterpret_cast<uint64_t>(p.Q + base + row0 * D);
      const uint64_t gs =
          (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(gq >> 32)))) << 32) |
          uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(gq))));
      const uint32_t buf = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
          (lds_void*)(w8Q[wave] + ins * 512)));
      asm volatile(
          "s_mov_b32 m0, %0\n\t"
          "s_nop 0\n\t"
          "global_load_lds_dwordx4 %1, %2"
          :
          : "s"(__builtin_amdgcn_readfirstlane(buf)), "v"(static_cast<uint32_t>(src) * 2u),
            "s"(gs)
          : "memory", "m0");
    }
  }
  __device__ __forceinline__ void scale_q(const bf16x8 (&x)[NDC]) {
#pragma unroll
    for (int dc = 0; dc < NDC; ++dc)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        qop[dc][e] = static_cast<__bf16>(static_cast<float>(x[dc][e]) * p.scale_log2);
  }

  // O / l of a finished block into its rows: O[q][d], d = 32j + 8u + 4h + i
  __device__ __forceinline__ void store_o(int64_t base, int qb, float lsum) {
    const float inv = 1.0f / xor32_add(lsum);
    const int64_t q = static_cast<int64_t>(qb) * W8_BQ + 32 * wave + l32;
    uint16_t* orow = p.O + base + q * D;
#pragma unroll
    for (int j = 0; j < ND; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int d = 32 * j + 8 * u + 4 * h;
        const u32x2 v = {pk_bf16(o[j][4 * u] * inv, o[j][4 * u + 1] * inv),
                         pk_bf16(o[j][4 * u + 2] * inv, o[j][4 * u + 3] * inv)};
        *reinterpret_cast<u32x2*>(orow + d) = v;
      }
  }

  // one step at global step t (PAR = t % 2, KB = t % 4): S(t) = K(t) Q^T into
  // s (renamed to sv at the end), the softmax of sv into pw[PAR ^ 1], and
  // O += V(t - 2) P(t - 2) with P(t - 2) in pw[PAR]; K(t) in K buffer KB,
  // V(t - 2) in V buffer (KB + 2) % 4.  Flags:
  //   NEXT_S / NEXT_O  the next step computes S / O (its first fragments are
  //                    read at the end of this step, before the barrier);
  //   OZERO            O starts from zero (a block's first O step);
  //   SZERO            S starts from zero (a block's first KV step);
  //   CHECK / SHIFT    the rare-path check; whether it also shifts S(t), -m;
  //   QPF              also stage the next block's Q (8 more loads);
  //   QSW              at the end, load the next block's Q into qop.
  //   kb, kk / vb, vk: base and KV step of the K / V block this step loads
  //                    (K of step t + 3, V of step t + 1, possibly of the
  //                    next block)
  template <int PAR, int KB, bool DO_S, bool DO_SM, bool DO_O, bool NEXT_S, bool NEXT_O,
            bool OZERO, bool SZERO, bool CHECK, bool SHIFT, bool QPF = false, bool QSW = false>
  __device__ __forceinline__ void step(int64_t kb, int kk, int64_t vb, int vk,
                                       int64_t nq_base = 0, int nq_qb = 0) {
    const uint16_t* Kc = w8_kbuf<KB>();
    const uint16_t* Vc = w8_vbuf<(KB + 2) % 4>();
    const f32x16 sp = sv;  // S(t - 1) - m, for the rare path
    bf16x8 kf[8], vf[8];
    auto issue = [&](auto xc) {
      constexpr int x = decltype(xc)::value;
      if constexpr (DO_S) kf[x] = kfrag(Kc, x);
      if constexpr (DO_O) vf[x] = vfrag(Vc, x >> 1, x & 1);
    };
    if constexpr (DO_S) { kf[0] = kpf[0]; kf[1] = kpf[1]; }
    if constexpr (DO_O) { vf[0] = vpf[0]; vf[1] = vpf[1]; }
    if constexpr (DO_S) {
      dma(p.K, kb, k_src, kk * W8_KV, w8_kbuf<(KB + 3) % 4>());
      dma(p.V, vb, v_src, vk * W8_KV, w8_vbuf<(KB + 1) % 4>());
    }
    if constexpr (QPF) stage_q(nq_base, nq_qb);
    __builtin_amdgcn_sched_barrier(0);
    sd_static_for<8>([&](auto xc) {
      constexpr int x = decltype(xc)::value;
      if constexpr (x == 0) __builtin_amdgcn_s_setprio(1);
      if constexpr (x == 6) __builtin_amdgcn_s_setprio(0);
      if constexpr (DO_S) {
        const f32x16 z = {};
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[x], qop[x],
                                                    x == 0 ? (SZERO ? z : negm) : s, 0, 0, 0);
      }
      if constexpr (DO_O) {
        const f32x16 z = {};
        o[x >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            vf[x], __builtin_bit_cast(bf16x8, pw[PAR][x & 1]),
            (OZERO && (x & 1) == 0) ? z : o[x >> 1], 0, 0, 0);
      }
      if constexpr (x + 2 < 8) issue(std::integral_constant<int, x + 2>());
      if constexpr (DO_SM) expo2<PAR ^ 1, x>();
      if constexpr (DO_S && x == 7) sv = s;  // the next step's softmax reads S(t)
      constexpr int nm = (DO_S ? 1 : 0) + (DO_O ? 1 : 0);
      constexpr int nv = DO_SM ? (kSectionValu[x] + nm - 1) / nm : 0;
      sd_static_for<nm>([&](auto) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
        __builtin_amdgcn_sched_group_barrier(0x402, nv, 0); // its share of VALU
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (DO_SM) {
      if constexpr (CHECK) {
        if (__builtin_expect(__any(rsum_ > limit), 0)) rescale<PAR ^ 1, SHIFT>(sp);
      }
      l += rsum_;
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (QSW) {
      bf16x8 x[NDC];
#pragma unroll
      for (int dc = 0; dc < NDC; ++dc) x[dc] = kfrag(w8Q[wave], dc);
      scale_q(x);
    }
    // the next step's first fragments: K(t + 1) and V(t - 1), published at
    // the previous barrier (their loads were issued two steps ago)
    if constexpr (NEXT_S) {
      kpf[0] = kfrag(w8_kbuf<(KB + 1) % 4>(), 0);
      kpf[1] = kfrag(w8_kbuf<(KB + 1) % 4>(), 1);
    }
    if constexpr (NEXT_O) {
      vpf[0] = vfrag(w8_vbuf<(KB + 3) % 4>(), 0, 0);
      vpf[1] = vfrag(w8_vbuf<(KB + 3) % 4>(), 0, 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    // the previous step's loads landed (this step's may stay in flight), this
    // step's reads are done except the prefetch: publish / release
    // The count covers exactly the loads this step issued: a QPF step whose
    // block has no next block stages no Q (stage_q returns), and allowing 8
    // more would leave the previous step's K / V loads unwaited, which the
    // next step's fragment prefetch reads.
    constexpr int npf = (NEXT_S ? 2 : 0) + (NEXT_O ? 4 : 0);
    constexpr int nvm = DO_S ? 2 : 0;
    constexpr int nvq = nvm + (QPF ? 8 : 0);
    if (QPF && nq_qb >= 0)
      __builtin_amdgcn_s_waitcnt((nvq & 15) | ((nvq >> 4) << 14) | 0x0070 | (npf << 8));
    else
      __builtin_amdgcn_s_waitcnt((nvm & 15) | ((nvm >> 4) << 14) | 0x0070 | (npf << 8));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }

  // a block's S(0) (raw) is in sv: m = its maximum (0 if that is -inf), S(0) and
  // -m rebased
  __device__ __forceinline__ void start_block() {
    m = xor32_max(max16(sv));
    const bool unset = m == -INFINITY;
    set_limit(__any(unset));
    m = unset ? 0.0f : m;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sv[r] -= m;
      negm[r] = -m;
    }
  }
};

// Block jb of workgroup g is query block jb * G + perm(g): perm puts the
// workgroups of one XCD (g % 8 under round-robin dispatch) on consecutive
// blocks, so at any time an XCD works on the query blocks of one or two heads
// and its L2 serves their K / V to all of them.
__global__ __launch_bounds__(W8_THREADS, 1) void sdpa_w8_kernel(const SdpaArgs p) {
  SdpaW8 w{p};
  w.lane = threadIdx.x & 63;
  w.wave = threadIdx.x >> 6;
  w.l32 = w.lane & 31;
  w.h = w.lane >> 5;
  w.n = p.S / W8_KV;
  w.nqb = p.nqb;
  w.G = gridDim.x;
  w.g = blockIdx.x;
  const int total = p.nbh * p.nqb;
  w.nblk = (total - w.perm() + w.G - 1) / w.G;
  w.l = 0.0f;
  w.setup();
  const int n = w.n;  // >= 8, a multiple of 8
  int64_t cur_base;
  int cur_qb;
  w.block(0, cur_base, cur_qb);
  {
    bf16x8 x[SdpaW8::NDC];
    const int64_t q = static_cast<int64_t>(cur_qb) * W8_BQ + 32 * w.wave + w.l32;
#pragma unroll
    for (int dc = 0; dc < SdpaW8::NDC; ++dc)
      x[dc] = *reinterpret_cast<const bf16x8*>(p.Q + cur_base + q * W8_D + dc * 16 + 8 * w.h);
    w.scale_q(x);
  }
  // K(0), K(1), K(2) and V(0) of block 0 (with Q landed), then the pipeline
  w.dma(p.K, cur_base, w.k_src, 0, w8_kbuf<0>());
  w.dma(p.K, cur_base, w.k_src, W8_KV, w8_kbuf<1>());
  w.dma(p.K, cur_base, w.k_src, 2 * W8_KV, w8_kbuf<2>());
  w.dma(p.V, cur_base, w.v_src, 0, w8_vbuf<0>());
  __builtin_amdgcn_s_waitcnt(0x0070);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  w.kpf[0] = w.kfrag(w8_kbuf<0>(), 0);
  w.kpf[1] = w.kfrag(w8_kbuf<0>(), 1);
  //          PAR KB S  SM O  NS NO OZ SZ CK SH
  w.step<0, 0, 1, 0, 0, 1, 0, 0, 1, 0, 0>(cur_base, 3, cur_base, 1);
  w.start_block();
  w.step<1, 1, 1, 1, 0, 1, 1, 0, 0, 0, 0>(cur_base, 4, cur_base, 2);
  // one path per block: steps 2 .. n - 1 of block jb, then the next block's
  // steps 0 and 1, which also finish block jb (its last softmax and O
  // products) before its O is stored.  After the last block the "next"
  // block's steps run for nothing: their loads repeat the last block's last
  // K / V rows (still in L2), nothing reads them, and no Q is staged.
  for (int jb = 0;; ++jb) {
    const int64_t cb = cur_base;
    w.step<0, 2, 1, 1, 1, 1, 1, 1, 0, 1, 1>(cb, 5, cb, 3);
    w.step<1, 3, 1, 1, 1, 1, 1, 0, 0, 1, 1>(cb, 6, cb, 4);
    for (int i = 4; i + 4 < n; i += 4) {
      w.step<0, 0, 1, 1, 1, 1, 1, 0, 0, 1, 1>(cb, i + 3, cb, i + 1);
      w.step<1, 1, 1, 1, 1, 1, 1, 0, 0, 1, 1>(cb, i + 4, cb, i + 2);
      w.step<0, 2, 1, 1, 1, 1, 1, 0, 0, 1, 1>(cb, i + 5, cb, i + 3);
      w.step<1, 3, 1, 1, 1, 1, 1, 0, 0, 1, 1>(cb, i + 6, cb, i + 4);
    }
    const bool last = jb + 1 == w.nblk;
    int64_t nb = cb;
    int nq = -1;
    if (!last) w.block(jb + 1, nb, nq);
    const auto nk = [&](int k) { return last ? n - 1 : k; };  // KV step of the next block
    // steps n - 4 .. n - 1: the next block's first K / V blocks, its Q staged
    // and then loaded into qop
    w.step<0, 0, 1, 1, 1, 1, 1, 0, 0, 1, 1, true, false>(cb, n - 1, cb, n - 3, nb, nq);
    w.step<1, 1, 1, 1, 1, 1, 1, 0, 0, 1, 1>(nb, nk(0), cb, n - 2);
    w.step<0, 2, 1, 1, 1, 1, 1, 0, 0, 1, 1>(nb, nk(1), cb, n - 1);
    w.step<1, 3, 1, 1, 1, 1, 1, 0, 0, 1, 1, false, true>(nb, nk(2), nb, nk(0));
    // the next block's steps 0 and 1 with this block's last softmax / O
    w.step<0, 0, 1, 1, 1, 1, 1, 0, 1, 1, 0>(nb, nk(3), nb, nk(1));
    w.l_prev = w.l;
    w.l = 0.0f;
    w.start_block();
    w.step<1, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0>(nb, nk(4), nb, nk(2));
    w.store_o(cb, cur_qb, w.l_prev);
    if (last) break;
    cur_base = nb;
    cur_qb = nq;
  }
  // the unused loads of the last block's "next" block land before the end
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
}

// The kernel for `blocks` blocks of 128 queries.
int form_of(int64_t blocks, int64_t S, int64_t D, bool causal) {
  // (256 blocks of 128 queries and fewer leave sdpa_w8_kernel half the CUs:
  // 1 x 8 x 2048 x 128 46.6 us against 40 to 42 in sdpa_fwd_kernel)
  if (D == W8_D && !causal && S % W8_BQ == 0 && blocks > 256) return TTLH_SDPA_EIGHT_WAVES;
  // Two groups of waves: up to one workgroup per CU, and under the causal mask
  // up to two rounds of long blocks, whose shares of a CU would differ most (512
  // blocks of S = 2016: 62 us against 69; of S = 480: 28 against 24; 384
  // blocks without the mask: 84 against 72).  Three KV blocks do not pay for
  // the second group.
  return S > 192 && (blocks <= 256 || (causal && blocks <= 512 && S >= 1024))
             ? TTLH_SDPA_TWO_GROUPS
             : TTLH_SDPA_ONE_GROUP;
}

template <int D, bool CAUSAL>
int launch(SdpaArgs a, hipStream_t s) {
  // heads dispatched together: a divisor of an XCD's share of the heads whose
  // K and V (2 x 2 S D bytes a head) fit its 4 MiB L2
  const int share = a.nbh % 8 == 0 ? a.nbh / 8 : 1;
  const int64_t fit = (int64_t(4) << 20) / (int64_t(4) * a.S * D);
  a.heads_together = 1;
  for (int g = 1; g <= share && g <= fit; ++g)
    if (share % g == 0) a.heads_together = g;
  const int form = form_of(static_cast<int64_t>(a.nbh) * a.nqb, a.S, D, CAUSAL);
  if (form == TTLH_SDPA_EIGHT_WAVES) {
    SdpaArgs b = a;
    b.nqb = a.S / W8_BQ;
    // persistent: one workgroup per CU (at most), each walking its blocks
    int dev = 0, cus = 0;
    TTLH_HIP_CHECK(hipGetDevice(&dev));
    TTLH_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    TTLH_REQUIRE(cus > 0, TTLH_EHIP, "ttlh_sdpa_fwd: the device reports no CUs");
    const int64_t total = static_cast<int64_t>(b.nbh) * b.nqb;
    const int grid = static_cast<int>(total < cus ? total : cus);
    hipLaunchKernelGGL(sdpa_w8_kernel, dim3(grid), dim3(W8_THREADS), 0, s, b);
    return check_launch("sdpa_w8_kernel");
  }
  const bool two = form == TTLH_SDPA_TWO_GROUPS;
  const dim3 grid(static_cast<uint32_t>(static_cast<int64_t>(a.nbh) * a.nqb));
  const bool ragged = a.S % BQ != 0;  // S % 32 == 0 only
  if (two && ragged)
    hipLaunchKernelGGL((sdpa_fwd_kernel<D, CAUSAL, true, 2>), grid, dim3(2 * kThreads), 0, s, a);
  else if (two)
    hipLaunchKernelGGL((sdpa_fwd_kernel<D, CAUSAL, false, 2>), grid, dim3(2 * kThreads), 0, s, a);
  else if (ragged)
    hipLaunchKernelGGL((sdpa_fwd_kernel<D, CAUSAL, true, 1>), grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((sdpa_fwd_kernel<D, CAUSAL, false, 1>), grid, dim3(kThreads), 0, s, a);
  return check_launch("sdpa_fwd_kernel");
}

}  // namespace
}  // namespace ttlh

using namespace ttlh;

extern "C" int ttlh_sdpa_fwd(const void* Q, const void* K, const void* V, void* O, int64_t B,
                             int64_t H, int64_t S, int64_t D, float scale, int causal,
                             void* stream) {
  clear_error();
  TTLH_REQUIRE(Q && K && V && O, TTLH_EINVAL, "ttlh_sdpa_fwd: null pointer");
  TTLH_REQUIRE(B > 0 && H > 0 && S > 0, TTLH_EINVAL, "ttlh_sdpa_fwd: empty problem");
  TTLH_REQUIRE(D == 64 || D == 128, TTLH_EUNSUPPORTED, "ttlh_sdpa_fwd: head_dim must be 64 or 128");
  TTLH_REQUIRE(S % 32 == 0, TTLH_EUNSUPPORTED, "ttlh_sdpa_fwd: seq_len must be a multiple of 32");
  TTLH_REQUIRE(B * H * ((S + BQ - 1) / BQ) < (int64_t(1) << 31), TTLH_EUNSUPPORTED,
               "ttlh_sdpa_fwd: too many query blocks");
  TTLH_REQUIRE(S * D < (int64_t(1) << 31), TTLH_EUNSUPPORTED, "ttlh_sdpa_fwd: seq_len too long");
  for (const void* ptr : {Q, K, V, static_cast<const void*>(O)})
    TTLH_REQUIRE((reinterpret_cast<uintptr_t>(ptr) & 15) == 0, TTLH_EINVAL,
                 "ttlh_sdpa_fwd: tensors must be 16-byte aligned");
  TTLH_REQUIRE(std::isfinite(scale), TTLH_EINVAL, "ttlh_sdpa_fwd: scale must be finite");
  SdpaArgs a;
  a.Q = static_cast<const uint16_t*>(Q);
  a.K = static_cast<const uint16_t*>(K);
  a.V = static_cast<const uint16_t*>(V);
  a.O = static_cast<uint16_t*>(O);
  a.S = static_cast<int32_t>(S);
  a.nqb = static_cast<int32_t>((S + BQ - 1) / BQ);
  a.nbh = static_cast<int32_t>(B * H);
  a.scale_log2 = scale * 1.4426950408889634f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (D == 128) return causal ? launch<128, true>(a, s) : launch<128, false>(a, s);
  return causal ? launch<64, true>(a, s) : launch<64, false>(a, s);
}

extern "C" int ttlh_sdpa_fwd_form(int64_t B, int64_t H, int64_t S, int64_t D, int causal) {
  return form_of(B * H * ((S + BQ - 1) / BQ), S, D, causal != 0);
}
