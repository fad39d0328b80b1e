// Fused online-softmax attention forward for fp32 inputs on the bf16 matrix core, with fp32's
// accuracy (the `fused` entry's fp32 inputs on grids that fill the chip; fa_f32.hpp takes the rest).
//
// The fp32 matrix core bounds fa_f32.hpp: 64 FLOP per cycle and SIMD against the bf16 one's 1024.
// Here every fp32 operand (Q, K, V and P) is split into three bf16 terms h + m + l, whose sum has
// more than fp32's 24 bits (an operand below 2^-112 keeps an absolute 2^-134) and whose range is
// fp32's, and a product takes the six term products down to 2^-18 of it (h h; h m, m h; m m, h l,
// l h), which leaves out less than 2^-25. They are exact in the fp32 accumulator. That is
// 1024 / 6 / 64 = 2.7x the fp32 matrix core's rate, and a smaller error: the five small products have
// an accumulator of their own, so O's main chain rounds once per 16 keys, not per 2. Against
// float64 (2-norms; fa_f32.hpp -> here): 4x16x512 3.6e-7 -> 2.2e-7, 4x16x2048 5.2e-7 -> 3.6e-7,
// 4x4x8192 8.8e-7 -> 6.4e-7, causal 4x4x8000 3.8e-7 -> 2.8e-7, 2x4x4000 with Q, K x3 1.5e-6 -> 6.0e-7.
//
// Otherwise the fused kernels' scheme (fa_mfma.hpp): S^T = K Q^T and O^T += V^T P^T, a wave owning 32
// queries, P^T straight from the S^T accumulator, m raised lazily. A workgroup stages 32-key tiles:
// a thread loads 8 dims of a K and of a V row a tile ahead, splits them once for its four query waves
// and writes the three planes to LDS (two stages, one barrier per tile). KS == 2: two key groups of
// four query waves walk alternate tiles and are merged at the end, which gives a CU its two waves per
// SIMD from one workgroup.
//
// Measured, us a call: 4x16x2048 607 -> 393 (113 -> 175 TFLOP/s), 4x16x4096 2320 -> 1475 (186), causal
// 4x16x1024 114 -> 62, 2x4x4000 293 -> 179. At those sizes the six products run at ~1.1 PFLOP/s of bf16
// matrix work, about what a large bf16 product reaches under the card's power cap. Counters at
// 4x16x2048: matrix core busy 52 % of the cycles, VALU 58 %, a VALU instruction beside 35 % of the MFMA
// cycles; interleaving the staging with the products by scheduling groups, or a raised wave priority
// for them, moved nothing (within 1 %), three waves per SIMD spill (146 VGPRs, 8 % slower), and
// keeping each wave's own tiles in registers (no LDS, as fa_f32.hpp) loses 5 % to fa_f32.hpp because
// every wave then splits its operands itself.
// Two fp16 terms per operand (three products) are a third faster still, but hold neither a small column
// of V beside ordinary ones nor fp32's range: below 2^-20 a value of V keeps an absolute 2^-44, a product is off by
// up to 2^-21, and a check of every element sends a tenth of N(0, 1) heads of 2048 keys to wider terms.
#pragma once

#include "common.hpp"
#include "fa_mfma.hpp"   // k_swz, v_swz: the K and V tile layouts

namespace pa {

// x = h + m + l in bf16, each term the rounding of what the ones before it leave: 24 significant
// bits and more, over fp32's exponent range.
struct Bf3 {
  bf16x8 h, m, l;
};
__device__ __forceinline__ Bf3 split3(const float (&x)[8]) {
  Bf3 t;
  float r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) t.h[j] = (bf16)x[j];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = x[j] - (float)t.h[j];
#pragma unroll
  for (int j = 0; j < 8; ++j) t.m[j] = (bf16)r[j];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] -= (float)t.m[j];
#pragma unroll
  for (int j = 0; j < 8; ++j) t.l[j] = (bf16)r[j];
  return t;
}
// split3 of values that may lie past the largest float that rounds to a finite bf16 (a rare,
// wave-uniform branch): a finite one takes its truncation as h, an infinite one has h alone.
__device__ __forceinline__ Bf3 split3_checked(const float (&x)[8]) {
  constexpr float kBf16Max = 3.38953139e38f;
  Bf3 t = split3(x);
  float mx = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(x[j]));
  if (__builtin_amdgcn_ballot_w64(mx > kBf16Max) != 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (fabsf(x[j]) > kBf16Max) {
        const float h = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[j]) & 0xffff0000u);
        const float r = __builtin_isinf(x[j]) ? 0.f : x[j] - h;
        t.h[j] = (bf16)h;
        t.m[j] = (bf16)r;
        t.l[j] = (bf16)(r - (float)t.m[j]);
      }
  }
  return t;
}
// hi += a.h b.h, lo += the five products of the next two orders; what is left out (m l, l m, l l)
// is below 2^-25 of a b.
__device__ __forceinline__ void mfma_bf3(const Bf3& a, const Bf3& b, f32x16& hi, f32x16& lo) {
  lo = mfma32x32x16(a.l, b.h, lo);
  lo = mfma32x32x16(a.h, b.l, lo);
  lo = mfma32x32x16(a.m, b.m, lo);
  lo = mfma32x32x16(a.m, b.h, lo);
  lo = mfma32x32x16(a.h, b.m, lo);
  hi = mfma32x32x16(a.h, b.h, hi);
}
// hi + lo. Where an operand was infinite, hi has the product's value (infinite or NaN) and lo may be
// a NaN; the median is then one of the finite bounds, and hi stays what it is.
__device__ __forceinline__ float join_bf3(float hi, float lo) {
  return hi + __builtin_amdgcn_fmed3f(lo, -3.4e38f, 3.4e38f);
}

template <int D, int NQ, int KS>
__global__ void __launch_bounds__(NQ * KS * kWave)
__attribute__((amdgpu_waves_per_eu(2)))
fa_f32x3_fwd(const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
             float* __restrict__ O, int N, int num_qblocks, int total_blocks, float scale_log2, int causal) {
  constexpr int BM = NQ * 32, BN = 32;
  constexpr int CR = D / 8, RB = D * 2, PLANE = BN * RB, MAT = 3 * PLANE;   // bf16 planes of a tile
  constexpr int STEPS = D / 16, NDB = D / 32;
  constexpr int CPT = BN * CR / (NQ * kWave);   // 8-dim chunks of K and of V per thread and tile
  // m is set to a row's max plus kLazyLog2 and raised again only when the max has passed it, so
  // P = 2^(s c - m) stays at most 1, a row's largest between 2^-8 and 1: no single product P V overflows
  // where V does not, and a row's sum of them later than with m at the max.
  constexpr float kLazyLog2 = 8.f;
  static_assert(D == 64 && CPT * NQ * kWave == BN * CR, "whole chunks per thread");
  __shared__ __attribute__((aligned(1024))) unsigned char k_lds0[KS * MAT], v_lds0[KS * MAT], k_lds1[KS * MAT], v_lds1[KS * MAT];
  __shared__ float red_ml[KS > 1 ? (KS - 1) * NQ * 2 * kWave : 1];
  const int g = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / (NQ * kWave));   // key group
  const int tid = (int)threadIdx.x % (NQ * kWave), lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lq = lane % 32, hi = lane / 32;

  int bh, qb;
  if (causal) {   // the longest blocks of every head first; with B*H a multiple of 8 a head keeps its XCD
    const int heads = total_blocks / num_qblocks;
    qb = num_qblocks - 1 - (int)blockIdx.x / heads;
    bh = (int)blockIdx.x % heads;
  } else {
    const int blk = xcd_remap(blockIdx.x, total_blocks);
    bh = blk / num_qblocks;
    qb = blk % num_qblocks;
  }
  const int q0 = qb * BM, q0w = q0 + wave * 32, qrow = q0w + lq;
  const size_t base = (size_t)bh * N * D;
  const uint32_t head_bytes = (uint32_t)((size_t)N * D * 4);
  const rsrc_t q_rs = make_rsrc(Q + base, head_bytes);
  const rsrc_t k_rs = make_rsrc(K + base, head_bytes);
  const rsrc_t v_rs = make_rsrc(V + base, head_bytes);

  // (Loaded vectors are bit-cast as a whole before their elements are taken.)
  auto load8 = [](rsrc_t rs, uint32_t off, float (&x)[8]) __attribute__((always_inline)) {
    const f32x4 a = __builtin_bit_cast(f32x4, load16(rs, off)), b = __builtin_bit_cast(f32x4, load16(rs, off + 16));
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = a[j], x[4 + j] = b[j];
  };

  // Q^T operand terms: dims 16 kk + 8 hi .. + 7 of row qrow (rows past N read as zero).
  Bf3 qf[STEPS];
#pragma unroll
  for (int kk = 0; kk < STEPS; ++kk) {
    float x[8];
    load8(q_rs, (uint32_t)((qrow * D + 16 * kk + 8 * hi) * 4), x);
    qf[kk] = split3_checked(x);
  }

  // Staging: a thread carries CPT chunks of its key group's K and V tiles, global to registers one
  // tile ahead, then split into the planes. Key group g's iteration j is tile j KS + g.
  uint32_t src[CPT];
  int k_dst[CPT], v_dst[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int slot = i * NQ * kWave + tid, row = slot / CR, ch = slot % CR;
    src[i] = (uint32_t)((row * D + ch * 8) * 4);
    k_dst[i] = g * MAT + row * RB + ((ch ^ k_swz<CR>(row)) * 16);
    v_dst[i] = g * MAT + row * RB + ((ch ^ v_swz<CR>(row)) * 16);
  }
  float kx[CPT][8], vx[CPT][8];
  auto gload = [&](int j) __attribute__((always_inline)) {
    const uint32_t off = (uint32_t)((j * KS + g) * BN * D * 4);
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      load8(k_rs, src[i] + off, kx[i]);
      load8(v_rs, src[i] + off, vx[i]);
    }
  };
  auto stage = [&](unsigned char* ks, unsigned char* vs) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const Bf3 a = split3_checked(kx[i]);
      *reinterpret_cast<bf16x8*>(ks + k_dst[i]) = a.h;
      *reinterpret_cast<bf16x8*>(ks + PLANE + k_dst[i]) = a.m;
      *reinterpret_cast<bf16x8*>(ks + 2 * PLANE + k_dst[i]) = a.l;
      const Bf3 b = split3_checked(vx[i]);
      *reinterpret_cast<bf16x8*>(vs + v_dst[i]) = b.h;
      *reinterpret_cast<bf16x8*>(vs + PLANE + v_dst[i]) = b.m;
      *reinterpret_cast<bf16x8*>(vs + 2 * PLANE + v_dst[i]) = b.l;
    }
  };

  // Operand addresses within a plane, as in fa_mfma.hpp: K row lq, chunk 2 kk + hi; V transposed.
  int k_addr[STEPS];
#pragma unroll
  for (int kk = 0; kk < STEPS; ++kk) k_addr[kk] = g * MAT + lq * RB + (((2 * kk + hi) ^ k_swz<CR>(lq)) * 16);
  const int g16 = lane / 16, i16 = lane % 16;
  const int v_row = hi * 4 + i16 / 4;
  const int v_cl = 2 * (g16 % 2) + (i16 % 4) / 2;
  int v_addr[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
    v_addr[db] = g * MAT + v_row * RB + (((4 * db + v_cl) ^ v_swz<CR>(v_row)) * 16) + 8 * (i16 % 2);

  float m_run = -INFINITY, l_run = 0.f;
  f32x16 oh[NDB], ol[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) oh[db] = f32x16{}, ol[db] = f32x16{};

  const int kv_end = causal ? min(N, q0 + BM) : N;
  const int ntiles = (kv_end + BN - 1) / BN;
  const int nit = (ntiles + KS - 1) / KS;
  const int wave_tiles = causal ? min(ntiles, q0w / BN + 1) : ntiles;    // tiles this wave's rows see
  const int clean_tiles = causal ? min(N / BN, q0w / BN) : N / BN;       // of these, without a mask

  auto compute = [&](const unsigned char* ks, const unsigned char* vs, int t) __attribute__((always_inline)) {
    f32x16 sh = f32x16{}, sl = f32x16{};
#pragma unroll
    for (int kk = 0; kk < STEPS; ++kk) {
      Bf3 a;
      a.h = *reinterpret_cast<const bf16x8*>(ks + k_addr[kk]);
      a.m = *reinterpret_cast<const bf16x8*>(ks + PLANE + k_addr[kk]);
      a.l = *reinterpret_cast<const bf16x8*>(ks + 2 * PLANE + k_addr[kk]);
      mfma_bf3(a, qf[kk], sh, sl);
    }
    float s[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = join_bf3(sh[r], sl[r]);
    if (t >= clean_tiles) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = t * BN + 8 * (r / 4) + 4 * hi + r % 4;
        if (key >= N || (causal && key > qrow)) s[r] = -INFINITY;
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    // (A row is raised for its own max alone: causal rows' bits do not depend on later tokens.)
    const float m_new = fmaxf(m_run, fmaf(half_max(mx), scale_log2, kLazyLog2));
    const bool raise = m_new > m_run + kLazyLog2;
    if (__builtin_amdgcn_ballot_w64(raise) != 0) {
      const float alpha = raise ? exp2_fast(m_run - m_new) : 1.f;   // m_run = -inf -> 0
      m_run = raise ? m_new : m_run;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db) oh[db] *= alpha, ol[db] *= alpha;
    }
    const float nm = m_run == -INFINITY ? 0.f : -m_run;   // no visible key so far: P = 0
    float p[2][8];
    float sum[2] = {0.f, 0.f};                            // the tile's sum first, then one add to l
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      p[r / 8][r % 8] = exp2_fast(fmaf(s[r], scale_log2, nm));
      sum[r % 2] += p[r / 8][r % 8];
    }
    l_run += sum[0] + sum[1];
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2) {
      const Bf3 pf = split3(p[k2]);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        bf16x8 a[3];
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) {
          const unsigned char* p0 = vs + pl * PLANE + k2 * 16 * RB + v_addr[db];
          const i16x4 a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<i16x4>)(p0));
          const i16x4 a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<i16x4>)(p0 + 8 * RB));
          a[pl] = __builtin_bit_cast(bf16x8, i16x8{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]});
        }
        mfma_bf3(Bf3{a[0], a[1], a[2]}, pf, oh[db], ol[db]);
      }
    }
  };

  // Tile j + 1 is staged, and tile j + 2 loaded, before tile j's products; one barrier per tile
  // (offsets past the head load zeros).
  gload(0);
  stage(k_lds0, v_lds0);
  gload(1);
  __syncthreads();
  for (int j = 0; j < nit; j += 2) {
    stage(k_lds1, v_lds1);
    gload(j + 2);
    if (j * KS + g < wave_tiles) compute(k_lds0, v_lds0, j * KS + g);
    __syncthreads();
    if (j + 1 < nit) {
      stage(k_lds0, v_lds0);
      gload(j + 3);
      if ((j + 1) * KS + g < wave_tiles) compute(k_lds1, v_lds1, (j + 1) * KS + g);
      __syncthreads();
    }
  }

  f32x16 o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = join_bf3(oh[db][r], ol[db][r]);
  float l = half_sum(l_run);
  // Key groups: group 0 merges the others' (m, l, O), handed over through the free stages.
  if constexpr (KS > 1) {
    static_assert(KS == 2 && NQ * NDB * 16 * kWave * 4 <= 2 * KS * MAT, "merge through two stages");
    float* red_o = reinterpret_cast<float*>(wave < NQ / 2 ? k_lds0 : v_lds0) + (wave % (NQ / 2)) * (NDB * 16 * kWave);
    float* ml = red_ml + wave * 2 * kWave;
    if (g == 1) {
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) red_o[(db * 16 + r) * kWave + lane] = o[db][r];
      ml[lane] = m_run;
      ml[kWave + lane] = l;
    }
    __syncthreads();
    if (g == 1) return;
    const float m1 = ml[lane], l1 = ml[kWave + lane];
    const float m = fmaxf(m_run, m1);
    const float sc0 = m_run == -INFINITY ? 0.f : exp2_fast(m_run - m);
    const float sc1 = m1 == -INFINITY ? 0.f : exp2_fast(m1 - m);   // a group without visible keys adds nothing
    l = sc0 * l + sc1 * l1;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] = sc0 * o[db][r] + sc1 * red_o[(db * 16 + r) * kWave + lane];
  }
  if (qrow < N) {
    const float inv = 1.f / l;
    float* orow = O + base + (size_t)qrow * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        f32x4 w;
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) w[rr] = o[db][g4 * 4 + rr] * inv;
        *reinterpret_cast<f32x4*>(orow + db * 32 + g4 * 8 + hi * 4) = w;
      }
  }
}

}  // namespace pa
