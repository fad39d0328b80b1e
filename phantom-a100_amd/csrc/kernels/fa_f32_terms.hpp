// Fused online-softmax attention forward for fp32 inputs on the 16-bit matrix core, with fp32's
// accuracy (the `fused` entry's fp32 inputs on grids that fill the chip; fa_f32.hpp takes the rest).
//
// The fp32 matrix core bounds fa_f32.hpp: 64 FLOP per cycle and SIMD against the 16-bit one's 1024. Here
// every fp32 operand (Q, K, V and P) is split into terms whose products are exact in the fp32
// accumulator, and the small products have an accumulator of their own, so O's main chain rounds once
// per 16 keys, not per 2. Two forms of the same block:
//  * F16x2: x = h + l / 2^11 in fp16 (h = round(x), l = round(2^11 (x - h)): 24 bits, l normal wherever h
//    is), three products (h h; h l, l h; what is left out is 2^-24 of a product and below). Its range:
//    |q|, |k| <= 4096, |v| <= 255 (V is taken 2^8 larger), and no 8 dims of a V row all below 2^-20, so
//    that what falls below the terms (2^-36 absolute) is below fp32's own rounding of the scores, and
//    2^-24 of its row in V. Every thread looks at the values that it splits.
//  * Bf16x3: x = h + m + l in bf16 over fp32's whole range, six products (h h; h m, m h; m m, h l, l h).
//    Taken by a workgroup whose inputs were out of F16x2's range, as soon as Q or its first tile shows it
//    (V x300 at 4x16x2048: 421 us, against 310 in range, timed with their host calls), else at the end of its block, which it then starts again.
// Against float64 (2-norms; fa_f32.hpp -> F16x2, Bf16x3): 4x16x512 3.6e-7 -> 2.4e-7, 2.2e-7; 4x16x2048
// 5.2e-7 -> 3.8e-7, 3.6e-7; 4x4x8192 8.8e-7 -> 6.4e-7, 6.4e-7; 2x4x4000 5.1e-7 -> 3.8e-7, 3.6e-7.
//
// Otherwise the fused kernels' scheme (fa_mfma.hpp): S^T = K Q^T and O^T += V^T P^T, a wave owning 32
// queries, P^T straight from the S^T accumulator, m raised lazily. A workgroup stages 32-key tiles:
// a thread loads 8 dims of a K and of a V row a tile ahead, splits them once for its four query waves
// and writes the planes to LDS (two stages, one barrier per tile). KS == 2: two key groups of
// four query waves walk alternate tiles and are merged at the end, which gives a CU its two waves per
// SIMD from one workgroup.
//
// Measured, fa_f32.hpp -> Bf16x3 -> F16x2: 4x16x2048 601 -> 380 -> 250 us (275 TFLOP/s), 4x16x4096 2322
// -> 1479 -> 956, causal 4x16x1024 114 -> 62 -> 47, 2x4x4000 292 -> 182 -> 122. With two waves per SIMD
// the matrix products (24 MFMAs of 32 cycles per wave and tile, half of Bf16x3's) and the VALU (the
// splits, the exponentials: about twice that) overlap only in part; three waves per SIMD spill (323 us).
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

// The two ways to take an operand. mfma: hi += the largest term product, lo += the small ones;
// join: the value of the two accumulators.
struct Bf16x3 {
  typedef Bf3 Op;
  typedef bf16 Elem;
  typedef bf16x8 Vec;
  static constexpr int PLANES = 3;
  static constexpr float kShift = 0.f, kVScale = 1.f;
  static constexpr bool kRanged = false;
  static __device__ __forceinline__ Op split_input(const float (&x)[8]) { return split3_checked(x); }
  static __device__ __forceinline__ Op split(const float (&x)[8]) { return split3(x); }
  static __device__ __forceinline__ Vec plane(const Op& t, int i) { return i == 0 ? t.h : i == 1 ? t.m : t.l; }
  static __device__ __forceinline__ Op from_planes(const Vec (&p)[3]) { return Op{p[0], p[1], p[2]}; }
  static __device__ __forceinline__ void mfma(const Op& a, const Op& b, f32x16& hi, f32x16& lo) { mfma_bf3(a, b, hi, lo); }
  static __device__ __forceinline__ float join(float hi, float lo) { return join_bf3(hi, lo); }
};
struct F16x2 {
  struct Op {
    f16x8 h, l;
  };
  typedef f16 Elem;
  typedef f16x8 Vec;
  static constexpr int PLANES = 2;
  static constexpr float kShift = 15.f;     // P <= 2^15
  static constexpr float kVScale = 256.f;
  static constexpr bool kRanged = true;
  static __device__ __forceinline__ Op split(const float (&x)[8]) {
    Op t;
#pragma unroll
    for (int j = 0; j < 8; ++j) t.h[j] = (f16)x[j];
#pragma unroll
    for (int j = 0; j < 8; ++j) t.l[j] = (f16)((x[j] - (float)t.h[j]) * 2048.f);
    return t;
  }
  static __device__ __forceinline__ Op split_input(const float (&x)[8]) { return split(x); }
  static __device__ __forceinline__ Vec plane(const Op& t, int i) { return i == 0 ? t.h : t.l; }
  static __device__ __forceinline__ Op from_planes(const Vec (&p)[2]) { return Op{p[0], p[1]}; }
  static __device__ __forceinline__ void mfma(const Op& a, const Op& b, f32x16& hi, f32x16& lo) {
    lo = mfma32x32x16(a.l, b.h, lo);
    lo = mfma32x32x16(a.h, b.l, lo);
    hi = mfma32x32x16(a.h, b.h, hi);
  }
  static __device__ __forceinline__ float join(float hi, float lo) { return fmaf(lo, 1.f / 2048.f, hi); }
};

// One block of queries of one head. False (F16x2 only): an input was out of its range, and nothing
// was stored.
template <typename TM, int D, int NQ, int KS>
__device__ __forceinline__ bool f32_terms_block(const float* __restrict__ Q, const float* __restrict__ K,
                                                const float* __restrict__ V, float* __restrict__ O, int N, int bh, int qb,
                                                float scale_log2, int causal, unsigned char* k_lds0, unsigned char* v_lds0,
                                                unsigned char* k_lds1, unsigned char* v_lds1, float* red_ml, int* red_bad) {
  typedef typename TM::Op Op;
  typedef typename TM::Vec Vec;
  constexpr int PLANES = TM::PLANES;
  constexpr int BM = NQ * 32, BN = 32;
  constexpr int CR = D / 8, RB = D * 2, PLANE = BN * RB, MAT = PLANES * PLANE;   // term planes of a tile
  constexpr int STEPS = D / 16, NDB = D / 32;
  constexpr int CPT = BN * CR / (NQ * kWave);   // 8-dim chunks of K and of V per thread and tile
  // m is set to a row's max plus kLazyLog2 and raised again only when the max has passed it, so
  // P = 2^(s c - m) stays at most 1 (P V cannot overflow where V does not), F16x2: 2^15.
  constexpr float kLazyLog2 = 8.f;
  constexpr float kQKMax = 4096.f, kVMax = 255.f, kVLow = 0x1p-20f;   // F16x2's range
  static_assert(D == 64 && CPT * NQ * kWave == BN * CR, "whole chunks per thread");
  const int g = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / (NQ * kWave));   // key group
  const int tid = (int)threadIdx.x % (NQ * kWave), lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lq = lane % 32, hi = lane / 32;

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
  Op qf[STEPS];
  float qk_max = 0.f, v_max = 0.f;   // F16x2: what its range check looks at
  bool v_low = false;
  auto abs_max = [](const float (&x)[8]) __attribute__((always_inline)) {
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(x[j]));
    return m;
  };
#pragma unroll
  for (int kk = 0; kk < STEPS; ++kk) {
    float x[8];
    load8(q_rs, (uint32_t)((qrow * D + 16 * kk + 8 * hi) * 4), x);
    if constexpr (TM::kRanged) qk_max = fmaxf(qk_max, abs_max(x));
    qf[kk] = TM::split_input(x);
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
      if constexpr (TM::kRanged) {
        qk_max = fmaxf(qk_max, abs_max(kx[i]));
        const float m = abs_max(vx[i]);
        v_max = fmaxf(v_max, m);
        v_low |= m < kVLow && m > 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) vx[i][j] *= TM::kVScale;
      }
      const Op a = TM::split_input(kx[i]), b = TM::split_input(vx[i]);
#pragma unroll
      for (int pl = 0; pl < PLANES; ++pl) {
        *reinterpret_cast<Vec*>(ks + pl * PLANE + k_dst[i]) = TM::plane(a, pl);
        *reinterpret_cast<Vec*>(vs + pl * PLANE + v_dst[i]) = TM::plane(b, pl);
      }
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
      Vec a[PLANES];
#pragma unroll
      for (int pl = 0; pl < PLANES; ++pl) a[pl] = *reinterpret_cast<const Vec*>(ks + pl * PLANE + k_addr[kk]);
      TM::mfma(TM::from_planes(a), qf[kk], sh, sl);
    }
    float s[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = TM::join(sh[r], sl[r]);
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
    const float m_new = fmaxf(m_run, fmaf(half_max(mx), scale_log2, kLazyLog2));
    if (__builtin_amdgcn_ballot_w64(m_new > m_run + kLazyLog2) != 0) {
      const float alpha = m_new > m_run ? exp2_fast(m_run - m_new) : 1.f;   // m_run = -inf -> 0
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db) oh[db] *= alpha, ol[db] *= alpha;
    }
    const float nm = m_run == -INFINITY ? 0.f : TM::kShift - m_run;   // no visible key so far: P = 0
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
      const Op pf = TM::split(p[k2]);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        Vec a[PLANES];
#pragma unroll
        for (int pl = 0; pl < PLANES; ++pl) {
          const unsigned char* p0 = vs + pl * PLANE + k2 * 16 * RB + v_addr[db];
          const i16x4 a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<i16x4>)(p0));
          const i16x4 a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<i16x4>)(p0 + 8 * RB));
          a[pl] = __builtin_bit_cast(Vec, i16x8{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]});
        }
        TM::mfma(TM::from_planes(a), pf, oh[db], ol[db]);
      }
    }
  };

  // F16x2: whether a value that some thread has split so far was out of range (all threads get the
  // same answer). (A NaN is in range: it goes through the terms to where it belongs.)
  auto out_of_range = [&]() __attribute__((always_inline)) {
    const bool bad = __builtin_amdgcn_ballot_w64(qk_max > kQKMax || v_max > kVMax || v_low) != 0;
    if (lane == 0) red_bad[(int)threadIdx.x / kWave] = bad;
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int w = 0; w < NQ * KS; ++w) any |= red_bad[w];
    return __builtin_amdgcn_readfirstlane(any) != 0;
  };

  // Tile j + 1 is staged, and tile j + 2 loaded, before tile j's products; one barrier per tile
  // (offsets past the head load zeros).
  gload(0);
  stage(k_lds0, v_lds0);
  gload(1);
  if constexpr (TM::kRanged) {   // Q and the first tile: inputs of another scale show here
    if (out_of_range()) {
      __syncthreads();
      return false;
    }
  } else {
    __syncthreads();
  }
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

  if constexpr (TM::kRanged) {
    if (out_of_range()) {
      __syncthreads();   // (Bf16x3 writes what slower waves may still read)
      return false;
    }
  }

  f32x16 o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = TM::join(oh[db][r], ol[db][r]);
  float l = half_sum(l_run);
  // Key groups: group 0 merges the others' (m, l, O), handed over through the free stages.
  if constexpr (KS > 1) {
    static_assert(KS == 2 && NQ * NDB * 16 * kWave * 4 <= 2 * KS * 3 * PLANE, "merge through two stages");
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
    if (g == 1) return true;
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
    const float inv = 1.f / (TM::kVScale * l);
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
  return true;
}

template <int D, int NQ, int KS>
__global__ void __launch_bounds__(NQ * KS * kWave)
__attribute__((amdgpu_waves_per_eu(2)))
fa_f32_terms_fwd(const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
             float* __restrict__ O, int N, int num_qblocks, int total_blocks, float scale_log2, int causal) {
  constexpr int MAT = 3 * 32 * D * 2;   // the planes of a 32-key tile in the larger form
  __shared__ __attribute__((aligned(1024))) unsigned char k_lds0[KS * MAT], v_lds0[KS * MAT], k_lds1[KS * MAT], v_lds1[KS * MAT];
  __shared__ float red_ml[KS > 1 ? (KS - 1) * NQ * 2 * kWave : 1];
  __shared__ int red_bad[NQ * KS];
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
  if (!f32_terms_block<F16x2, D, NQ, KS>(Q, K, V, O, N, bh, qb, scale_log2, causal, k_lds0, v_lds0, k_lds1, v_lds1, red_ml,
                                         red_bad))
    f32_terms_block<Bf16x3, D, NQ, KS>(Q, K, V, O, N, bh, qb, scale_log2, causal, k_lds0, v_lds0, k_lds1, v_lds1, red_ml,
                                       red_bad);
}

}  // namespace pa
