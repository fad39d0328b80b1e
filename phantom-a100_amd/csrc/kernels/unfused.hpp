// Unfused attention paths (the `naive` and `tiled` entries): the full fp32 score matrix S is
// written to a caller-provided [BH][N][N] workspace, normalised in place, then multiplied by V.
// They exist for API completeness and as an independent GPU cross-check of the fused kernels;
// any head dim d >= 1 is accepted, fp32 or fp16 storage, fp32 arithmetic.
//
//   naive (/root/reference/csrc/kernels/naive.cuh:10-64): the same three passes (scores, softmax
//         by row max / sum / normalise, P.V) as plain loops, a wave taking a few rows of each product.
//   tiled (/root/reference/csrc/kernels/tiled.cuh:16-117): rows of whole 16-byte pieces up to 128
//         dims: the scores on the matrix core (tiled_scores_mfma), then softmax and P.V in one pass
//         over them (tiled_softmax_pv). Other head dims and unaligned tensors: 64x64 output tiles
//         with 4x4 register blocking per thread and LDS-staged operands. Softmax with one wave per
//         row, the row held in registers up to 8192 keys (one read of S); longer rows take one
//         workgroup per row, in register-held segments whose max the workgroup agrees on before
//         their sums (one read of S up to 32768 keys, two beyond). Causal P.V skips key tiles
//         right of the diagonal.
#pragma once

#include "common.hpp"
#include "fa_mfma.hpp"   // v_swz: the V tile layout of the fused kernel, reused by tiled_softmax_pv

namespace pa {

// ------------------------------------------------------------------------------------ naive
// The reference's three unfused passes, each a plain loop per lane, laid out by waves: every
// workgroup is 4 waves, and a wave owns R rows of the product it writes (64 keys of the score rows,
// 64 head dims of the output rows; a whole softmax row), so the operand that the rows bring (query
// rows, P rows) is the same address in every lane, and the per-lane operand (a K row, a V column)
// serves R rows. One row per wave spent an L1 access on every FMA (a lane's K row piece, a V element);
// with the rows' operands in scalar registers, R FMAs share it, and what is left is the latency of
// the loads, issued 16 elements at a time: fp32 2x8x333 d = 80 298 -> 56 us, fp32 8x16x1024 d = 128
// 19.8 -> 2.3 ms, fp16 324x128 d = 64 232 -> 78 us, fp32 42x128 52 -> 19 us, same bits. Grids are
// flattened into x: row groups times column blocks.

// S[h][i][j0 + lane] for the wave's R query rows i and 64 keys from j0; keys after i are -inf when
// causal. A lane's K row element serves the R rows, whose Q elements are the same address in every
// lane (scalar loads; a row past N reads row N - 1 and is not stored). PIECES (rows of whole 16-byte
// pieces, 16-byte aligned): K rows are read a 16-byte piece per load instead of an element (one load
// then touches the wave's 64 K rows once per piece, not once per element); a score's products are
// summed in dim order either way.
template <typename T, bool PIECES, int R>
__global__ void __launch_bounds__(256)
naive_scores(const T* __restrict__ Q, const T* __restrict__ K, float* __restrict__ S, int N, int d,
             float scale, int causal, int key_blocks) {
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int unit = (int)blockIdx.x * 4 + wave;   // (R query rows, 64-key block)
  const int i0 = unit / key_blocks * R;
  const int j = (unit % key_blocks) * kWave + (int)threadIdx.x % kWave;
  if (i0 >= N || j >= N) return;
  const size_t head = (size_t)blockIdx.y * N;
  const T* q[R];
  float dot[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    q[r] = Q + (head + min(i0 + r, N - 1)) * d;
    dot[r] = 0.f;
  }
  if (!(causal && j > i0 + R - 1)) {   // (masked for every row: the products are not needed)
    const T* kj = K + (head + j) * d;
    if constexpr (PIECES) {
      constexpr int E = 16 / (int)sizeof(T);   // elements per piece
      constexpr int U = 16 / E;                // pieces per step: their loads are issued together
      typedef T VecE __attribute__((ext_vector_type(E)));
      int c = 0;
      for (; c + 16 <= d; c += 16) {
        VecE kv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) kv[u] = __builtin_bit_cast(VecE, *reinterpret_cast<const u32x4*>(kj + c + u * E));
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int e = 0; e < 16; ++e) dot[r] = fmaf(to_f32(q[r][c + e]), to_f32(kv[e / E][e % E]), dot[r]);
      }
      for (; c < d; c += E) {
        const VecE kv = __builtin_bit_cast(VecE, *reinterpret_cast<const u32x4*>(kj + c));
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int e = 0; e < E; ++e) dot[r] = fmaf(to_f32(q[r][c + e]), to_f32(kv[e]), dot[r]);
      }
    } else {
      for (int c = 0; c < d; ++c) {
        const float kv = to_f32(kj[c]);
#pragma unroll
        for (int r = 0; r < R; ++r) dot[r] = fmaf(to_f32(q[r][c]), kv, dot[r]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (i0 + r < N) S[(head + i0 + r) * N + j] = (causal && j > i0 + r) ? -INFINITY : scale * dot[r];
}

// Row r of S in place: max, sum of exp(s - max), then exp(s - max) / sum, each a strided pass
// of the wave's 64 lanes over the row followed by a wave all-reduce (DPP and lane swaps).
__global__ void __launch_bounds__(256)
naive_softmax(float* __restrict__ S, int N, long long rows) {
  const long long r = (long long)blockIdx.x * 4 + threadIdx.x / kWave;
  if (r >= rows) return;
  const int lane = (int)threadIdx.x % kWave;
  float* srow = S + r * N;
  float mx = -INFINITY;
  for (int j = lane; j < N; j += kWave) mx = fmaxf(mx, srow[j]);
  mx = wave_allreduce(mx, MaxOp{});
  float sum = 0.f;
  for (int j = lane; j < N; j += kWave) sum += expf(srow[j] - mx);
  sum = wave_allreduce(sum, SumOp{});
  const float rcp = 1.f / sum;
  for (int j = lane; j < N; j += kWave) srow[j] = expf(srow[j] - mx) * rcp;
}

// O[h][i][c0 + lane] = sum over keys j of P[h][i][j] V[h][j][c0 + lane], for the wave's R rows i and
// 64 head dims from c0, the keys in order. A V element serves the R rows, whose probabilities are the
// same address in every lane (scalar loads; a row past N reads row N - 1 and is not stored). With
// causal, the keys after the last of the rows, whose probabilities are zero, are left out.
template <typename T, int R>
__global__ void __launch_bounds__(256)
naive_pv(const float* __restrict__ P, const T* __restrict__ V, T* __restrict__ O, int N, int d, int causal,
         int dim_blocks) {
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int unit = (int)blockIdx.x * 4 + wave;   // (R query rows, 64-dim block)
  const int i0 = unit / dim_blocks * R;
  const int c = (unit % dim_blocks) * kWave + (int)threadIdx.x % kWave;
  if (i0 >= N || c >= d) return;
  const size_t head = (size_t)blockIdx.y * N;
  const float* p[R];
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    p[r] = P + (head + min(i0 + r, N - 1)) * N;
    acc[r] = 0.f;
  }
  const T* vc = V + head * d + c;
  const int n = causal ? min(N, i0 + R) : N;
  constexpr int U = 16;   // keys per step: their loads are issued together
  int j = 0;
  for (; j + U <= n; j += U) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = to_f32(vc[(size_t)(j + u) * d]);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) acc[r] = fmaf(p[r][j + u], v[u], acc[r]);
  }
  for (; j < n; ++j) {
    const float v = to_f32(vc[(size_t)j * d]);
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = fmaf(p[r][j], v, acc[r]);
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (i0 + r < N) O[(head + i0 + r) * d + c] = from_f32<T>(acc[r]);
}

// ------------------------------------------------------------------------------------ tiled
constexpr int kTile = 64;   // output tile edge
constexpr int kTk = 16;     // reduction chunk

// S[i0:i0+64, j0:j0+64] = scale * Q_tile . K_tile^T (keys after the query -> -inf when causal).
// Operands are staged transposed ([k][row]) so each thread reads its 4 rows / 4 columns as one
// float4 from LDS.
template <typename T>
__global__ void __launch_bounds__(256)
tiled_scores(const T* __restrict__ Q, const T* __restrict__ K, float* __restrict__ S, int N, int d,
             float scale, int causal) {
  __shared__ __attribute__((aligned(16))) float qs[kTk][kTile + 4];
  __shared__ __attribute__((aligned(16))) float ksm[kTk][kTile + 4];
  const int bh = blockIdx.z;
  const int i0 = blockIdx.y * kTile, j0 = blockIdx.x * kTile;
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  const T* Qb = Q + (size_t)bh * N * d;
  const T* Kb = K + (size_t)bh * N * d;
  float acc[4][4] = {};
  for (int c0 = 0; c0 < d; c0 += kTk) {
    // 64 rows x 16 dims per operand = 1024 elements, 4 per thread; consecutive threads read
    // consecutive dims of one row.
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int idx = tid + e * 256;
      const int r = idx / kTk, c = idx % kTk;
      const int qi = i0 + r, kj = j0 + r, cc = c0 + c;
      qs[c][r] = (qi < N && cc < d) ? to_f32(Qb[(size_t)qi * d + cc]) : 0.f;
      ksm[c][r] = (kj < N && cc < d) ? to_f32(Kb[(size_t)kj * d + cc]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kTk; ++c) {
      const float4 a = *reinterpret_cast<const float4*>(&qs[c][ty * 4]);
      const float4 b = *reinterpret_cast<const float4*>(&ksm[c][tx * 4]);
      const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int w = 0; w < 4; ++w) acc[u][w] = fmaf(av[u], bv[w], acc[u][w]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = i0 + ty * 4 + u;
    if (i >= N) continue;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int j = j0 + tx * 4 + w;
      if (j < N) S[((size_t)bh * N + i) * N + j] = (causal && j > i) ? -INFINITY : acc[u][w] * scale;
    }
  }
}

// ---- Matrix-core form (head dims in whole 16-byte pieces up to 128, 16-byte aligned tensors): two
// kernels, the scores and one pass over them for softmax and P.V together.
//
// What bounds it is the score workspace, 4 bytes per score and pass over it. Three kernels passed over
// it four times (write, softmax read and write, P.V read); these two pass over it twice. The workspace
// holds the raw dot products in the order in which the matrix core makes and takes them: each strip of
// 32 query rows of a head (its last strip has the rb rows left) is a run of rb * N floats, the keys in
// groups of 4 (the last group has the w keys left), so that the score of key k and the strip's row r is
//     strip[rb * (k - k % 4) + w * r + k % 4],
// and the strips fill a head's N * N floats exactly. A lane of a 32 x 32 S^T block (one query, groups
// of 4 keys) then stores 16 contiguous bytes, a wave 1 KB per instruction, and the second kernel loads
// its P^T operands the same way. (A strip starts 16-byte aligned only where N * N * head does: the
// vectors are declared with an element's alignment.)
//
// Measured, three kernels -> two, us a call: fp16 4x16x2048 d = 64 983 -> 561, causal 922 -> 405, 4x8x4096
// 1771 -> 919, 8x32x256 58 -> 38 (4x16x4096: the scores stored at 3.9 TB/s, read at 5.1); fp32 4x16x2048
// 1327 -> 758 (both kernels also near the fp32 matrix core's rate). Rows and head dims that took the VALU
// kernels: fp16 1x8x2000 d = 80 407 -> 61, 2x32x2047 d = 32 2022 -> 468, 1x1x4096 d = 96 640 -> 60; fp32
// 1x16x333 d = 40 91 -> 20. Passes over a few heads at a time, whose scores stay in the memory-side
// cache (192 MiB), gained 8 % at 4x16x2048 but lost up to 20 % on causal rows and smaller grids.
// Against float64 (2-norms) the error is no larger on N(0, 1) inputs (fp32 1x5x3392 d = 128 causal 5.2e-7
// -> 3.8e-7; fp16 its output's rounding) and within 1.4 % with q and k times 3, where the scores' own
// roundings set it; the largest element's error falls there as often as it grows.
typedef float Score4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr uint32_t kNoRow = 0x80000000u;   // an offset past every head (a head is below 2 GiB)

// S^T blocks of 128 queries x 128 keys per workgroup, 64 x 64 per wave as 2 x 2 blocks of 32 x 32.
// With causal, blocks whose keys all come after their queries are neither computed nor stored (the
// second kernel does not read them). The operands are read straight from memory in the MFMA layout; rows
// past N and dims past d read as zero through the buffer's range. fp16: one 32x32x16 step takes dims
// 16 kk + 8 (l / 32) .. + 7 of row l % 32. fp32: 16 steps of 32x32x2 take dims 16 (l / 32) + 0 .. 15 of a
// 32-dim chunk, in Q and K alike.
template <typename T>
__global__ void __launch_bounds__(256)
tiled_scores_mfma(const T* __restrict__ Q, const T* __restrict__ K, float* __restrict__ S, int N, int d, int causal) {
  const int bh = blockIdx.z;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r0 = blockIdx.y * 128 + (wave / 2) * 64;   // first query, first key of the wave
  const int c0 = blockIdx.x * 128 + (wave % 2) * 64;
  if (r0 >= N || c0 >= N || (causal && c0 > r0 + 63)) return;
  const int lr = lane % 32, hk = lane / 32;
  const uint32_t head_bytes = (uint32_t)((size_t)N * d * sizeof(T));
  const rsrc_t q_rs = make_rsrc(Q + (size_t)bh * N * d, head_bytes);
  const rsrc_t k_rs = make_rsrc(K + (size_t)bh * N * d, head_bytes);
  f32x16 acc[2][2];   // [key block][query block]
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) acc[kb][qb] = f32x16{};
  if constexpr (std::is_same<T, f16>::value) {
    for (int c = 0; c < d; c += 32) {
      f16x8 a[2][2], b[2][2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int col = c + 16 * kk + 8 * hk;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          a[kk][x] = __builtin_bit_cast(f16x8, load16(k_rs, col < d ? (uint32_t)((c0 + 32 * x + lr) * d + col) * 2 : kNoRow));
          b[kk][x] = __builtin_bit_cast(f16x8, load16(q_rs, col < d ? (uint32_t)((r0 + 32 * x + lr) * d + col) * 2 : kNoRow));
        }
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int qb = 0; qb < 2; ++qb) acc[kb][qb] = mfma32x32x16(a[kk][kb], b[kk][qb], acc[kb][qb]);
    }
  } else {
    for (int c = 0; c < d; c += 32) {
      f32x4 a[2][4], b[2][4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int col = c + 16 * hk + 4 * v;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          a[x][v] = __builtin_bit_cast(f32x4, load16(k_rs, col < d ? (uint32_t)((c0 + 32 * x + lr) * d + col) * 4 : kNoRow));
          b[x][v] = __builtin_bit_cast(f32x4, load16(q_rs, col < d ? (uint32_t)((r0 + 32 * x + lr) * d + col) * 4 : kNoRow));
        }
      }
#pragma unroll
      for (int kk = 0; kk < 16; ++kk)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int qb = 0; qb < 2; ++qb)
            acc[kb][qb] = mfma32x32x2(a[kb][kk / 4][kk % 4], b[qb][kk / 4][kk % 4], acc[kb][qb]);
    }
  }
  // Register r of a block holds key 8 (r / 4) + 4 hk + r % 4 and query lr.
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int i0 = r0 + 32 * qb;
    const int rb = min(32, N - i0);
    if (lr >= rb) continue;
    float* strip = S + (size_t)bh * N * N + (size_t)i0 * N;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int key = c0 + 32 * kb + 8 * g + 4 * hk, w = N - key;
        if (w >= 4) {
          Score4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = acc[kb][qb][4 * g + e];
          *reinterpret_cast<Score4*>(strip + rb * key + 4 * lr) = x;
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (e < w) strip[rb * key + w * lr + e] = acc[kb][qb][4 * g + e];
        }
      }
  }
}

// O = softmax(scale S) V in one pass over the strips: the fused kernels' online softmax (fa_mfma.hpp)
// with the S^T blocks loaded instead of computed. A wave owns a strip of 32 query rows; per tile of BN
// keys, the row max (m raised, and l and O rescaled, only when a row's max has outgrown it by 2^8),
// P = 2^(S c - m), and O^T += V^T P^T on the matrix core from a V tile in LDS.
// fp16 V: P (taken 2^7 larger, at most 2^15) as two fp16 terms, the lo one 2^11 larger still and with an
// accumulator of its own, on the fp16 matrix core: 22 bits of a weight down to 2^-21 of its row's
// largest, an absolute 2^-43 of that below, which an fp16 output does not show. (The two accumulators
// leave three waves per SIMD at 64 dims, two past them; against one unscaled accumulator, four and three
// waves, us: 4x16x2048 d = 64 575 -> 578, causal 391 -> 401, d = 128 676 -> 658, 1x1x4096 d = 96 58.7 -> 59.5.)
// V^T read with ds_read_b64_tr_b16. fp32 V: P and V as they are on the fp32 matrix core, whose two k-slots
// take the keys that the two lane halves hold.
// V goes to LDS with direct loads (two stages), the next tile's scores to registers, during the current
// tile; several workgroups per CU keep enough of both in flight. KS > 1: the keys are dealt tile by
// tile to KS waves of one strip, each with its own V stages, (m, l, O) merged at the end, for grids
// that would leave CUs without a workgroup.
template <typename T, int NDB, int KS>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(std::is_same<T, float>::value ? (KS == 1 && NDB <= 2 ? 4 : 3) : (KS == 1 && NDB == 1 ? 4 : 2))))
tiled_softmax_pv(const float* __restrict__ S, const T* __restrict__ V, T* __restrict__ O, int N, int d, float scale_log2,
                 int causal) {
  constexpr bool HALF = std::is_same<T, f16>::value;
  constexpr int NQ = 4 / KS, BN = KS == 1 ? 64 : 32;
  constexpr int DP = NDB <= 2 ? 64 : 128;           // dims of a V row in LDS
  constexpr int RB = DP * (int)sizeof(T), CR = RB / 16, EPC = 16 / (int)sizeof(T);
  constexpr int TILE_BYTES = BN * RB, THREADS = NQ * kWave;
  constexpr int CPT = BN * CR / THREADS;            // 16-byte V chunks per thread per tile
  constexpr int NG = BN / 8;                        // groups of 4 keys per lane and tile
  constexpr float kLazyLog2 = 8.f, kTermShift = HALF ? 7.f : 0.f, kLoScale = 2048.f;
  __shared__ __attribute__((aligned(1024))) unsigned char v_lds[KS * 2 * TILE_BYTES];
  __shared__ float red_ml[KS > 1 ? (KS - 1) * 2 * kWave : 1];
  const int bh = blockIdx.y;
  const int g = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / THREADS);   // key group
  const int tid = (int)threadIdx.x % THREADS, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lq = lane % 32, hi = lane / 32;
  const int qblk = causal ? (int)(gridDim.x - 1 - blockIdx.x) : (int)blockIdx.x;   // longest causal rows first
  const int q0 = qblk * 32 * NQ, i0 = q0 + 32 * wave, qrow = i0 + lq;
  const int rb = min(32, N - i0);                   // rows of the wave's strip (none: rb <= 0)
  const float* strip = S + (size_t)bh * N * N + (size_t)min(i0, N - 1) * N;
  const rsrc_t v_rs = make_rsrc(V + (size_t)bh * N * d, (uint32_t)((size_t)N * d * sizeof(T)));
  unsigned char* lds = v_lds + g * 2 * TILE_BYTES;

  // V tile: chunk swizzle by row. fp16: the fused kernels'. fp32: rows 4 apart, read by the two lane
  // halves at the same dim, differ by half the banks.
  auto swz = [](int row) { return HALF ? v_swz<CR>(row) : 8 * ((row >> 2) & 1); };
  uint32_t v_src[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int slot = i * THREADS + tid, row = slot / CR, c = (slot % CR) ^ swz(row);
    v_src[i] = c * EPC < d ? (uint32_t)(row * d + c * EPC) * (uint32_t)sizeof(T) : kNoRow;
  }
  auto load_v = [&](int stage, int k0) {
#pragma unroll
    for (int i = 0; i < CPT; ++i)
      load16_to_lds(v_rs, lds + stage * TILE_BYTES + (i * THREADS + wave * kWave) * 16, v_src[i],
                    (uint32_t)k0 * (uint32_t)(d * sizeof(T)));
  };
  int v_addr[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    if constexpr (HALF) {   // the transposed reads of fa_mfma.hpp
      const int g16 = lane / 16, i16 = lane % 16, v_row = hi * 4 + i16 / 4, v_cl = 2 * (g16 % 2) + (i16 % 4) / 2;
      v_addr[db] = v_row * RB + (((4 * db + v_cl) ^ swz(v_row)) * 16) + 8 * (i16 % 2);
    } else {                // V[4 hi][32 db + lq]; rows 8 further on have the same swizzle
      v_addr[db] = 4 * hi * RB + (((8 * db + lq / 4) ^ swz(4 * hi)) * 16) + 4 * (lq % 4);
    }
  }
  // Scores of a tile: group i of the lane is keys k0 + 8 i + 4 hi .. + 3 of its row. Rows past the
  // strip read its last row (not stored); keys past N are not read.
  const int pitch = max(rb, 1), lrow = min(lq, pitch - 1);
  const uint32_t s_off = (uint32_t)(pitch * 4 * hi + 4 * lrow);   // this lane's offset from key group 8 i
  auto load_s = [&](f32x4 (&x)[NG], int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NG; ++i) x[i] = *reinterpret_cast<const Score4*>(strip + pitch * (k0 + 8 * i) + s_off);
  };
  // The tile that N ends in, an element per load (keys past N read the strip's first score; masked).
  auto load_last = [&](f32x4 (&x)[NG], int k0) __attribute__((always_inline)) {
    int w0 = N - k0 - 4 * hi;   // keys left from the lane's first one
    asm volatile("" : "+v"(w0));
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const int w = w0 - 8 * i;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = strip[e < w ? pitch * (N - w) + min(w, 4) * lrow + e : 0];
      x[i] = f32x4{y[0], y[1], y[2], y[3]};
    }
  };

  float m_run = -INFINITY, l_run = 0.f;
  f32x16 o[NDB], o_lo[HALF ? NDB : 1];   // o_lo: the lo terms' products
#pragma unroll
  for (int db = 0; db < NDB; ++db) o[db] = f32x16{};
#pragma unroll
  for (int db = 0; db < (HALF ? NDB : 1); ++db) o_lo[db] = f32x16{};
  const int kv_end = causal ? min(N, q0 + 32 * NQ) : N;
  const int ntiles = (kv_end + BN - 1) / BN, nit = (ntiles + KS - 1) / KS;
  const int wave_end = rb <= 0 ? 0 : causal ? min(N, i0 + 32) : N;   // keys that the wave's rows see
  const int wave_tiles = (wave_end + BN - 1) / BN;
  const int clean_tiles = causal ? min(N, i0 + 1) / BN : N / BN;       // of these, without a mask

  auto compute = [&](f32x4 (&x)[NG], const unsigned char* vs, int t) __attribute__((always_inline)) {
    if (t >= clean_tiles) {
      // Key t BN + 8 i + 4 hi + e is visible iff 8 i + e <= lim (hidden from the compiler, which would
      // keep the limit of every element in registers).
      int lim = (causal ? min(N - 1, qrow) : N - 1) - t * BN - 4 * hi;
      asm volatile("" : "+v"(lim));
#pragma unroll
      for (int i = 0; i < NG; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (8 * i + e > lim) x[i][e] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, x[i][e]);
    // (A row is raised for its own max alone: causal rows' bits do not depend on later tokens.)
    const float m_new = fmaxf(m_run, half_max(mx) * scale_log2);
    const bool raise = m_new > m_run + kLazyLog2;
    if (__builtin_amdgcn_ballot_w64(raise) != 0) {
      const float alpha = raise ? exp2_fast(m_run - m_new) : 1.f;   // m_run = -inf -> 0
      m_run = raise ? m_new : m_run;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        o[db] *= alpha;
        if constexpr (HALF) o_lo[db] *= alpha;
      }
    }
    const float nm = m_run == -INFINITY ? 0.f : kTermShift - m_run;   // no visible key so far: P = 0
    float sum = 0.f;                                                  // the tile's sum, then one add to l
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[i][e] = exp2_fast(fmaf(x[i][e], scale_log2, nm));
        sum += x[i][e];
      }
    l_run += sum;
    if constexpr (HALF) {
      // P's terms for 16 keys. (The lo terms read the packed halves of the hi ones, as in fa_mfma.hpp.)
      auto terms = [&](int ks, f16x8& ph, f16x8& pl) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          const float p0 = x[2 * ks + j / 4][j % 4], p1 = x[2 * ks + j / 4][j % 4 + 1];
          f16x2 h = {(f16)p0, (f16)p1};
          asm("" : "+v"(h));
          ph[j] = h[0], ph[j + 1] = h[1];
          pl[j] = (f16)fmaf(-kLoScale, (float)h[0], kLoScale * p0);
          pl[j + 1] = (f16)fmaf(-kLoScale, (float)h[1], kLoScale * p1);
        }
      };
      auto v_op = [&](int ks, int db) __attribute__((always_inline)) {
        const unsigned char* p0 = vs + ks * 16 * RB + v_addr[db];
        const i16x4 a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<i16x4>)(p0));
        const i16x4 a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<i16x4>)(p0 + 8 * RB));
        return __builtin_bit_cast(f16x8, i16x8{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]});
      };
#pragma unroll
      for (int ks = 0; ks < BN / 16; ++ks) {
        f16x8 ph, pl;
        terms(ks, ph, pl);
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          const f16x8 a = v_op(ks, db);
          o_lo[db] = mfma32x32x16(a, pl, o_lo[db]);
          o[db] = mfma32x32x16(a, ph, o[db]);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < NG; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int db = 0; db < NDB; ++db)
            o[db] = mfma32x32x2(*reinterpret_cast<const float*>(vs + (8 * i + e) * RB + v_addr[db]), x[i][e], o[db]);
    }
  };

  // Key group g's iteration j is tile j KS + g. At the top of an iteration its tile has landed and
  // every wave is done with the stage that the next tile goes to.
  const int full_tiles = min(wave_tiles, N / BN);
  f32x4 x[NG], xn[NG];
  if (g < ntiles) load_v(0, g * BN);
  if (g < full_tiles) load_s(x, g * BN);
#pragma unroll 1
  for (int j = 0; j < nit; ++j) {
    const int t = j * KS + g;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t + KS < ntiles) load_v((j + 1) & 1, (t + KS) * BN);
    if (t + KS < full_tiles) load_s(xn, (t + KS) * BN);
    if (t < wave_tiles) {
      if (t >= full_tiles) load_last(x, t * BN);
      compute(x, lds + (j & 1) * TILE_BYTES, t);
    }
#pragma unroll
    for (int i = 0; i < NG; ++i) x[i] = xn[i];
  }
  if constexpr (HALF)
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] = fmaf(o_lo[db][r], 1.f / kLoScale, o[db][r]);
  float l = half_sum(l_run);
  if constexpr (KS > 1) {
    static_assert((KS - 1) * NDB * 16 * kWave * 4 <= KS * 2 * TILE_BYTES, "merge through the stages");
    __syncthreads();
    if (g > 0) {
      float* red_o = reinterpret_cast<float*>(v_lds) + (g - 1) * NDB * 16 * kWave;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) red_o[(db * 16 + r) * kWave + lane] = o[db][r];
      red_ml[(g - 1) * 2 * kWave + lane] = m_run;
      red_ml[(g - 1) * 2 * kWave + kWave + lane] = l;
    }
    __syncthreads();
    if (g > 0) return;
#pragma unroll 1
    for (int x = 0; x < KS - 1; ++x) {
      const float* red_o = reinterpret_cast<const float*>(v_lds) + x * NDB * 16 * kWave;
      const float m1 = red_ml[x * 2 * kWave + lane], l1 = red_ml[x * 2 * kWave + kWave + lane];
      const float m = fmaxf(m_run, m1);
      const float sc0 = m_run == -INFINITY ? 0.f : exp2_fast(m_run - m);
      const float sc1 = m1 == -INFINITY ? 0.f : exp2_fast(m1 - m);   // a group without visible keys adds nothing
      m_run = m;
      l = sc0 * l + sc1 * l1;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] = sc0 * o[db][r] + sc1 * red_o[(db * 16 + r) * kWave + lane];
    }
  }
  // The weights are normalised after P.V, so fp32 values near the largest float can overflow sums that
  // normalised weights would not (above FLT_MAX / (2^8 N)): those rows again, with normalised weights. fp32
  // 4x16x2048 789 us, 1.6 ms with an infinity in one head, 3.9 ms with every value at 3e38.
  const float inv = 1.f / l;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    if (__builtin_amdgcn_ballot_w64(qrow < N && any_not_finite(o[db]) && __builtin_isfinite(l)) != 0) {
      constexpr int KEYS = HALF ? 8 : KS == 1 && NDB <= 2 ? 2 : 4;   // (what the registers hold)
      f32x16 acc;
      retake_rows<KEYS>(acc, V + (size_t)bh * N * d, d, 32 * db, wave_end, [&](int k0, float (&p)[KEYS]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < KEYS; ++k) {
          const int key = min(k0 + k, N - 1), k4 = key & ~3;
          const float s = strip[pitch * k4 + min(4, N - k4) * lrow + key % 4];
          p[k] = causal && key > qrow ? -1.f : exp2_fast(fmaf(s, scale_log2, kTermShift - m_run)) * inv;
        }
      });
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] = __builtin_isfinite(o[db][r]) ? o[db][r] * inv : acc[r];
    } else {
      o[db] *= inv;
    }
  }
  // Register r of block db holds dim 32 db + 8 (r / 4) + 4 hi + r % 4 of query qrow.
  if (qrow < N) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    T* orow = O + ((size_t)bh * N + qrow) * d;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int c = 32 * db + 8 * g4 + 4 * hi;
        T4 w;
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) w[rr] = from_f32<T>(o[db][g4 * 4 + rr]);
        if (c < d) *reinterpret_cast<T4*>(orow + c) = w;
      }
  }
}

// ---- General form (any head dim): the scores row by row in the workspace, softmax in place, P.V.
// One wave per row, the whole row held in registers (rows of at most 64 * VPL keys): S is read
// once and P written once, 8 bytes per score (the naive softmax reads S three times). The max
// first, then the sum of exp(x - max) kept in place, then P = e / sum; element j of the row sits in
// lane j % 64, slot j / 64, so every load and store of a wave covers 256 contiguous bytes.
template <int VPL>
__global__ void __launch_bounds__(256)
tiled_softmax_rows(float* __restrict__ S, int N) {
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int bh = blockIdx.y;
  const int i = blockIdx.x * 4 + wave;
  if (i >= N) return;  // whole wave leaves together
  float* row = S + ((size_t)bh * N + i) * N;
  float x[VPL];
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < VPL; ++k) {
    const int j = lane + k * kWave;
    x[k] = j < N ? row[j] : -INFINITY;
    m = fmaxf(m, x[k]);
  }
  m = wave_allreduce(m, MaxOp{});
  float l = 0.f;
#pragma unroll
  for (int k = 0; k < VPL; ++k) {
    x[k] = expf(x[k] - m);   // -inf (masked or past N) -> 0; every row has a finite score
    l += x[k];
  }
  l = wave_allreduce(l, SumOp{});
  const float inv = 1.f / l;
#pragma unroll
  for (int k = 0; k < VPL; ++k) {
    const int j = lane + k * kWave;
    if (j < N) row[j] = x[k] * inv;
  }
}

// Rows longer than the one-wave register kernel holds (N > 64 * 128): one 256-lane workgroup per
// row. The row is cut into segments of 256 * VPL keys, each held in registers (key
// j0 + 256 k + t in slot k of thread t, so every load and store of a wave covers 256 contiguous
// bytes). Per segment, the workgroup first agrees on the segment's max (wave all-reduce, then the
// four wave maxima through LDS); where it exceeds the row's running max m, the per-thread sums are
// multiplied by exp(m - m_new) once, and then every key of the segment adds exp(x - m) against the
// same, workgroup-uniform m. So m needs no per-lane state and the end is a plain sum. A row of one
// segment (N <= 256 * VPL) keeps its exponentials in registers and writes P from them (S read
// once); longer rows read each segment again for P = exp(x - m) / l.
template <int VPL>
__global__ void __launch_bounds__(256)
tiled_softmax_segments(float* __restrict__ S, int N) {
  constexpr int SEG = 256 * VPL;
  // Two slots so that consecutive reductions need one barrier each: reduction r writes slot r % 2
  // after every thread has passed reduction r - 1's barrier, i.e. after the reads of slot r % 2 by
  // reduction r - 2.
  __shared__ float part[2][4];
  const int t = (int)threadIdx.x, wave = t / kWave, lane = t % kWave;
  float* row = S + ((size_t)blockIdx.y * N + blockIdx.x) * N;
  int slot = 0;
  auto block_reduce = [&](float v, auto op) {
    v = wave_allreduce(v, op);
    if (lane == 0) part[slot][wave] = v;
    __syncthreads();
    const float r = op(op(part[slot][0], part[slot][1]), op(part[slot][2], part[slot][3]));
    slot ^= 1;
    return r;
  };
  const int segments = (N + SEG - 1) / SEG;
  float x[VPL];
  float m = -INFINITY, l = 0.f;
  for (int sg = 0; sg < segments; ++sg) {
    const int j0 = sg * SEG;
    float smax = -INFINITY;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int j = j0 + k * 256 + t;
      x[k] = j < N ? row[j] : -INFINITY;
      smax = fmaxf(smax, x[k]);
    }
    smax = block_reduce(smax, MaxOp{});
    if (smax > m) {   // workgroup-uniform; l is still 0 while m is -inf
      l = m == -INFINITY ? 0.f : l * expf(m - smax);
      m = smax;
    }
    // Key 0 is visible in every row (causal or not), so m is finite from the first segment on.
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      x[k] = expf(x[k] - m);   // masked or past N: exp(-inf) = 0
      l += x[k];
    }
  }
  const float inv = 1.f / block_reduce(l, SumOp{});
  if (segments == 1) {
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int j = k * 256 + t;
      if (j < N) row[j] = x[k] * inv;
    }
  } else {
    for (int j = t; j < N; j += 256) row[j] = expf(row[j] - m) * inv;
  }
}

// O[i0:i0+64, c0:c0+64] = P_rows . V_cols; with causal, P is zero right of the diagonal so
// the key loop stops at the tile's last row.
template <typename T>
__global__ void __launch_bounds__(256)
tiled_pv(const float* __restrict__ P, const T* __restrict__ V, T* __restrict__ O, int N, int d, int causal) {
  __shared__ __attribute__((aligned(16))) float ps[kTk][kTile + 4];
  __shared__ __attribute__((aligned(16))) float vsm[kTk][kTile + 4];
  const int bh = blockIdx.z;
  const int i0 = blockIdx.y * kTile, c0 = blockIdx.x * kTile;
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  const float* Pb = P + (size_t)bh * N * N;
  const T* Vb = V + (size_t)bh * N * d;
  const int k_end = causal ? min(N, i0 + kTile) : N;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < k_end; k0 += kTk) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int idx = tid + e * 256;
      // P: 64 rows x 16 keys, consecutive threads read consecutive keys of one row.
      const int r = idx / kTk, kk = idx % kTk;
      const int pi = i0 + r, pj = k0 + kk;
      ps[kk][r] = (pi < N && pj < N) ? Pb[(size_t)pi * N + pj] : 0.f;
      // V: 16 keys x 64 dims, consecutive threads read consecutive dims of one key.
      const int vk = idx / kTile, vc = idx % kTile;
      const int gk = k0 + vk, gc = c0 + vc;
      vsm[vk][vc] = (gk < N && gc < d) ? to_f32(Vb[(size_t)gk * d + gc]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kTk; ++kk) {
      const float4 a = *reinterpret_cast<const float4*>(&ps[kk][ty * 4]);
      const float4 b = *reinterpret_cast<const float4*>(&vsm[kk][tx * 4]);
      const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int w = 0; w < 4; ++w) acc[u][w] = fmaf(av[u], bv[w], acc[u][w]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = i0 + ty * 4 + u;
    if (i >= N) continue;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int c = c0 + tx * 4 + w;
      if (c < d) O[((size_t)bh * N + i) * d + c] = from_f32<T>(acc[u][w]);
    }
  }
}

}  // namespace pa
