// The reference's v1 single-head fp32 kernels (legacy_naive / legacy_tiled /
// legacy_fused), rebuilt for gfx950.
//
// Reference behaviour (csrc/legacy/legacy_ops.cu:10-51 and
// src/legacy/{naive,tiled,fused}_attention.cu of shrvan30/flash-attention-cuda):
// q, k, v and o are (N, 64) fp32, one head, no mask, and
// o = softmax(q k^T / sqrt(64)) v in fp32. The three v1 kernels compute the
// same function with different algorithms:
//   naive  an exact row max over every key first, then the exponentials and
//          the weighted sum (naive_attention.cu:45-110, three passes there);
//   tiled  an online softmax over 32-key tiles with O renormalised at every
//          tile, O = (l_old * e^(m_old - m_new) O + e^(m_tile - m_new) PV) / l_new
//          (tiled_attention.cu:170-205);
//   fused  the same online softmax with the two factors computed once per
//          tile (fused_attention.cu:160-183).
// The v1 warp reductions return each thread's own value
// (softmax_stable.cu / fused_attention.cu:26-52), so every row is independent.
//
// This build keeps the three entry points and their arithmetic contract
// (fp32 in, fp32 products and sums, fp32 out); the kernels are its own:
//   block   = 16 waves over 16 QT query rows (QT = 1, or 2 on long inputs);
//             wave w takes the w-th sixteenth of the keys (in 16-key blocks),
//             so a block is one query tile and needs no other block's result.
//   product = v_mfma_f32_16x16x4_f32 (fp32 operands, fp32 accumulation):
//             S^T = K Q^T, step s over head dims [4 s, +4) in their order, so
//             a score is the sum of 64 fused multiply-adds from dim 0 to dim
//             63 (lane group g = lane / 16 supplies dim 4 s + g: a K or Q
//             fragment is four 16-byte loads of a row and sixteen lane-group
//             swaps); O^T += V^T P^T with P straight from
//             the S^T accumulators (lane group g, element i: key 4 g + i of
//             the block, query lane % 16), step i over the keys {4 g + i}, and
//             the head dims taken as [4 m + d] for row m of tile d, so a V
//             fragment is one 16-byte load. No wave shares a key with another:
//             K and V go from memory to registers, nothing is staged.
//   merge   the sixteen states (m, l, o) of each row meet in LDS.
//   naive   pass 1 folds only the row max (the waves' maxima merged in
//             LDS), pass 2 accumulates e^(s - m) and e^(s - m) v with that
//             exact max, one division at the end.
//   tiled   online softmax, O kept normalised after every 16-key block.
//   fused   online softmax, O unnormalised, one division at the end.
// What bounds it: issue of fp32 MFMAs (32 of 32 cycles per 16-key block and
// wave) and of about as many cycles of VALU work (exponentials, transposes) on
// the CUs that have a block, N / 16 of them up to N = 4096. Measured (fused,
// us per call) against one wave per 64 rows and key quarter with every K and V
// row broadcast from LDS: N = 256 48.1 -> 9.5, 1024 180 -> 20.6, 2048 355 ->
// 33.6, 4096 741 -> 67.7 (64 TFLOP/s), 8192 1482 -> 219, 16384 2935 -> 799;
// error against float64 at N = 2048 4.9e-7 -> 3.6e-7 (relative, 2-norm).
// The launch is asynchronous on the caller's stream (the v1 launchers
// synchronised the device after every call, naive_attention.cu:150).

#include "fa_internal.h"

namespace fa {
namespace {

constexpr int kLegacyWaves = 16;                          // key shares per block
constexpr int kLegacyThreads = kLegacyWaves * kWave;      // 1024
constexpr int kLegacyKeys = 16;                           // keys per step
constexpr int kLegacyPitch = kHeadDim + 4;                // floats per merged row in LDS

enum LegacyMode { kNaive = 0, kTiled = 1, kFused = 2 };

// One row's fragment: x[a][b] is head dim 16 a + 4 b + g.
struct RowFrag {
  float x[4][4];
};
template <bool BY32>
__device__ __forceinline__ void swap_groups(float &a, float &b) {
  const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
  // Lane groups 2, 3 of a with 0, 1 of b, or groups 1, 3 of a with 0, 2 of b.
  const auto r = BY32 ? __builtin_amdgcn_permlane32_swap(ua, ub, false, false)
                      : __builtin_amdgcn_permlane16_swap(ua, ub, false, false);
  const unsigned ra = r[0], rb = r[1];
  a = __builtin_bit_cast(float, ra);
  b = __builtin_bit_cast(float, rb);
}
// Head dims [16 a + 4 g, +4) of a row per load a.
__device__ __forceinline__ void load_row(const float *__restrict__ base, int row, int g,
                                         floatx4 (&y)[4]) {
  const float *const p = base + static_cast<size_t>(row) * kHeadDim + 4 * g;
#pragma unroll
  for (int a = 0; a < 4; ++a) y[a] = *reinterpret_cast<const floatx4 *>(p + 16 * a);
}
// The fragment of a loaded row: a 4 x 4 transpose between the four registers
// of a load and the four lane groups.
__device__ __forceinline__ void transpose_row(const floatx4 (&y)[4], RowFrag &f) {
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) f.x[a][b] = y[a][b];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    swap_groups<true>(f.x[a][0], f.x[a][2]);
    swap_groups<true>(f.x[a][1], f.x[a][3]);
    swap_groups<false>(f.x[a][0], f.x[a][1]);
    swap_groups<false>(f.x[a][2], f.x[a][3]);
  }
}

// max / sum over the four lanes that hold one query (lane % 16).
__device__ __forceinline__ float max_groups(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}
__device__ __forceinline__ float sum_groups(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}

// Scores of one query tile against 16 keys: element i is key key0 + 4 g + i,
// -inf at or past n.
__device__ __forceinline__ floatx4 scores(const RowFrag &kf, const RowFrag &qf, int key0, int g,
                                          int n, float scale) {
  floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.x[a][b], qf.x[a][b], s, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] *= scale;
  if (key0 + kLegacyKeys > n) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (key0 + 4 * g + i >= n) s[i] = -INFINITY;
  }
  return s;
}

template <int MODE, int QT>
__global__ __launch_bounds__(kLegacyThreads, 4) void legacy_attention_kernel(
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
    float *__restrict__ o, int n, float scale) {
  constexpr int kRows = 16 * QT;
  __shared__ __attribute__((aligned(16))) float acc_lds[kLegacyWaves * kRows * kLegacyPitch];
  __shared__ float m_lds[kLegacyWaves][kRows], l_lds[kLegacyWaves][kRows];

  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int col = lane & 15, g = lane >> 4;
  const int row0 = static_cast<int>(blockIdx.x) * kRows;
  // This wave's keys [begin, end): n / 16 of them, in whole 16-key blocks.
  const int blocks = (n + kLegacyKeys - 1) / kLegacyKeys;
  const int share = (blocks + kLegacyWaves - 1) / kLegacyWaves;
  const int begin = min(wave * share, blocks) * kLegacyKeys;
  const int end = min(min((wave + 1) * share, blocks) * kLegacyKeys, n);

  RowFrag qf[QT];  // query row0 + 16 t + col (rows past n: the last one, not stored)
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    floatx4 y[4];
    load_row(q, min(row0 + 16 * t + col, n - 1), g, y);
    transpose_row(y, qf[t]);
  }
  // O^T tiles: tile d, element e: head dim 16 g + 4 e + d of query col.
  floatx4 acc[QT][4];
  float m[QT], l[QT];  // l: this lane's keys only
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    m[t] = -INFINITY;
    l[t] = 0.f;
#pragma unroll
    for (int d = 0; d < 4; ++d) acc[t][d] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  if (MODE == kNaive) {
    // Pass 1: the exact row max over every key.
    floatx4 ky[4];
    if (QT == 1) load_row(k, min(begin + col, n - 1), g, ky);
    for (int key0 = begin; key0 < end; key0 += kLegacyKeys) {
      RowFrag kf;
      if (QT > 1) load_row(k, min(key0 + col, n - 1), g, ky);
      transpose_row(ky, kf);
      if (QT == 1 && key0 + kLegacyKeys < end)
        load_row(k, min(key0 + kLegacyKeys + col, n - 1), g, ky);
#pragma unroll
      for (int t = 0; t < QT; ++t) {
        const floatx4 s = scores(kf, qf[t], key0, g, n, scale);
#pragma unroll
        for (int i = 0; i < 4; ++i) m[t] = fmaxf(m[t], s[i]);
      }
    }
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      m[t] = max_groups(m[t]);
      if (g == 0) m_lds[wave][16 * t + col] = m[t];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int w = 0; w < kLegacyWaves; ++w) m[t] = fmaxf(m[t], m_lds[w][16 * t + col]);
    __syncthreads();
  }

  // Pass 2 (naive) or the only pass (tiled, fused).
  // One query tile: the rows of the next 16-key block are requested before
  // this one's products (4096 rows: 72 -> 69 us; two tiles leave no registers
  // for it).
  floatx4 ky[4], vy[4];
  // vy[i][d]: head dim 4 col + d of key key0 + 4 g + i.
  auto load_v = [&](int key0) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      vy[i] = *reinterpret_cast<const floatx4 *>(
          v + static_cast<size_t>(min(key0 + 4 * g + i, n - 1)) * kHeadDim + 4 * col);
  };
  if (QT == 1) {
    load_row(k, min(begin + col, n - 1), g, ky);
    load_v(min(begin, n - 1));
  }
  for (int key0 = begin; key0 < end; key0 += kLegacyKeys) {
    RowFrag kf;
    if (QT > 1) {
      load_row(k, min(key0 + col, n - 1), g, ky);
      load_v(key0);
    }
    transpose_row(ky, kf);
    floatx4 vf[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) vf[i] = vy[i];
    if (key0 + kLegacyKeys > n) {
      // (A key past n has weight 0, which would not cancel an inf or NaN.)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (key0 + 4 * g + i >= n) vf[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    if (QT == 1 && key0 + kLegacyKeys < end) {
      load_row(k, min(key0 + kLegacyKeys + col, n - 1), g, ky);
      load_v(key0 + kLegacyKeys);
    }
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      floatx4 s = scores(kf, qf[t], key0, g, n, scale);
      float lt = 0.f;
      if (MODE == kNaive) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[i] = s[i] == -INFINITY ? 0.f : expf(s[i] - m[t]);
          lt += s[i];
        }
        l[t] += lt;
      } else {
        const float mt = max_groups(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])));
        const float m_new = fmaxf(m[t], mt);
        // (No score above -inf yet: nothing to rescale, and -inf - -inf is NaN.)
        const float a_old = m[t] == m_new ? 1.0f : expf(m[t] - m_new);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[i] = s[i] == -INFINITY ? 0.f : expf(s[i] - m_new);
          lt += s[i];
        }
        float c_old = a_old;
        if (MODE == kTiled) {
          // O stays normalised: O = O * (l a_old / l_new) + sum_j (p_j / l_new) v_j,
          // with the row sums of the four lanes.
          const float l_old = l[t];
          lt = sum_groups(lt);
          l[t] = l_old * a_old + lt;
          const float inv = l[t] > 0.f ? 1.0f / l[t] : 0.f;
          c_old = l_old * a_old * inv;
#pragma unroll
          for (int i = 0; i < 4; ++i) s[i] *= inv;
        } else {
          l[t] = l[t] * a_old + lt;
        }
        if (__builtin_amdgcn_ballot_w64(c_old != 1.0f) != 0) {
#pragma unroll
          for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[t][d][e] *= c_old;
        }
        m[t] = m_new;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d)
          acc[t][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][d], s[i], acc[t][d], 0, 0, 0);
    }
  }

  // Merge the sixteen states of each row.
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int row = 16 * t + col;
    float *const mine = acc_lds + (wave * kRows + row) * kLegacyPitch + 16 * g;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *reinterpret_cast<floatx4 *>(mine + 4 * e) =
          floatx4{acc[t][0][e], acc[t][1][e], acc[t][2][e], acc[t][3][e]};
    const float l_row = MODE == kTiled ? l[t] : sum_groups(l[t]);
    if (g == 0) {
      m_lds[wave][row] = m[t];
      l_lds[wave][row] = l_row;
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int row = 16 * t + wave;  // the wave finishes one row per tile, lane = head dim
    float m_all = -INFINITY;
#pragma unroll
    for (int w = 0; w < kLegacyWaves; ++w) m_all = fmaxf(m_all, m_lds[w][row]);
    float l_all = 0.f, x = 0.f;
#pragma unroll
    for (int w = 0; w < kLegacyWaves; ++w) {
      // Weight of wave w's sums: e^(m_w - m_all) (tiled states are
      // normalised, so their sums are o_w * l_w).
      const float lw = l_lds[w][row];
      float f = lw > 0.f ? expf(m_lds[w][row] - m_all) : 0.f;
      l_all += f * lw;
      if (MODE == kTiled) f *= lw;
      x = fmaf(f, acc_lds[(w * kRows + row) * kLegacyPitch + lane], x);
    }
    if (row0 + row < n)
      o[static_cast<size_t>(row0 + row) * kHeadDim + lane] = x * (l_all > 0.f ? 1.0f / l_all : 0.f);
  }
}

template <int QT>
void launch_mode(const float *q, const float *k, const float *v, float *o, int n, int variant,
                 hipStream_t stream) {
  const float scale = 1.0f / sqrtf(static_cast<float>(kHeadDim));
  const dim3 blocks(static_cast<unsigned>((n + 16 * QT - 1) / (16 * QT))), threads(kLegacyThreads);
  switch (variant) {
    case kNaive:
      hipLaunchKernelGGL((legacy_attention_kernel<kNaive, QT>), blocks, threads, 0, stream, q, k, v,
                         o, n, scale);
      break;
    case kTiled:
      hipLaunchKernelGGL((legacy_attention_kernel<kTiled, QT>), blocks, threads, 0, stream, q, k, v,
                         o, n, scale);
      break;
    default:
      hipLaunchKernelGGL((legacy_attention_kernel<kFused, QT>), blocks, threads, 0, stream, q, k, v,
                         o, n, scale);
      break;
  }
}

}  // namespace

int launch_legacy_attention(const float *q, const float *k, const float *v, float *o, int n,
                            int variant, hipStream_t stream) {
  // 32 rows per block halve the K and V reads per row, and still give every
  // CU a block from 8192 rows on.
  if (n >= 8192)
    launch_mode<2>(q, k, v, o, n, variant, stream);
  else
    launch_mode<1>(q, k, v, o, n, variant, stream);
  return check_hip(hipGetLastError(), "legacy_attention_kernel launch");
}

}  // namespace fa
