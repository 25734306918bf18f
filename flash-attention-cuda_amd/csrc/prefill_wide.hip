// Causal / full prefill for head_dim 64 on large grids: 64 query rows per wave.
//
// The same function, products, softmax and precision rules as prefill.hip
// (its header describes them; prefill.cu:164-343 of shrvan30/flash-attention-
// cuda is the reference behaviour). What differs is the shape of a wave's work:
//   wave   = 64 query rows as two groups (A, B) of 32 rows. Every K and V
//            fragment it reads from LDS feeds both groups, so a product costs
//            half the LDS reads it costs a 32-row wave.
//   block  = 4 waves, 256 query rows of one (b, h), one stream of 64-key tiles
//            through a K ring of kStages tiles and a V ring of kStages + 1
//            (72 KiB LDS, filled by direct global->LDS loads); two blocks per
//            CU, <= 256 VGPRs, so each SIMD runs one wave of each block.
//   grid   = one block per (b, h, 256-row query tile), heaviest tile first.
//
// What bounds it: the SIMD's issue of VALU and MFMA instructions, and the
// clock the chip holds at that power. B8 H12 S4096 full: 1.20 M cycles per
// SIMD in two-half blocks, 1.06 M in one-half blocks, 0.92 M here (matrix
// cores busy 37, 42 and 48 %), at 1.5-2.0 GHz in all three.
//
// Main loop, per 32-key block j of the tiles every row of the wave sees whole:
//   X:  QK of group B(j) | second half of P_B(j-1), row max of S_A(j)
//       PV and row sums of group B(j-1) | first half of P_A(j)
//   Y:  QK of group A(j+1) | second half of P_A(j), row max of S_B(j)
//       PV and row sums of group A(j) | first half of P_B(j)
// so each line's MFMAs (left) run under VALU work (right) that does not depend
// on them: the exponentials of a block's keys 16-31 are put off to the next
// line, which otherwise would hold four MFMAs and only the row max. One S
// tile, one K block and one V block per wave are enough; K(j+1) is read after
// QK B(j) has consumed K(j), V(j) after PV B(j-1) has consumed V(j-1).
// The tile that needs a mask (the wave's causal diagonal, the ragged end) takes
// a plain step without the pipeline. Split-P passes run the same loop with P's
// low parts and twice the PV products.
//
// The running max: m moves by prefill.hip's rule (lazy from 1024 keys on). A
// row's tile max is compared with one threshold kept in raw score units, which
// is brought up to date (m, row sum) only when some row of the group passes
// it, so an ordinary block pays 8 max3, the lane-pair max and one compare.
// The rounded mass sums the squares of the fp32 weights with v_fma_f32: on
// gfx950 v_dot2_f32_f16 does not run beside an MFMA (a register-only loop with
// a block's mix of instructions: 509 ns per pair of waves with dot2, 389 with
// v_fma_f32).

#include <type_traits>

#include "fa_internal.h"
#include "mfma_tile.h"
#include "prefill_common.h"

namespace fa {
namespace {

constexpr int kD = 64;
constexpr int kWideWaves = 4;
constexpr int kWideThreads = kWideWaves * kWave;
constexpr int kWideRows = kWideWaves * 64;  // query rows per block
constexpr int kTileKeys = 64;
constexpr unsigned kTileBytes = kTileKeys * kD * 2;  // 8 KiB
constexpr int kStages = 4;                            // K ring; the V ring has one more
constexpr int kTileLoads = 4;                         // global->LDS loads of a wave per tile

// Softmax state of one 32-row group (one query per lane pair).
struct Group {
  float m;         // the max P is taken against (log2 domain, scaled by c)
  float thr;       // raw score above which m may have to move
  float r;         // this lane's share of the rounded mass, units of m
  floatx4 lacc;    // row sum: element 0
  floatx16 o[2];   // O^T accumulators
};

__device__ __forceinline__ float row_max(const floatx16 &s) {
  float mx = -INFINITY;
#pragma unroll
  for (int a = 0; a < 16; ++a) mx = fmaxf(mx, s[a]);
  return max_lane_pair(mx);
}

// Some row's block max is above its threshold: the rule of prefill.hip's
// tile_max (m moves, for every row of the group that rose, when one row's max
// exceeds m by more than slack, or carries more than kLazyMaxDominant of its
// row sum), then the threshold for the blocks to come:
// m + min(slack, max(0, log2(row sum * kLazyMaxDominant))). The row sum only
// grows until then, so the kept threshold is never too high.
__device__ __forceinline__ void move_max(float mx, float c_scale, float inv_c, float slack,
                                         Group &st) {
  float mx_c;
  {
    // No contraction: with mx_c rounded once, the block that sets m has its
    // largest weight at exp2(0) = 1 exactly.
#pragma clang fp contract(off)
    mx_c = mx * c_scale;
  }
  const float pm = fast_exp2(mx_c - st.m);
  const bool move = mx_c > st.m + slack || pm > fmaxf(1.0f, kLazyMaxDominant * st.lacc[0]);
  if (__builtin_amdgcn_ballot_w64(move) != 0) {
    const float m_new = fmaxf(st.m, mx_c);
    const float alpha = fast_exp2(st.m - m_new);
    st.m = m_new;
    // A largest weight of exactly 1 takes no rounding: half of it off the
    // mass in each lane of the pair.
    st.r = st.r * (alpha * alpha) - (mx_c == m_new ? 0.5f : 0.0f);
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int a = 0; a < 16; ++a) st.o[db][a] *= alpha;
    st.lacc[0] *= alpha;
  }
  const float rise = __builtin_amdgcn_logf(fmaxf(kLazyMaxDominant * st.lacc[0], 1.0f));
  st.thr = (st.m + fminf(slack, rise)) * inv_c;
}
__device__ __forceinline__ void check_max(float mx, float c_scale, float inv_c, float slack,
                                          Group &st) {
  if (__builtin_amdgcn_ballot_w64(mx > st.thr) != 0) move_max(mx, c_scale, inv_c, slack, st);
}

// P^T of a 32-key block (keys 0-15, keys 16-31), lo with split P only.
struct Weights {
  half8 hi[2], lo[2];
};

// The H-th 16 keys of P^T from their exponents (log2 domain, m taken off).
template <bool SPLIT, int H>
__device__ __forceinline__ void exp_half(const float (&x)[8], Group &st, Weights &p) {
  float sq0 = 0.f, sq1 = 0.f;
#pragma unroll
  for (int t = 0; t < 8; t += 2) {
    const float e0 = fast_exp2(x[t]), e1 = fast_exp2(x[t + 1]);
    const half2 hi = {static_cast<_Float16>(e0), static_cast<_Float16>(e1)};
    p.hi[H][t] = hi[0];
    p.hi[H][t + 1] = hi[1];
    if (SPLIT) {
      p.lo[H][t] = static_cast<_Float16>(e0 - static_cast<float>(hi[0]));
      p.lo[H][t + 1] = static_cast<_Float16>(e1 - static_cast<float>(hi[1]));
    } else {
      sq0 = fmaf(e0, e0, sq0);
      sq1 = fmaf(e1, e1, sq1);
    }
  }
  if (!SPLIT) st.r += sq0 + sq1;
}
template <int H>
__device__ __forceinline__ void exponents(const floatx16 &s, float c_scale, const Group &st,
                                          float (&x)[8]) {
#pragma unroll
  for (int t = 0; t < 8; ++t) x[t] = fmaf(s[8 * H + t], c_scale, -st.m);
}

// A masked block's P^T.
template <bool SPLIT>
__device__ __forceinline__ void exp_masked(const floatx16 &s, float c_scale, Group &st,
                                           Weights &p) {
  float sq = 0.f;
#pragma unroll
  for (int a = 0; a < 16; a += 2) {
    // (-inf * c is NaN when c = 0.)
    const float p0 = s[a] == -INFINITY ? 0.f : fast_exp2(fmaf(s[a], c_scale, -st.m));
    const float p1 = s[a + 1] == -INFINITY ? 0.f : fast_exp2(fmaf(s[a + 1], c_scale, -st.m));
    const half2 hi = {static_cast<_Float16>(p0), static_cast<_Float16>(p1)};
    p.hi[a >> 3][a & 7] = hi[0];
    p.hi[a >> 3][(a & 7) + 1] = hi[1];
    if (SPLIT) {
      p.lo[a >> 3][a & 7] = static_cast<_Float16>(p0 - static_cast<float>(hi[0]));
      p.lo[a >> 3][(a & 7) + 1] = static_cast<_Float16>(p1 - static_cast<float>(hi[1]));
    } else {
      sq = fmaf(p0, p0, sq);
      sq = fmaf(p1, p1, sq);
    }
  }
  if (!SPLIT) st.r += sq;
}

__device__ __forceinline__ void read_k(unsigned tile, int kb, const FragOffsetsD<kD> &fo,
                                       half8 (&kf)[4]) {
  const unsigned base = uniform_lds_u(tile + kb * (kTileBytes / 2));
#pragma unroll
  for (int i = 0; i < 4; ++i)
    kf[i] = *reinterpret_cast<__attribute__((address_space(3))) const half8 *>(
        opaque_lds_at(base, fo.k[i]));
}
__device__ __forceinline__ void read_v(unsigned tile, int kb, const FragOffsetsD<kD> &fo,
                                       half8 (&vf)[2][2]) {
  const unsigned base = uniform_lds_u(tile + kb * (kTileBytes / 2));
#pragma unroll
  for (int db = 0; db < 2; ++db) {
    lds_half *p = opaque_lds_at(base, fo.v[db]);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int part = 0; part < 2; ++part) {
        const short4v r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) short4v *)(p + (16 * ks + 8 * part) * kD));
        const half4 v4 = __builtin_bit_cast(half4, r);
#pragma unroll
        for (int e = 0; e < 4; ++e) vf[ks][db][4 * part + e] = v4[e];
      }
  }
}
__device__ __forceinline__ void qk(const half8 (&kf)[4], const half8 (&qf)[4], floatx16 &s) {
#pragma unroll
  for (int a = 0; a < 16; ++a) s[a] = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) s = mfma(kf[i], qf[i], s);
}
// O^T += V^T P^T and the row sums of P (6 MFMAs, 12 with split P).
template <bool SPLIT>
__device__ __forceinline__ void pv(const half8 (&vf)[2][2], const Weights &p, const half8 &sel,
                                   Group &st) {
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
    for (int db = 0; db < 2; ++db) st.o[db] = mfma(vf[ks][db], p.hi[ks], st.o[db]);
    st.lacc = mfma16(sel, p.hi[ks], st.lacc);
    if (SPLIT) {
#pragma unroll
      for (int db = 0; db < 2; ++db) st.o[db] = mfma(vf[ks][db], p.lo[ks], st.o[db]);
      st.lacc = mfma16(sel, p.lo[ks], st.lacc);
    }
  }
}

// Scheduling of one line of the main loop: its DS LDS reads first, then each
// of its N MFMAs followed by up to W VALU instructions.
template <int N, int W, int DS>
__device__ __forceinline__ void interleave() {
  if constexpr (DS > 0) __builtin_amdgcn_sched_group_barrier(0x100, DS, 0);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, W, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
}
// Values a line computes for later lines: a use here keeps the compiler from
// sinking their computation to where they are consumed.
template <bool SPLIT, int H>
__device__ __forceinline__ void keep(const Weights &p, const Group &st) {
  asm volatile("" ::"v"(p.hi[H]), "v"(st.r));
  if (SPLIT) asm volatile("" ::"v"(p.lo[H]));
}
__device__ __forceinline__ void keep(const float (&x)[8]) {
#pragma unroll
  for (int t = 0; t < 8; ++t) asm volatile("" ::"v"(x[t]));
}

template <bool CAUSAL, bool OUT_F32>
__global__ __launch_bounds__(kWideThreads, 2) void prefill_wide_kernel(
    const _Float16 *__restrict__ q, const _Float16 *__restrict__ k,
    const _Float16 *__restrict__ v, void *__restrict__ o, int seq, int n_qtiles, int bh_count,
    int group, float c_scale, bool negate_q, bool split_all) {
  __shared__ __attribute__((aligned(1024))) _Float16 lds[(2 * kStages + 1) * kTileBytes / 2];
  static_assert(kWideWaves * 32 * kD * 4 <= sizeof(lds), "output staging fits in LDS");
  const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
  const int rw = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int pos = static_cast<int>(blockIdx.x);
  const int qtile = n_qtiles - 1 - pos / bh_count;
  int bh = home_head(pos, bh_count);
  if (group > 1) bh = grouped_head(bh, bh_count);
  const size_t head_off = static_cast<size_t>(bh) * seq * kD;
  const size_t kv_off = static_cast<size_t>(bh / group) * seq * kD;
  const _Float16 *const kp = k + kv_off;
  const _Float16 *const vp = v + kv_off;

  const int q0 = qtile * kWideRows;
  const int qw0 = q0 + rw * 64;  // the wave's rows [qw0, +64): group g holds [qw0 + 32 g, +32)
  const int key_end = CAUSAL ? min(seq, q0 + kWideRows) : seq;
  const int n_tiles = (key_end + kTileKeys - 1) / kTileKeys;
  // Tiles that every row of the wave sees whole. At most one more holds keys
  // that the wave sees (below wave_end) and needs a mask.
  const int n_full = CAUSAL ? min(qw0, seq) / kTileKeys : seq / kTileKeys;
  const int wave_end = CAUSAL ? min(seq, qw0 + 64) : seq;
  // The rules of prefill.hip for short rows (split P) and the lazy max.
  const bool short_rows = split_all || (CAUSAL ? q0 : seq) < kSplitPRowsBelow;
  const float slack = (CAUSAL ? q0 : seq) >= kLazyMaxRowsFrom ? kLazyMaxSlack : 0.f;
  const float inv_c = 1.0f / c_scale;

  const unsigned kring = lds_addr(lds);
  const unsigned vring = kring + kStages * kTileBytes;
  auto ktile = [&](int t) { return kring + (t % kStages) * kTileBytes; };
  auto vtile = [&](int t) { return vring + (t % (kStages + 1)) * kTileBytes; };
  // Wave rw loads rows [16 rw, +16) of a K and of a V tile, 8 rows per load.
  unsigned voff[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (2 * rw + i) * 8 + lane / 8, p = lane % 8;
    voff[0][i] = 2u * static_cast<unsigned>(r * kD + ((p ^ k_swz(r)) << 3));
    voff[1][i] = 2u * static_cast<unsigned>(r * kD + ((p ^ v_swz(r)) << 3));
  }
  auto issue = [&](int t) {
    if (t >= n_tiles) return;
    const int key0 = t * kTileKeys;
    const unsigned ks = ktile(t) + rw * 2048, vs = vtile(t) + rw * 2048;
    if (key0 + kTileKeys <= seq) {
      const _Float16 *const kb = kp + static_cast<size_t>(key0) * kD;
      const _Float16 *const vb = vp + static_cast<size_t>(key0) * kD;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        global_to_lds16_sbase_at(kb, voff[0][i], ks + i * 1024);
        global_to_lds16_sbase_at(vb, voff[1][i], vs + i * 1024);
      }
    } else {  // rows past the end: the last row, masked (K) or weighted by 0 (V)
      const int ln = fresh_lane();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = (2 * rw + i) * 8 + ln / 8, p = ln % 8;
        const size_t row = static_cast<size_t>(min(key0 + r, seq - 1)) * kD;
        global_to_lds16_at(kp + row + ((p ^ k_swz(r)) << 3), ks + i * 1024);
        global_to_lds16_at(vp + row + ((p ^ v_swz(r)) << 3), vs + i * 1024);
      }
    }
  };

  const FragOffsetsD<kD> fo = frag_offsets_d<kD>(lane);
  const half8 sel = rowsum_selector(lane);
  half8 qf[2][4];  // Q^T fragments: query qw0 + 32 g + lane % 32, head dims [32 (lane / 32) + 8 s, +8)
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const _Float16 *const qrow =
        q + head_off + static_cast<size_t>(min(qw0 + 32 * g + (lane & 31), seq - 1)) * kD +
        (lane >> 5) * 32;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[g][s] = *reinterpret_cast<const half8 *>(qrow + 8 * s);
  }
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (negate_q) qf[g][s] = -qf[g][s];
      // Waited for here: a Q load pending inside the loop would make the
      // compiler wait there for every load of the rings.
      asm volatile("" ::"v"(qf[g][s]));
    }
  Group st[2];

  auto start = [&]() {  // the first kStages tiles on their way, tile 0 resident
#pragma unroll
    for (int t = 0; t < kStages; ++t) issue(t);
    if (kStages - 1 < n_tiles)
      wait_loads<(kStages - 1) * kTileLoads>();
    else
      wait_loads<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // Every wave passes this once per tile t of the block: tile t + 1 becomes
  // resident, and no wave reads K tile t or V tile t - 1 any more (each has
  // drained its LDS reads), so the loads of tile t + kStages may go to the
  // stages these held.
  auto boundary = [&](int t) {
    if (t + kStages - 1 < n_tiles)
      wait_loads<(kStages - 2) * kTileLoads>();
    else
      wait_loads<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(t + kStages);
  };
  // One tile without the pipeline, masked, P split or not.
  auto plain_tile = [&](auto split_p, int t) {
    constexpr bool SPLIT = decltype(split_p)::value;
    const int ln = fresh_lane();
    for (int kb = 0; kb < 2; ++kb) {
      const int key0 = t * kTileKeys + kb * 32;
      if (key0 >= wave_end) break;
      half8 kf[4], vf[2][2];
      read_k(ktile(t), kb, fo, kf);
      read_v(vtile(t), kb, fo, vf);
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int row0 = qw0 + 32 * g;
        if (CAUSAL && key0 >= row0 + 32) continue;
        floatx16 s;
        qk(kf, qf[g], s);
        // Element a holds key key0 + 8 (a / 4) + 4 (ln / 32) + a % 4.
        const int lim = (CAUSAL ? min(row0 + (ln & 31), seq - 1) : seq - 1) - key0 - 4 * (ln >> 5);
#pragma unroll
        for (int a = 0; a < 16; ++a)
          s[a] = (8 * (a >> 2) + (a & 3) <= lim) ? s[a] : -INFINITY;
        check_max(row_max(s), c_scale, inv_c, slack, st[g]);
        Weights p;
        exp_masked<SPLIT>(s, c_scale, st[g], p);
        pv<SPLIT>(vf, p, sel, st[g]);
      }
    }
  };

  // The whole key range, P split or not.
  auto sweep = [&](auto split_p) {
    constexpr bool SPLIT = decltype(split_p)::value;
    constexpr int kPv = SPLIT ? 12 : 6;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      st[g].m = kNegHuge;
      st[g].thr = -INFINITY;
      st[g].r = 0.f;
      st[g].lacc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int a = 0; a < 16; ++a) st[g].o[db][a] = 0.f;
    }
    if (n_full > 0) {
      half8 kf[4], vf[2][2];
      Weights pa, pb;
      floatx16 sa, sb;
      float xa[8], xb[8];
      // PV B(-1): zero weights on zero V.
#pragma unroll
      for (int i = 0; i < 8; ++i) xb[i] = -INFINITY;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        pb.hi[ks] = half8{};
        pb.lo[ks] = half8{};
        vf[ks][0] = half8{};
        vf[ks][1] = half8{};
      }
      read_k(ktile(0), 0, fo, kf);
      qk(kf, qf[0], sa);
      for (int t = 0; t < n_full; ++t) {
        const unsigned kt = ktile(t), kn = ktile(t + 1), vt = vtile(t);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // K(2 t + 2), read below, is in tile t + 1 (past the last tile: any
          // bits of the ring, and the S they give is not used).
          if (h == 1) boundary(t);
          float x0[8];
          qk(kf, qf[1], sb);
          exp_half<SPLIT, 1>(xb, st[1], pb);
          float mx = row_max(sa);
          interleave<4, 10, 0>();
          keep<SPLIT, 1>(pb, st[1]);
          check_max(mx, c_scale, inv_c, slack, st[0]);

          read_k(h == 0 ? kt : kn, h ^ 1, fo, kf);
          pv<SPLIT>(vf, pb, sel, st[1]);
          exponents<0>(sa, c_scale, st[0], x0);
          exp_half<SPLIT, 0>(x0, st[0], pa);
          exponents<1>(sa, c_scale, st[0], xa);
          interleave<kPv, 8, 4>();
          keep<SPLIT, 0>(pa, st[0]);
          keep(xa);

          read_v(vt, h, fo, vf);
          qk(kf, qf[0], sa);
          exp_half<SPLIT, 1>(xa, st[0], pa);
          mx = row_max(sb);
          interleave<4, 10, 8>();
          keep<SPLIT, 1>(pa, st[0]);
          check_max(mx, c_scale, inv_c, slack, st[1]);

          pv<SPLIT>(vf, pa, sel, st[0]);
          exponents<0>(sb, c_scale, st[1], x0);
          exp_half<SPLIT, 0>(x0, st[1], pb);
          exponents<1>(sb, c_scale, st[1], xb);
          interleave<kPv, 8, 0>();
          keep<SPLIT, 0>(pb, st[1]);
          keep(xb);
        }
      }
      exp_half<SPLIT, 1>(xb, st[1], pb);
      pv<SPLIT>(vf, pb, sel, st[1]);
    }
    if (n_full * kTileKeys < wave_end) plain_tile(split_p, n_full);
  };
  auto finish = [&](int t) {  // the barriers of the tiles from t on
    for (; t < n_tiles; ++t) boundary(t);
    wait_loads<0>();
    __syncthreads();
  };

  bool split = short_rows;  // any wave of the block / this wave: a split-P pass
  bool wave_split = short_rows;
  if (!short_rows) {
    start();
    sweep(std::false_type{});
    finish(n_full);
    // The rounded-mass rule of prefill.hip, judged per wave: waves with a
    // peaky row run again with split P, the block's other waves keep their
    // rows and only load tiles.
    float *const verdicts = reinterpret_cast<float *>(lds);
    const int ln = fresh_lane();
    bool peaky = false;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const float l_row = st[g].lacc[0];
      const float r_row = st[g].r + __shfl_xor(st[g].r, 32);
      peaky = peaky || (qw0 + 32 * g + (ln & 31) < seq &&
                        r_row > kRedoRoundedMassAbove * l_row * l_row);
    }
    wave_split = __builtin_amdgcn_ballot_w64(peaky) != 0;
    if (ln == 0) verdicts[rw] = wave_split ? 1.0f : 0.0f;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWideWaves; ++w) split = split || verdicts[w] != 0.0f;
    __syncthreads();  // every wave has read the verdicts before the LDS is written again
  }
  if (split) {
    start();
    if (wave_split) sweep(std::true_type{});
    finish(wave_split ? n_full : 0);
  }

  // Epilogue: each group's 32 rows through the wave's staging area, stored as
  // whole rows (see prefill.hip). LDS operations of a wave complete in order,
  // so the second group may reuse the area without a barrier.
  using OutT = typename std::conditional<OUT_F32, float, _Float16>::type;
  constexpr int kRowBytes = kD * static_cast<int>(sizeof(OutT));
  constexpr int kChunksOut = kRowBytes / 16;
  constexpr int kRowsPerStore = kWave / kChunksOut;
  const int ln = fresh_lane();
  const int col = ln & 31, hg = ln >> 5;
  const int swz = col & (kChunksOut - 1);
  const int chunk = ln % kChunksOut;
  char *const stage = reinterpret_cast<char *>(lds) + rw * (32 * kRowBytes);
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const float l_tot = st[g].lacc[0];
    const float inv_l = l_tot > 0.f ? 1.0f / l_tot : 0.f;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        if constexpr (OUT_F32) {
          floatx4 r;
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] = st[g].o[db][4 * jj + e] * inv_l;
          *reinterpret_cast<floatx4 *>(stage + col * kRowBytes +
                                       16 * ((8 * db + 2 * jj + hg) ^ swz)) = r;
        } else {
          half4 r;
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] = static_cast<_Float16>(st[g].o[db][4 * jj + e] * inv_l);
          *reinterpret_cast<half4 *>(stage + col * kRowBytes + 16 * ((4 * db + jj) ^ swz) +
                                     8 * hg) = r;
        }
      }
#pragma unroll
    for (int i = 0; i < 32 / kRowsPerStore; ++i) {
      const int r = i * kRowsPerStore + ln / kChunksOut;
      const int row = qw0 + 32 * g + r;
      const floatx4 val = *reinterpret_cast<const floatx4 *>(
          stage + r * kRowBytes + 16 * (chunk ^ (r & (kChunksOut - 1))));
      if (row < seq)
        __builtin_nontemporal_store(
            val, reinterpret_cast<floatx4 *>(
                     reinterpret_cast<char *>(static_cast<OutT *>(o) + head_off +
                                              static_cast<size_t>(row) * kD) +
                     16 * chunk));
    }
  }
}

// Rounds of a grid of equal items over the 2 cu resident blocks, the last one
// at what it takes: a round with at most one block per CU runs ~0.62 of one
// with two.
float rounds(long long items, int cu) {
  const long long whole = items / (2 * cu), rest = items % (2 * cu);
  return static_cast<float>(whole) + (rest == 0 ? 0.f : rest <= cu ? 0.62f : 1.0f);
}

}  // namespace

// 256-row blocks against prefill.hip's one-half blocks of 128 rows. Per row
// they take ~0.87 of the time, but twice as long per block, so the rounds they
// leave half empty cost more (us, wide / one half, same box, B H S):
//   full: 8 12 4096 460 / 514, 40 12 1024 181 / 198, 2 14 4096 151 / 168,
//     4 14 2048 80 / 87; one round of wide blocks against 1.3 or 1.5 of narrow
//     ones: 3 14 2048 75 / 68, 8 12 1024 43 / 38;
//   causal (items of many lengths fill the rounds, but the blocks' plain
//     diagonal tiles and split-P rows weigh more on short sequences):
//     8 12 4096 261 / 276, 4 12 8192 476 / 514, 16 12 2048 157 / 163;
//     3.5 items per CU, 4 14 4096 161 / 159; 16 14 1024 66 / 57.
bool prefill_wide_pays(int bh, int seq, bool causal, int cu) {
  if (cu <= 0 || seq < 512) return false;
  const long long wide = static_cast<long long>(bh) * ((seq + kWideRows - 1) / kWideRows);
  const long long narrow = static_cast<long long>(bh) * ((seq + 127) / 128);
  if (causal) return seq >= 2048 && wide >= 5LL * cu;
  return narrow > 2LL * cu && 2.0f * rounds(wide, cu) < 1.15f * rounds(narrow, cu);
}

void launch_prefill_wide(const void *q, const void *k, const void *v, void *o, bool out_f32,
                         int bh, int seq, int group, bool causal, float c_scale, bool negate_q,
                         bool split_all, hipStream_t stream) {
  const int n_qtiles = (seq + kWideRows - 1) / kWideRows;
  const auto kernel = causal ? (out_f32 ? prefill_wide_kernel<true, true>
                                        : prefill_wide_kernel<true, false>)
                             : (out_f32 ? prefill_wide_kernel<false, true>
                                        : prefill_wide_kernel<false, false>);
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(bh) * n_qtiles), dim3(kWideThreads), 0,
                     stream, static_cast<const _Float16 *>(q), static_cast<const _Float16 *>(k),
                     static_cast<const _Float16 *>(v), o, seq, n_qtiles, bh, group, c_scale,
                     negate_q, split_all);
}

}  // namespace fa
