// What the prefill kernels share: the precision rules of P and of the running
// max, and the block -> head placement.
#pragma once

#include "fa_internal.h"

namespace fa {

// head_dim 64 on large grids, 64 query rows per wave (prefill_wide.hip):
// whether a shape takes it, and its launch (the arguments of launch_d).
bool prefill_wide_pays(int bh, int seq, bool causal, int cu);
void launch_prefill_wide(const void *q, const void *k, const void *v, void *o, bool out_f32,
                         int bh, int seq, int group, bool causal, float c_scale, bool negate_q,
                         bool split_all, hipStream_t stream);

namespace {

[[maybe_unused]] constexpr int kSplitPRowsBelow = 256;  // rows with fewer keys than this: split P
// A block is recomputed with split P when, for one of its rows, the squared
// normalised weights that took a single fp16 rounding sum to more than this
// (see the precision note at the top of prefill.hip).
[[maybe_unused]] constexpr float kRedoRoundedMassAbove = 0.03f;
// |scale| * sqrt(D) above this (1 is the standard 1/sqrt(D)): rows are peaky
// from the scale alone, so the first (single-rounding) pass is skipped.
[[maybe_unused]] constexpr float kSplitAllWidth = 1.5f;  // used by the head_dim 64 build
[[maybe_unused]] constexpr float kNegHuge = -3.0e38f;
// The max that P is taken against moves only when a row's tile max exceeds it
// by more than this (log2 units), so P <= 2^8 and O is rescaled on few steps...
[[maybe_unused]] constexpr float kLazyMaxSlack = 8.0f;
// ...or when the tile max's weight exceeds this fraction of the row sum so
// far: a key that carries a large share of its row is then taken at the exact
// max, where its P = 1 is exact and leaves the rounded mass.
[[maybe_unused]] constexpr float kLazyMaxDominant = 1.0f / 16;
[[maybe_unused]] constexpr int kLazyMaxRowsFrom = 1024;  // keys a row sees (at least) to take the lazy max

// The lane index read afresh from the hardware (v_mbcnt, in volatile asm so
// that the compiler cannot merge it with the kernel's first lane index). The
// code after the main loop (masked tail, verdict, epilogue) derives its
// per-lane values from this instead of from values computed before the loop,
// which the compiler otherwise keeps live across it: at 256 VGPRs they went
// to scratch (5 per lane at head_dim 64, 11-15 at 128), each item stored and
// reloaded them, and their write-backs were 2.5-3.4 MB of a C3 launch's HBM
// writes (C3 46.2 -> 45.8 us, C2 full 27.1 -> 26.4 us without them).
__device__ __forceinline__ int fresh_lane() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

// Block -> (b, h) with XCD affinity. The grid stays in level-major order
// (every head's heaviest query tile first), and blocks go to the 8 XCDs
// round-robin (block i on XCD i % 8). Head h is "at home" on XCD h % 8:
// within a level each XCD fills its positions with its home heads first and
// the leftover heads take the spare positions in a fixed order, so most of a
// head's blocks share one XCD's L2 (for 14 heads, 89 % of the blocks).
__host__ __device__ __forceinline__ int home_head(int i, int n_bh) {
  const int level = i / n_bh;
  const int k = i - level * n_bh;
  const int base = (level * n_bh) & 7;
  const int x = (base + k) & 7;     // XCD of this block
  const int d_x = (x - base) & 7;   // first position of XCD x in this level
  const int r = (k - d_x) >> 3;     // rank of position k among XCD x's
  const int nhome_x = (n_bh - x + 7) >> 3;
  if (r < nhome_x) return x + 8 * r;
  // A spare position: its index among all spares (XCDs in order, then rank)
  // selects the matching overflow head (XCDs in order, then head rank).
  int s = r - nhome_x;
  for (int y = 0; y < x; ++y) {
    const int npos = (n_bh - ((y - base) & 7) + 7) >> 3;
    const int nhome = (n_bh - y + 7) >> 3;
    s += npos > nhome ? npos - nhome : 0;
  }
  for (int y = 0; y < 8; ++y) {
    const int npos = (n_bh - ((y - base) & 7) + 7) >> 3;
    const int nhome = (n_bh - y + 7) >> 3;
    const int over = nhome > npos ? nhome - npos : 0;
    if (s < over) return y + 8 * (npos + s);
    s -= over;
  }
  return 0;  // unreachable: spare positions and overflow heads are equal in number
}

// Grouped queries: the placement heads of XCD x (x, x + 8, x + 16, ...) are
// given a contiguous run of query heads, in XCD order, so the query heads
// that read one K/V head (consecutive indices) mostly share an XCD and its
// L2 holds one copy of that K/V head.
__host__ __device__ __forceinline__ int grouped_head(int h, int n_bh) {
  const int x = h & 7;
  int start = 0;
  for (int y = 0; y < x; ++y) start += (n_bh - y + 7) >> 3;
  return start + (h >> 3);
}

}  // namespace
}  // namespace fa
