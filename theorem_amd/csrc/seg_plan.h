// How many segments a call of the segmented Gated DeltaNet recurrence is cut
// into (segments.h), and what workspace they take.  Host code without HIP: also
// compiled by the host-side checks.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace thm {
namespace {
namespace seg {

// Segments of a call: `out` of the output kernel, each of `per` transition
// segments of `len` chunks (the last may be shorter, none is empty).
struct Plan {
  int64_t out, per, len;
  int64_t segs(int64_t NT) const { return (NT + len - 1) / len; }
};

// What a plan costs, in us on MI355X (only the ratios matter): workgroups per
// (b, head) and segment and the serial period of a chunk in the transition and
// the output kernel, the combine kernel's start and step, and the period in one
// piece.
struct Costs {
  int64_t one_tiles, t_tiles, o_tiles;
  double one_period, t_period, c_start, c_step, o_period;
};

// The plan of least estimated time on `cu` CUs: a launch of workgroups that
// each walk n chunks takes a start that grows with the share of the CUs in use,
// and n periods; one CU holds one workgroup of these kernels (LDS), so more
// workgroups than CUs run in rounds.  Two segments never gain (the transitions
// of the first alone take about as long as its outputs); a plan has to save
// 5 %.
inline Plan plan_segments(int64_t BH, int64_t NT, const Costs& k, int64_t cu) {
  cu = std::max<int64_t>(cu, 1);
  auto launch = [&](int64_t wgs, double start, double period, int64_t chunks) {
    const double share = std::min(1.0, (double)wgs / cu);
    return (double)((wgs + cu - 1) / cu) * (start + 5.0 * share + period * chunks);
  };
  Plan best = {1, 1, std::max<int64_t>(NT, 1)};
  double t_best = 0.95 * launch(BH * k.one_tiles, 3.0, k.one_period, NT);
  for (int64_t out = 3; out <= 32 && out <= NT; ++out) {
    for (int64_t per = 1; per <= 4 && out * per <= NT; ++per) {
      const int64_t len = (NT + out * per - 1) / (out * per);
      const int64_t nt = (NT + len - 1) / len;  // transition segments
      const int64_t no = (nt + per - 1) / per;  // output segments
      if (no < 3) continue;
      const double t = launch(BH * (nt - 1) * k.t_tiles, 4.0, k.t_period, len) + k.c_start + k.c_step * (nt - 2) +
                       launch(BH * k.o_tiles * no, 3.0, k.o_period, len * per);
      if (t < t_best) {
        t_best = t;
        best = {no, per, len};
      }
    }
  }
  return best;
}

// Workspace of a plan: P of segments 1 .. nt - 2, the states and the redo
// flags, in bytes.
inline int64_t p_bytes(const Plan& p, int64_t BH, int64_t NT, int64_t K) {
  return p.out > 1 ? (p.segs(NT) - 2) * BH * K * K * 4 : 0;
}
inline int64_t s_bytes(const Plan& p, int64_t BH, int64_t NT, int64_t K, int64_t V) {
  return p.out > 1 ? (p.segs(NT) - 1) * BH * K * V * 4 : 0;
}
inline int64_t redo_bytes(const Plan& p, int64_t BH, int64_t V) { return p.out > 1 ? BH * (V / 16) * 4 : 0; }

// ---------------------------------------------------------------------------
// The bf16 forward from chunk records (chunk_fwd_rec.hip).  Measured at K = V
// = 128: period 2.0-2.1 us (outputs), 2.3-2.4 (transitions), 1.65 per combine
// step; the combine kernel's start is larger at K = 128, where a step reads 64
// KB of P.  Whole forwards, in one piece -> best of five plans of one transition
// segment per output segment -> this rule, us:
//   K = V = 128: 16 heads, 32 chunks 77 -> 54 -> 55, 128 chunks 274 -> 119 ->
//     120; 32 heads, 32 chunks 82 -> 70 -> 73; 4 heads, 64 chunks 139 -> 63 -> 63;
//   K = V = 64: 16 heads, 12 chunks 27.6 -> 23.5 -> 23.5; 32 heads, 16 chunks 36
//     -> 28.5 -> 28.5; 4 heads, 64 chunks 111 -> 37 -> 37; 63 heads, 24 chunks
//     56 -> 50 -> 51.
// 128 workgroups or more in one piece do not gain at K = 128 (64 heads, 32
// chunks: 86, 96 at best), nor do short sequences: with a start of 3 us, 40
// heads, 32 chunks 83 -> 90, 12 heads, 16 chunks 43 -> 45.
inline Plan plan_fwd(int64_t BH, int64_t NT, int64_t K, int64_t V, int64_t cu) {
  const int64_t nvt = V / 64;
  return plan_segments(BH, NT, {nvt, 1, nvt, 2.02, 2.4, K == 128 ? 5.0 : 3.0, K == 128 ? 1.65 : 0.9, 2.1}, cu);
}

// V-tile width of the fp32 delta form's segment launches.  Staging a chunk of k and
// w (an fp32 -> bf16 hi + lo split of each) and its barriers take a large part
// of a period and the LDS stage leaves one workgroup per CU: where P and V both
// make whole tiles of 128, twice the waves share them (period 4.7 us for 64
// columns -> 5.3 for 128).  B = 2, T = 2048, H = 8: transitions 42.4 -> 27.7 us,
// outputs 37.2 -> 30.5, combine 8.4 -> 13.3 (8 segments instead of 5).
constexpr int h_seg_cols(int64_t K, int64_t V) { return K == 128 && V == 128 ? 128 : 64; }

// chunk_fwd_h, delta form; one piece on grids that fill the GPU without
// segments (256 workgroups of 64 columns).  In one piece -> this rule, us; the
// first figure with k, w and u in the 256 MiB memory-side cache (as the kernel
// that wrote them leaves them), the second from HBM:
//   bf16, the small-grid kernel against transitions and the DMA kernel: K = V =
//     128, 16 heads, 128 chunks 139 -> 114, 225 -> 131; 4 heads, 128 chunks 137
//     -> 74, 175 -> 83; K = V = 64, 3 heads, 128 chunks 86 -> 38, 113 -> 42.
//     From the cache a chunk in one piece takes 1.1 us at K = 128 and 0.75 at K
//     = 64, from HBM 1.4 and 1.2: the rule's periods lie between, so that
//     neither loses.  At K = 64, V = 128, whose segments cost more than V = 64's
//     and save less, calls that fit the cache are reckoned nearer to it: 12
//     heads, 32 chunks 26 -> 31 with segments, 32 heads, 96 chunks 70 -> 85, but
//     128 chunks (past the cache) 183 -> 119;
//   fp32, register kernel (at K = 64 the small-grid kernel in one piece): 16
//     heads of K = V = 128, 32 chunks 137 -> 81 -> 80, 4 heads, 64 chunks 268
//     -> 74 -> 74; 16 heads of K = V = 64, 64 chunks 97 -> 50 -> 50.  With 128
//     columns a workgroup (h_seg_cols; kernel trace, sums of the three
//     launches): 16 heads, 32 chunks 71, 4 heads, 64 chunks 77, 8 heads, 128
//     chunks 126 (530 in one piece), 32 heads, 16 chunks 60 (72).
inline Plan plan_h(int64_t BH, int64_t NT, int64_t K, int64_t V, bool f32, int64_t cu) {
  const int64_t nvt = V / 64;
  if (f32) {
    if (h_seg_cols(K, V) == 128)
      return plan_segments(BH, NT, {nvt, (K + V) / 128, V / 128, 4.7, 5.3, 3.0, 1.65, 6.4}, cu);
    const double period = K == 128 ? 4.7 : 2.5;
    return plan_segments(BH, NT, {nvt, (K + V) / 64, nvt, K == 128 ? period : 1.7, period, 3.0, 1.2, period}, cu);
  }
  const int64_t bytes = BH * NT * (64 * 2 * (2 * K + 2 * V) + K * V * 4);  // k, w, u, v_new; h
  const double one = K == 64 && V == 128 && bytes <= (INT64_C(1) << 28) ? 1.05 : 1.2;
  return plan_segments(BH, NT, {V / 32, 1, nvt, one, 2.2, K == 128 ? 5.0 : 3.0, K == 128 ? 1.65 : 0.9, 2.6}, cu);
}

}  // namespace seg
}  // namespace
}  // namespace thm
