// Segments of the Gated DeltaNet state recurrence (gfx950): the state at the
// start of each of several segments of a sequence, so that the segments can
// run side by side (chunk_fwd_rec.hip, chunk_fwd_h.hip).
//
// A chunk maps the state S affinely, so a segment of chunks maps it to P S + Q
// with P [K x K] and Q [K x V].  The columns of a state evolve independently:
// the transition kernel forms [P | Q] as the same recurrence on K + V columns
// that start from [I | 0] (segment 0: only Q, from h0), every segment at once,
// and the combine kernel runs S <- P S + Q over the segments.
#pragma once

#include "h_layout.h"
#include "mfma.h"
#include "rec_cfg.h"
#include "seg_plan.h"
#include "vmem.h"

namespace thm {
namespace {
namespace seg {

using rec::kBT;
using rec::kTileV;

// A operand of 16-row block ib, contraction step s2 (32 elements, paired
// order), of a swizzled [64 x K] tile (h_layout.h).
__device__ __forceinline__ bf16x8 row_frag(const char* tile, int ib, int s2, int lane, int row_bytes) {
  // (volatile: merged two-address reads land in registers that must then be copied together)
  typedef const volatile __attribute__((address_space(3))) u32x2 piece;
  const u32x2 a = *(piece*)(tile + hl::pair_frag_off(16 * ib, 32 * s2, lane, row_bytes));
  const u32x2 b = *(piece*)(tile + hl::pair_frag_off(16 * ib, 32 * s2 + 16, lane, row_bytes));
  return __builtin_bit_cast(bf16x8, u32x4{a[0], a[1], b[0], b[1]});
}

// A operands of row block ib, contraction step s2, of the record's A: hi and
// lo.  Block (ib, 2 s2 + 1) lies above the diagonal for ib = 2 s2: zero.
__device__ __forceinline__ void a_frags(const char* r, int ib, int s2, int lane, bf16x8& ah, bf16x8& al) {
  const int p = rec::block(ib, 2 * s2);
  const u32x4 x0 = *reinterpret_cast<const u32x4*>(r + p * rec::kBlockBytes + 16 * lane);
  u32x4 x1 = {0u, 0u, 0u, 0u};
  if (2 * s2 + 1 <= ib) x1 = *reinterpret_cast<const u32x4*>(r + (p + 1) * rec::kBlockBytes + 16 * lane);
  ah = __builtin_bit_cast(bf16x8, u32x4{x0[0], x0[1], x1[0], x1[1]});
  al = __builtin_bit_cast(bf16x8, u32x4{x0[2], x0[3], x1[2], x1[3]});
}

__device__ __forceinline__ bf16x8 pair_bf16(f32x4 a, f32x4 b) {
  const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  return to_bf16x8(f);
}

// k^T fragment (16 state rows kb, chunk rows 32 s2 .. + 31, paired order).
__device__ __forceinline__ bf16x8 kT_frag(const char* tk, int kb, int s2, int lane, int row_bytes) {
  return concat(ds_read_tr16(reinterpret_cast<const bf16*>(tk + hl::tr_frag_off(32 * s2, 16 * kb, lane, row_bytes))),
                ds_read_tr16(reinterpret_cast<const bf16*>(tk + hl::tr_frag_off(32 * s2 + 16, 16 * kb, lane, row_bytes))));
}

// Chunks of segment `seg` when NT chunks are cut into `nseg` of `len` (the last may be shorter).
struct Span {
  int64_t c0, n;
};
__device__ __forceinline__ Span span_of(int64_t seg, int64_t len, int64_t NT) {
  const int64_t c0 = seg * len;
  return {c0, NT - c0 < len ? NT - c0 : len};
}

// ---------------------------------------------------------------------------
// Transition kernel: [P | Q] of segments 0 .. nseg - 2.  One workgroup per
// (b, head, segment), wave w on 32 columns: waves below K / 32 on P, the rest
// on Q.  Each wave runs the whole recurrence of its columns from the staged
// chunk (DMA'd two chunks ahead into a 3-stage ring), so the waves share
// nothing but the tiles and one barrier per chunk.  From the record (v_new =
// A (beta (v - e^g k S)), vw = v) or, WU, from w and u (v_new = u - w S, vw =
// u, g the gates or nullptr).  Two
// 16-column tiles per wave: each LDS fragment feeds two products (one tile
// per wave would double the LDS reads, which take about as long as the MFMAs).
template <int K, int V, bool WU, bool HAS_G>
__global__ void __launch_bounds__((rec::TCfg<K, V, WU>::kThreads))
chunk_transition_kernel(const bf16* __restrict__ k, const bf16* __restrict__ w, const bf16* __restrict__ vw,
                        const float* __restrict__ g, const char* __restrict__ records,
                        const float* __restrict__ h0, char* __restrict__ pbuf, char* __restrict__ sbuf, int64_t T,
                        int64_t H, int64_t NT, int64_t BH, int64_t len) {
  using C = rec::TCfg<K, V, WU>;
  constexpr int KB = K / 16, KB2 = KB / 2, CT = C::kCT;
  __shared__ __attribute__((aligned(1024))) char lds[C::kLds];

  const int64_t seg = blockIdx.x / BH, bh = blockIdx.x - seg * BH;
  const int64_t b = bh / H, hh = bh - b * H;
  const Span sp = span_of(seg, len, NT);

  const int tid = threadIdx.x;
  const int wi = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, grp = lane >> 4, li = lane & 15;
  const bool is_p = wi < C::kPWaves;
  const bool active = !(is_p && seg == 0);  // segment 0 starts from a known state: no P
  const int n0 = 16 * CT * (is_p ? wi : wi - C::kPWaves);

  // v of this wave's columns; a wave of P reads any and masks it to zero (no
  // branch between the products).
  const int v_tile = is_p ? 0 : (n0 / kTileV) * C::kTileVB, vc = n0 % kTileV;
  const uint32_t vmask = is_p ? 0u : ~0u;

  const int64_t tsk = H * K * 2, tsv = H * V * 2;
  const char* const k0 = reinterpret_cast<const char*>(k) + ((b * T + sp.c0 * kBT) * H + hh) * K * 2;
  const char* const v0 = reinterpret_cast<const char*>(vw) + ((b * T + sp.c0 * kBT) * H + hh) * V * 2;
  // The third source: the records, or the w rows.
  const char* const r0 = WU ? reinterpret_cast<const char*>(w) + ((b * T + sp.c0 * kBT) * H + hh) * K * 2
                            : records + rec::offset(bh, sp.c0, NT);
  const int64_t rcs = WU ? kBT * tsk : rec::kBytes;
  const char* const g0 = WU && HAS_G ? reinterpret_cast<const char*>(g) + ((b * T + sp.c0 * kBT) * H + hh) * 4 : nullptr;

  // This wave's DMA instructions of a chunk: j = wi + i kWaves of the list
  // (k tile, v tiles, record or w tile), each to its KiB of the stage; wave 0
  // also gathers the gates for WU.
  uint32_t voff[C::kDma], loff[C::kDma];
  bool from_k[C::kDma], from_v[C::kDma];
#pragma unroll
  for (int i = 0; i < C::kDma; ++i) {
    const int j = wi + i * C::kWaves;
    from_k[i] = C::from_k(j);
    from_v[i] = C::from_v(j);
    voff[i] = C::src_off(j, lane, tsk, tsv);
    loff[i] = (uint32_t)(j * 1024);
  }
  const bool last_dma = wi + (C::kDma - 1) * C::kWaves < C::kInstr;  // else one instruction fewer
  // Chunk c into the stage at byte `st`.
  auto issue = [&](int64_t c, uint32_t st) {
    const char* kb = k0 + c * kBT * tsk;
    const char* vb = v0 + c * kBT * tsv;
    const char* rb = r0 + c * rcs;
    const uint32_t l0 = lds_address(lds) + st;
#pragma unroll
    for (int i = 0; i < C::kDma; ++i)
      if (i + 1 < C::kDma || last_dma)
        dma_b128(from_k[i] ? kb : from_v[i] ? vb : rb, voff[i], __builtin_amdgcn_readfirstlane(l0 + loff[i]));
    if constexpr (WU && HAS_G) {
      if (wi == 0)
        dma_b32(g0 + c * kBT * H * 4, (uint32_t)(lane * H * 4), __builtin_amdgcn_readfirstlane(l0 + C::kInstr * 1024));
    }
  };

  issue(0, 0);
  issue(sp.n > 1 ? 1 : 0, C::kStage);

  // S[ct][kb]: rows 16 kb + 4 grp + r of column n0 + 16 ct + li.
  f32x4 S[CT][KB];
  if (is_p) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[ct][kb][r] = 16 * kb + 4 * grp + r == n0 + 16 * ct + li ? 1.f : 0.f;
  } else if (seg == 0 && h0) {
    const float* hp = h0 + bh * (int64_t)(K * V) + 4 * grp * V + n0 + li;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[ct][kb][r] = hp[(16 * kb + r) * V + 16 * ct];
  } else {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) S[ct][kb] = zero4();
  }
  wait_vmcnt<0>();  // h0 and the first tiles; the loop counts from here

  // Stages of chunk c (st) and of chunk c + 2 (sn), by rotation.
  uint32_t st = 0, sn = 2 * C::kStage;
  auto next = [](uint32_t x) { return x == (C::kStages - 1) * C::kStage ? 0u : x + C::kStage; };
  for (int64_t c = 0; c < sp.n; ++c, st = next(st), sn = next(sn)) {
    if (WU && HAS_G && wi == 0) wait_vmcnt<C::kWait + (C::kStages - 2)>();
    else if (last_dma) wait_vmcnt<C::kWait>();
    else wait_vmcnt<C::kWait - (C::kStages - 2)>();
    lds_barrier();  // chunk c is in LDS; every wave is done with chunk c - 1
    {
      const int64_t cn = c + 2;  // into chunk c - 1's stage (a repeat of the last chunk at the end)
      issue(cn < sp.n ? cn : sp.n - 1, sn);
    }
    if (!active) continue;
    const char* tk = lds + st;
    const char* tv = tk + C::kOffV + v_tile;
    const char* tr = tk + C::kOffR;  // the record, or the w tile
    const float* gp = reinterpret_cast<const float*>(tk + C::kOffG);

    bf16x8 sb[CT][KB2];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int s2 = 0; s2 < KB2; ++s2) sb[ct][s2] = pair_bf16(S[ct][2 * s2], S[ct][2 * s2 + 1]);
    // Every product phase runs contraction step by step over all its
    // accumulators (8 or 16 independent MFMA chains), not block by block.
    f32x4 vn[CT][4];
    // Rows 16 jb + 4 grp .. + 3 of v or u of this lane's column of tile ct.
    auto v_rows = [&](int jb, int ct) {
      u32x2 vb = __builtin_bit_cast(
          u32x2, ds_read_tr16(reinterpret_cast<const bf16*>(tv + hl::tr_frag_off(16 * jb, vc + 16 * ct, lane, C::kRowV))));
      return __builtin_bit_cast(bf16x4, vb & vmask);
    };
    if constexpr (WU) {
      // v_new = u - w S; no u in the columns of P.
#pragma unroll
      for (int s2 = 0; s2 < KB2; ++s2) {
#pragma unroll
        for (int jb = 0; jb < 4; ++jb) {
          const bf16x8 wf = row_frag(tr, jb, s2, lane, C::kRowK);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) vn[ct][jb] = mfma16x16x32(wf, sb[ct][s2], s2 ? vn[ct][jb] : zero4());
        }
      }
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const bf16x4 uu = v_rows(jb, ct);
#pragma unroll
          for (int r = 0; r < 4; ++r) vn[ct][jb][r] = (float)uu[r] - vn[ct][jb][r];
        }
    } else {
      // k S.
      f32x4 t4[CT][4];
#pragma unroll
      for (int s2 = 0; s2 < KB2; ++s2) {
#pragma unroll
        for (int jb = 0; jb < 4; ++jb) {
          const bf16x8 kf = row_frag(tk, jb, s2, lane, C::kRowK);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) t4[ct][jb] = mfma16x16x32(kf, sb[ct][s2], s2 ? t4[ct][jb] : zero4());
        }
      }
      // t = beta (v - e^g k S); no v in the columns of P.
      bf16x8 tp[CT][2];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        const f32x4 bt = *reinterpret_cast<const f32x4*>(gp + rec::kBeta + 16 * jb + 4 * grp);
        const f32x4 eg = *reinterpret_cast<const f32x4*>(gp + rec::kEg + 16 * jb + 4 * grp);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const bf16x4 vv = v_rows(jb, ct);
#pragma unroll
          for (int r = 0; r < 4; ++r) t4[ct][jb][r] = bt[r] * ((float)vv[r] - eg[r] * t4[ct][jb][r]);
          if (jb & 1) tp[ct][jb / 2] = pair_bf16(t4[ct][jb - 1], t4[ct][jb]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // hoisting the next phase's reads further spills at K = 128
      // v_new = A t.
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        bf16x8 ah[4], al[4];
#pragma unroll
        for (int ib = 2 * s2; ib < 4; ++ib) a_frags(tr, ib, s2, lane, ah[ib], al[ib]);
#pragma unroll
        for (int ib = 2 * s2; ib < 4; ++ib)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) vn[ct][ib] = mfma16x16x32(ah[ib], tp[ct][s2], s2 ? vn[ct][ib] : zero4());
#pragma unroll
        for (int ib = 2 * s2; ib < 4; ++ib)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) vn[ct][ib] = mfma16x16x32(al[ib], tp[ct][s2], vn[ct][ib]);
      }
    }
    // Scaled by e^{g_last - g}, as the B operand.
    bf16x8 vh[CT][2];
    float decay = 1.f;
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      f32x4 fa = {1.f, 1.f, 1.f, 1.f}, fb = fa;
      if constexpr (WU && HAS_G) {
        const float gl = gp[kBT - 1];
        fa = *reinterpret_cast<const f32x4*>(gp + 32 * s2 + 4 * grp);
        fb = *reinterpret_cast<const f32x4*>(gp + 32 * s2 + 16 + 4 * grp);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          fa[r] = fast_exp(gl - fa[r]);
          fb[r] = fast_exp(gl - fb[r]);
        }
        decay = fast_exp(gl);
      } else if constexpr (!WU) {
        fa = *reinterpret_cast<const f32x4*>(gp + rec::kEgl + 32 * s2 + 4 * grp);
        fb = *reinterpret_cast<const f32x4*>(gp + rec::kEgl + 32 * s2 + 16 + 4 * grp);
        decay = gp[rec::kEg + kBT - 1];
      }
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) vh[ct][s2] = pair_bf16(vn[ct][2 * s2] * fa, vn[ct][2 * s2 + 1] * fb);
    }
    __builtin_amdgcn_sched_barrier(0);
    // S = e^{g_last} S + k^T v_new.
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const bf16x8 kt = kT_frag(tk, kb, s2, lane, C::kRowK);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          if (s2 == 0) S[ct][kb] *= decay;
          S[ct][kb] = mfma16x16x32(kt, vh[ct][s2], S[ct][kb]);
        }
      }
  }
  wait_vmcnt<0>();  // no DMA may still target this workgroup's LDS when it exits
  if (!active) return;

  // P in 16 x 16 blocks (row block, column block) of A-operand lanes (rec_cfg.h
  // p_slot), Q in blocks (column block, row block) of accumulator lanes.
  if (is_p) {
    const int slot = rec::p_slot(lane);
    char* const pb = pbuf + rec::p_off(seg, bh, BH, K) + (n0 / 16) * 1024 + 16 * slot;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        *reinterpret_cast<f32x4*>(pb + (kb * KB + ct) * 1024) = acc_to_row_quads(S[ct][kb]);
  } else {
    char* const sb = sbuf + rec::s_off(seg, bh, BH, K, V) + (n0 / 16) * KB * 1024 + 16 * lane;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) *reinterpret_cast<f32x4*>(sb + (ct * KB + kb) * 1024) = S[ct][kb];
  }
}

// ---------------------------------------------------------------------------
// Combine kernel: S_{s+1} = P_s S_s + Q_s for s = 1 .. nseg - 2, in place of
// Q_s (S_1 = Q_0).  One workgroup of K / 16 wavefronts per (b, head, 16
// columns); wave w forms row tile w of the new state and hands it to the
// others through LDS.  P and S as fp32 on v_mfma_f32_16x16x4_f32, exact
// products: the state is carried in fp32 from one end of a sequence to the
// other, as in one piece.  A serial chain of small steps: P and Q of the next
// two steps are in flight during one, and the products run in two accumulators.
// A segment's map can overflow where the states of the sequence do not (a
// column that is zero stays zero whatever P is), and P S is then no number:
// where any state of the 16 columns is not finite, redo[bh V / 16 + vt] says so
// and the kernels that walk the segments take those columns in one piece.
template <int K, int V>
__global__ void __launch_bounds__(4 * K)
chunk_combine_kernel(const char* __restrict__ pbuf, char* __restrict__ sbuf, uint32_t* __restrict__ redo, int64_t BH,
                     int64_t nseg) {
  constexpr int KB = K / 16, NVB = V / 16;
  constexpr int kAhead = 2;
  __shared__ __attribute__((aligned(16))) f32x4 xs[2][KB][64];  // one row tile's 4 rows per lane
  __shared__ uint32_t over[KB];
  const hl::BhTile bt = hl::xcd_tile(blockIdx.x, BH, NVB);  // one XCD reads one (b, head)'s P
  const int wi = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;

  auto q_at = [&](int64_t s) {
    return reinterpret_cast<f32x4*>(sbuf + rec::s_off(s, bt.bh, BH, K, V) + (bt.vt * KB + wi) * 1024 + 16 * lane);
  };
  f32x4 qn[kAhead];
  f32x4 pn[kAhead][KB];
  auto load = [&](int64_t s, int i) {
    qn[i] = *q_at(s);
    const char* pb = pbuf + rec::p_off(s, bt.bh, BH, K) + wi * KB * 1024 + 16 * lane;
#pragma unroll
    for (int nb = 0; nb < KB; ++nb) pn[i][nb] = *reinterpret_cast<const f32x4*>(pb + nb * 1024);
  };
  const int64_t last = nseg - 2;
  f32x4 S = *q_at(0);
  uint32_t top = 0;  // the largest magnitude's bits: infinities and NaN lie above every finite one
#pragma unroll
  for (int i = 0; i < kAhead; ++i) load(1 + i < last ? 1 + i : last, i);
  auto step = [&](int64_t s, int i) {
    const int f = (int)(s & 1);
    xs[f][wi][lane] = S;
    f32x4 p[KB];
#pragma unroll
    for (int nb = 0; nb < KB; ++nb) p[nb] = pn[i][nb];
    f32x4 acc[2] = {qn[i], zero4()};
    load(s + kAhead < last ? s + kAhead : last, i);
    lds_barrier();  // S_s is in LDS (the other buffer's readers finished before this barrier)
#pragma unroll
    for (int nb = 0; nb < KB; ++nb) {
      const f32x4 x = xs[f][nb][lane];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc[nb & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[nb][q], x[q], acc[nb & 1], 0, 0, 0);
    }
    S = acc[0] + acc[1];
    *q_at(s) = S;
#pragma unroll
    for (int r = 0; r < 4; ++r) top = max(top, __float_as_uint(S[r]) & 0x7fffffffu);
  };
  for (int64_t s = 1; s <= last; s += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (s + i <= last) step(s + i, i);  // uniform over the workgroup
  }
  const bool any = __any(top >= 0x7f800000u);
  if (lane == 0) over[wi] = any;
  lds_barrier();
  if (threadIdx.x == 0) {
    uint32_t o = 0;
#pragma unroll
    for (int i = 0; i < KB; ++i) o |= over[i];
    redo[bt.bh * NVB + bt.vt] = o;
  }
}

// Whether the columns [v0, v0 + cols) of sequence bh are walked in one piece
// after all (segment 0 takes every chunk, the others none).
template <int V>
__device__ __forceinline__ bool redo_columns(const uint32_t* redo, int64_t bh, int v0, int cols) {
  const uint32_t* p = redo + bh * (V / 16) + v0 / 16;
  uint32_t o = 0;
#pragma unroll
  for (int i = 0; i < cols / 16; ++i) o |= p[i];
  return o != 0;
}

// ---------------------------------------------------------------------------

}  // namespace seg
}  // namespace
}  // namespace thm
