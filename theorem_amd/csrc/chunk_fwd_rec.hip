// Whole chunked Gated DeltaNet forward for MI355X (gfx950) from (q, k, v,
// beta, gate): o and the final state, bf16 q, k, v.  Per (b, head), state S
// [K x V] fp32 (h0 or 0), per 64-token chunk c with A = (I + M)^{-1},
// M[i][j] = beta_i (k_i . k_j) e^{g_i - g_j} (j < i) and g_last the chunk's
// last gate:
//   v_new = A (beta (v - e^g k S))
//   o     = scale ( e^{g_i} q_i . S  +  sum_{j <= i} (q_i . k_j) e^{g_i - g_j} v_new_j )
//   S    <- e^{g_last} S + (k e^{g_last - g})^T v_new
// i.e. `_build_A`, recompute_w_u, chunk_fwd_h (delta form) and chunk_fwd_o of
// the reference (kernels/recompute_w_u/reference.py:48-149,
// kernels/chunk_fwd_h/kernel.py:61-138, kernels/chunk_fwd_o/kernel.py:52-136)
// with nothing between them but the chunk records (rec_cfg.h).
//
// Launches:
//   1. records (wy_build_A.hip): A, gates and factors of every chunk;
//   2. where the sequences alone leave the GPU idle, the state at the start of
//      each of several segments of the sequences (transition and combine
//      kernels below);
//   3. the output kernel, one workgroup per (b, head, segment, 64-column
//      V-tile).
//
// Segments.  A chunk maps S to (e^{g_last} I - ...) S + ..., so a segment of
// chunks maps it to P S + Q with P [K x K] and Q [K x V].  The columns of a
// state evolve independently, so the transition kernel forms [P | Q] as the
// same recurrence on K + V columns that start from [I | 0] (segment 0: only
// Q, from h0), every segment at once.  The combine kernel then runs
// S <- P S + Q over the segments.  The extra work is less than twice the recurrence's own,
// against a serial chain shorter by the number of segments: B = 1, T = 8192,
// H = 16, K = V = 128 (32 workgroups of 128 chunks without segments)
// 276 -> 107 us for the whole forward.
#include <algorithm>

#include "h_layout.h"
#include "mfma.h"
#include "rec_cfg.h"
#include "vmem.h"

namespace thm {

// wy_build_A.hip
hipError_t build_records(int64_t K, const void* k, const void* beta, const void* gate, int gate_mode,
                         void* records, int64_t B, int64_t T, int64_t H, hipStream_t s);

namespace {

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
  const int p = ib * (ib + 1) / 2 + 2 * s2;
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
// chunk (k, v and the record, DMA'd two chunks ahead into a 3-stage ring), so
// the waves share nothing but the tiles and one barrier per chunk.  Two
// 16-column tiles per wave: each LDS fragment feeds two products (one tile
// per wave would double the LDS reads, which take about as long as the MFMAs).
template <int K, int V>
__global__ void __launch_bounds__((rec::TCfg<K, V>::kThreads))
chunk_transition_kernel(const bf16* __restrict__ k, const bf16* __restrict__ v, const char* __restrict__ records,
                        const float* __restrict__ h0, char* __restrict__ pbuf, char* __restrict__ sbuf, int64_t T,
                        int64_t H, int64_t NT, int64_t BH, int64_t len) {
  using C = rec::TCfg<K, V>;
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
  const char* const v0 = reinterpret_cast<const char*>(v) + ((b * T + sp.c0 * kBT) * H + hh) * V * 2;
  const char* const r0 = records + rec::offset(bh, sp.c0, NT);

  // This wave's DMA instructions of a chunk: j = wi + i kWaves of the list
  // (k tile, v tiles, record).  Lane offset, LDS offset and source per i.
  uint32_t voff[C::kDma], loff[C::kDma];
  bool from_k[C::kDma], from_v[C::kDma];
#pragma unroll
  for (int i = 0; i < C::kDma; ++i) {
    const int j = wi + i * C::kWaves;
    constexpr int kPer = C::kTileVB / 1024;  // instructions per v tile
    from_k[i] = j < C::kKInstr;
    from_v[i] = !from_k[i] && j < C::kKInstr + C::kVInstr;
    const int x = from_k[i] ? j : from_v[i] ? j - C::kKInstr : j - C::kKInstr - C::kVInstr;
    voff[i] = from_k[i]   ? hl::dma_src_off(x * 64 + lane, C::kRowK, tsk)
              : from_v[i] ? hl::dma_src_off((x % kPer) * 64 + lane, C::kRowV, tsv) + (uint32_t)((x / kPer) * C::kRowV)
                          : (uint32_t)(x * 1024 + lane * 16);
    loff[i] = (uint32_t)(j * 1024);  // the stage holds the tiles in the list's order
  }
  const bool last_dma = wi + (C::kDma - 1) * C::kWaves < C::kInstr;  // else one instruction fewer
  // Chunk c into the stage at byte `st`.
  auto issue = [&](int64_t c, uint32_t st) {
    const char* kb = k0 + c * kBT * tsk;
    const char* vb = v0 + c * kBT * tsv;
    const char* rb = r0 + c * rec::kBytes;
    const uint32_t l0 = lds_address(lds) + st;
#pragma unroll
    for (int i = 0; i < C::kDma; ++i)
      if (i + 1 < C::kDma || last_dma)
        dma_b128(from_k[i] ? kb : from_v[i] ? vb : rb, voff[i], __builtin_amdgcn_readfirstlane(l0 + loff[i]));
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
    if (last_dma) wait_vmcnt<C::kWait>();
    else wait_vmcnt<C::kWait - (C::kStages - 2)>();
    lds_barrier();  // chunk c is in LDS; every wave is done with chunk c - 1
    {
      const int64_t cn = c + 2;  // into chunk c - 1's stage (a repeat of the last chunk at the end)
      issue(cn < sp.n ? cn : sp.n - 1, sn);
    }
    if (!active) continue;
    const char* tk = lds + st;
    const char* tv = tk + C::kTileK + v_tile;
    const char* tr = tk + C::kTileK + C::kNVT * C::kTileVB;
    const float* gp = reinterpret_cast<const float*>(tr + rec::kGateOff);

    bf16x8 sb[CT][KB2];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int s2 = 0; s2 < KB2; ++s2) sb[ct][s2] = pair_bf16(S[ct][2 * s2], S[ct][2 * s2 + 1]);
    // Every product phase runs contraction step by step over all its
    // accumulators (8 or 16 independent MFMA chains), not block by block.
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
        u32x2 vb = __builtin_bit_cast(
            u32x2, ds_read_tr16(reinterpret_cast<const bf16*>(tv + hl::tr_frag_off(16 * jb, vc + 16 * ct, lane, C::kRowV))));
        vb &= vmask;
        const bf16x4 vv = __builtin_bit_cast(bf16x4, vb);
#pragma unroll
        for (int r = 0; r < 4; ++r) t4[ct][jb][r] = bt[r] * ((float)vv[r] - eg[r] * t4[ct][jb][r]);
        if (jb & 1) tp[ct][jb / 2] = pair_bf16(t4[ct][jb - 1], t4[ct][jb]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // hoisting the next phase's reads further spills at K = 128
    // v_new = A t, then scaled by e^{g_last - g}.
    f32x4 vn[CT][4];
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
    bf16x8 vh[CT][2];
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const f32x4 fa = *reinterpret_cast<const f32x4*>(gp + rec::kEgl + 32 * s2 + 4 * grp);
      const f32x4 fb = *reinterpret_cast<const f32x4*>(gp + rec::kEgl + 32 * s2 + 16 + 4 * grp);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) vh[ct][s2] = pair_bf16(vn[ct][2 * s2] * fa, vn[ct][2 * s2 + 1] * fb);
    }
    __builtin_amdgcn_sched_barrier(0);
    // S = e^{g_last} S + k^T v_new.
    const float decay = gp[rec::kEg + kBT - 1];
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

  // P in 16 x 16 blocks (row block, column block) of A-operand lanes, as the
  // record's A blocks: lane (grp, li) holds P[16 kb + li][16 nb + 4 grp .. + 3]
  // as 4 bf16 hi then 4 lo; after acc_to_row_quads lane (g, 4 a + b) holds row
  // 4 g + a, columns 4 b .. + 3.  Q in blocks (column block, row block) of fp32
  // accumulator lanes.
  if (is_p) {
    const int slot = 16 * (li & 3) + 4 * grp + (li >> 2);
    char* const pb = pbuf + rec::p_off(seg, bh, BH, K) + (n0 / 16) * 1024 + 16 * slot;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        *reinterpret_cast<u32x4*>(pb + (kb * KB + ct) * 1024) = hi_lo4(acc_to_row_quads(S[ct][kb]));
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
// others through LDS as bf16 hi + lo.  With P as hi + lo from the transition
// kernel, three products (hi hi, hi lo, lo hi): ~2^-16 relative, as the fp32
// forms of the chunk kernels.  A serial chain of small steps: P and Q of the
// next two steps are in flight during one, and the three products run in
// accumulators of their own.
template <int K, int V>
__global__ void __launch_bounds__(4 * K)
chunk_combine_kernel(const char* __restrict__ pbuf, char* __restrict__ sbuf, int64_t BH, int64_t nseg) {
  constexpr int KB = K / 16, NVB = V / 16;
  constexpr int kAhead = 2;
  __shared__ __attribute__((aligned(16))) u32x4 xs[2][KB][64];  // hi, lo of one row tile's 4 rows per lane
  const hl::BhTile bt = hl::xcd_tile(blockIdx.x, BH, NVB);  // one XCD reads one (b, head)'s P
  const int wi = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;

  auto q_at = [&](int64_t s) {
    return reinterpret_cast<f32x4*>(sbuf + rec::s_off(s, bt.bh, BH, K, V) + (bt.vt * KB + wi) * 1024 + 16 * lane);
  };
  f32x4 qn[kAhead];
  u32x4 pn[kAhead][KB];
  auto load = [&](int64_t s, int i) {
    qn[i] = *q_at(s);
    const char* pb = pbuf + rec::p_off(s, bt.bh, BH, K) + wi * KB * 1024 + 16 * lane;
#pragma unroll
    for (int nb = 0; nb < KB; ++nb) pn[i][nb] = ldg16(pb + nb * 1024);
  };
  const int64_t last = nseg - 2;
  f32x4 S = *q_at(0);
#pragma unroll
  for (int i = 0; i < kAhead; ++i) load(1 + i < last ? 1 + i : last, i);
  auto step = [&](int64_t s, int i) {
    const int f = (int)(s & 1);
    xs[f][wi][lane] = hi_lo4(S);
    u32x4 p[KB];
#pragma unroll
    for (int nb = 0; nb < KB; ++nb) p[nb] = pn[i][nb];
    f32x4 hh = qn[i], hl = zero4(), lh = zero4();
    load(s + kAhead < last ? s + kAhead : last, i);
    lds_barrier();  // S_s is in LDS (the other buffer's readers finished before this barrier)
#pragma unroll
    for (int s2 = 0; s2 < KB / 2; ++s2) {
      const u32x4 a = p[2 * s2], b = p[2 * s2 + 1], x = xs[f][2 * s2][lane], y = xs[f][2 * s2 + 1][lane];
      const bf16x8 ph = __builtin_bit_cast(bf16x8, u32x4{a[0], a[1], b[0], b[1]});
      const bf16x8 pl = __builtin_bit_cast(bf16x8, u32x4{a[2], a[3], b[2], b[3]});
      const bf16x8 sh = __builtin_bit_cast(bf16x8, u32x4{x[0], x[1], y[0], y[1]});
      const bf16x8 sl = __builtin_bit_cast(bf16x8, u32x4{x[2], x[3], y[2], y[3]});
      hh = mfma16x16x32(ph, sh, hh);
      hl = mfma16x16x32(ph, sl, hl);
      lh = mfma16x16x32(pl, sh, lh);
    }
    S = hh + (hl + lh);
    *q_at(s) = S;
  };
  for (int64_t s = 1; s <= last; s += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (s + i <= last) step(s + i, i);  // uniform over the workgroup
  }
}

// ---------------------------------------------------------------------------
// Output kernel.  One 512-thread workgroup per (b, head, segment, V-tile of 64
// columns), 8 wavefronts in two roles that share SIMDs pairwise, as the fused
// kernel of chunk_fwd_fused.hip:
//   * state waves (0-3), 16 columns each, hold S in fp32 registers.  Phase 1:
//     hand S to the output waves as bf16 B-operand pairs, k S, t = beta (v -
//     e^g k S), v_new = A t, handed over the same way.  Phase 2: S = e^{g_last}
//     S + k^T (v_new e^{g_last - g}).  They issue all DMA: the next chunk's k,
//     q and gates between phase 1's row blocks, the A blocks and v of the
//     chunk after next behind the mid-chunk barrier (only phase 1 reads them);
//   * output waves (4-7).  Phase 1: the scores P[i][j] = (q_i . k_j)
//     e^{g_i - g_j}, j <= i, once per workgroup, as bf16 rows in LDS.  Phase
//     2: o = scale (e^{g_i} q S + P v_new) per 16-row block.
// The records bring A as MFMA operands and every gate factor, so the state
// waves convert nothing between chunks; the arithmetic is that kernel's.
template <int K, int V>
__global__ void __launch_bounds__(rec::kOThreads)
chunk_output_kernel(const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
                    const char* __restrict__ records, const float* __restrict__ h0,
                    const char* __restrict__ sbuf, bf16* __restrict__ o, float* __restrict__ ht, float scale,
                    int64_t T, int64_t H, int64_t NT, int64_t BH, int64_t nseg, int64_t len, int64_t t_per_seg) {
  using C = rec::OCfg<K>;
  constexpr int NVT = V / kTileV, KB2 = C::KB / 2;
  __shared__ __attribute__((aligned(1024))) char lds[C::kLds];

  const hl::BhTile bt = hl::xcd_tile(blockIdx.x, BH * nseg, NVT);
  const int64_t seg = bt.bh / BH, bh = bt.bh - seg * BH;
  const int64_t b = bh / H, hh = bh - b * H;
  const int v0 = (int)bt.vt * kTileV;
  const Span sp = span_of(seg, len, NT);

  const int tid = threadIdx.x;
  const int wi = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool state_wave = wi < 4;
  const int wq = wi & 3;
  const int lane = tid & 63, grp = lane >> 4, li = lane & 15;

  auto stage_k = [&](int s) { return lds + s * C::kStage; };
  auto stage_q = [&](int s) { return lds + s * C::kStage + C::kTileK; };
  auto stage_v = [&](int s) { return lds + s * C::kStage + 2 * C::kTileK; };
  auto stage_r = [&](int s) { return lds + s * C::kStage + 2 * C::kTileK + C::kTileVB; };
  char* const lp = lds + 2 * C::kStage;  // scores, 128-byte rows, swizzled
  // Hand-over slots, lane-major: 16 bytes per lane per B-operand pair.
  bf16x8* const ls = reinterpret_cast<bf16x8*>(lp + C::kPBytes) + wq * KB2 * 64 + lane;
  bf16x8* const lv = reinterpret_cast<bf16x8*>(lp + C::kPBytes + C::kSBytes) + wq * 2 * 64 + lane;

  // Global geometry in bytes, from the segment's first chunk.
  const int64_t tok0 = b * T + sp.c0 * kBT;
  const int64_t tsk = H * K * 2, tsv = H * V * 2;
  const int64_t kc0 = (tok0 * H + hh) * K * 2, vc0 = (tok0 * H + hh) * V * 2 + v0 * 2;
  const char* const r0 = records + rec::offset(bh, sp.c0, NT);
  bf16* const o0 = o + (tok0 * H + hh) * V;

  uint32_t koff[C::kKDma], voff[C::kVDma];
#pragma unroll
  for (int i = 0; i < C::kKDma; ++i) koff[i] = hl::dma_src_off((wq * C::kKDma + i) * 64 + lane, C::kRowK, tsk);
#pragma unroll
  for (int i = 0; i < C::kVDma; ++i) voff[i] = hl::dma_src_off((wq * C::kVDma + i) * 64 + lane, C::kRowV, tsv);

  auto issue_tile = [&](const bf16* src, int64_t c, char* dst) {
    const char* sb = reinterpret_cast<const char*>(src) + kc0 + c * kBT * tsk;
    const uint32_t l0 = lds_address(dst) + wq * C::kKDma * 1024;
#pragma unroll
    for (int i = 0; i < C::kKDma; ++i) dma_b128(sb, koff[i], __builtin_amdgcn_readfirstlane(l0 + i * 1024));
  };
  // Part m of the DMA of chunk c's k, q and gates into stage s.
  auto issue_part = [&](int64_t c, int s, int m) {
    if (m == 0) issue_tile(k, c, stage_k(s));
    else if (m == 1) issue_tile(q, c, stage_q(s));
    else if (m == 2 && wq == 0)
      dma_b128(r0 + c * rec::kBytes + rec::kGateOff, (uint32_t)(16 * lane),
               __builtin_amdgcn_readfirstlane(lds_address(stage_r(s) + rec::kGateOff)));
  };
  // DMA of chunk c's A blocks and v tile into stage s.
  auto issue_av = [&](int64_t c, int s) {
    const char* rb = r0 + c * rec::kBytes;
#pragma unroll
    for (int i = 0; i < C::kADma; ++i) {
      int x = wq + 4 * i;
      x = x < rec::kBlocks ? x : rec::kBlocks - 1;
      dma_b128(rb, (uint32_t)(x * rec::kBlockBytes + 16 * lane),
               __builtin_amdgcn_readfirstlane(lds_address(stage_r(s)) + x * rec::kBlockBytes));
    }
    const char* vb = reinterpret_cast<const char*>(v) + vc0 + c * kBT * tsv;
    const uint32_t lu = lds_address(stage_v(s)) + wq * C::kVDma * 1024;
#pragma unroll
    for (int i = 0; i < C::kVDma; ++i) dma_b128(vb, voff[i], __builtin_amdgcn_readfirstlane(lu + i * 1024));
  };

  auto rows_times_S = [&](const char* tile, int ib, const bf16x8* sbv) {
    f32x4 acc = zero4();
#pragma unroll
    for (int s2 = 0; s2 < KB2; ++s2) acc = mfma16x16x32(row_frag(tile, ib, s2, lane, C::kRowK), sbv[s2], acc);
    return acc;
  };
  // Row-tile stores after the quad transpose (8 bytes per lane).
  const uint32_t rowoff0 = hl::quadT_off(0, v0 + 16 * wq, lane, tsv, 2);
  auto store_rows = [&](bf16* base, int ib, f32x4 val) {
    const f32x4 t = quad_transpose(val);
    bf16x4 ov;
    ov[0] = (bf16)t[0]; ov[1] = (bf16)t[1]; ov[2] = (bf16)t[2]; ov[3] = (bf16)t[3];
    st_b64(base, rowoff0 + (uint32_t)(16 * ib * tsv), __builtin_bit_cast(u32x2, ov));
  };

  if (state_wave && sp.n > 0) {  // the first chunks' tiles, in flight with the state
    issue_av(0, 0);
#pragma unroll
    for (int m = 0; m < 3; ++m) issue_part(0, 0, m);
    issue_av(sp.n > 1 ? 1 : 0, 1);
  }
  // State S[kappa = 16 kb + 4 grp + r][n = v0 + 16 wq + li] in S[kb][r] (state waves).
  f32x4 S[C::KB];
  const int ncol = v0 + 16 * wq + li;
  const int64_t st_base = bh * (int64_t)(K * V);
#pragma unroll
  for (int kb = 0; kb < C::KB; ++kb) S[kb] = zero4();
  if (state_wave) {
    if (seg > 0) {
      const char* sp0 = sbuf + rec::s_off(seg * t_per_seg - 1, bh, BH, K, V) + (v0 / 16 + wq) * C::KB * 1024 + 16 * lane;
#pragma unroll
      for (int kb = 0; kb < C::KB; ++kb) S[kb] = *reinterpret_cast<const f32x4*>(sp0 + kb * 1024);
    } else if (h0) {
#pragma unroll
      for (int kb = 0; kb < C::KB; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[kb][r] = h0[st_base + (int64_t)(16 * kb + 4 * grp + r) * V + ncol];
    }
  }
  wait_vmcnt<0>();  // the state and the first tiles; the loop counts from here

  for (int64_t c = 0; c < sp.n; ++c) {
    const int s = (int)(c & 1);
    lds_barrier();  // A: chunk c is in LDS; every wave is done with chunk c - 1
    const char* tk = stage_k(s);
    const char* tq = stage_q(s);
    const float* gp = reinterpret_cast<const float*>(stage_r(s) + rec::kGateOff);

    f32x4 vn[4];  // state waves: v_new rows j = 16 jb + 4 grp + r of column 16 wq + li
    if (state_wave) {
      const int64_t cn = c + 1 < sp.n ? c + 1 : sp.n - 1;
      // S as the B operand, also handed to the output waves.
      bf16x8 sb[KB2];
#pragma unroll
      for (int s2 = 0; s2 < KB2; ++s2) {
        sb[s2] = pair_bf16(S[2 * s2], S[2 * s2 + 1]);
        ls[s2 * 64] = sb[s2];
      }
      const char* tr = stage_r(s);
      const char* tv = stage_v(s);
      f32x4 t4[4];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        issue_part(cn, s ^ 1, jb);  // between the row blocks, so the address unit drains while the MFMAs run
        const bf16x4 t = ds_read_tr16(reinterpret_cast<const bf16*>(tv + hl::tr_frag_off(16 * jb, 16 * wq, lane, C::kRowV)));
        const f32x4 ks = rows_times_S(tk, jb, sb);
        const f32x4 bt = *reinterpret_cast<const f32x4*>(gp + rec::kBeta + 16 * jb + 4 * grp);
        const f32x4 eg = *reinterpret_cast<const f32x4*>(gp + rec::kEg + 16 * jb + 4 * grp);
#pragma unroll
        for (int r = 0; r < 4; ++r) t4[jb][r] = bt[r] * ((float)t[r] - eg[r] * ks[r]);
      }
      const bf16x8 tp[2] = {pair_bf16(t4[0], t4[1]), pair_bf16(t4[2], t4[3])};
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        vn[ib] = zero4();
#pragma unroll
        for (int s2 = 0; s2 <= ib / 2; ++s2) {
          bf16x8 ah, al;
          a_frags(tr, ib, s2, lane, ah, al);
          vn[ib] = mfma16x16x32(ah, tp[s2], vn[ib]);
          vn[ib] = mfma16x16x32(al, tp[s2], vn[ib]);
        }
      }
      // v_new as the B operand of the local term, to the output waves.
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) lv[s2 * 64] = pair_bf16(vn[2 * s2], vn[2 * s2 + 1]);
    } else {
      // Scores: the ten 16 x 16 lower blocks shared out 3 / 3 / 2 / 2 over the
      // output waves; block (ib, jb)'s accumulator holds P^T[j = 16 jb + 4 grp
      // + r][i = 16 ib + li], 4 consecutive j of row i, one 8-byte write.
      constexpr int KS = K / 32;
      auto frags = [&](const char* tile, int rb, bf16x8* f) {
#pragma unroll
        for (int s2 = 0; s2 < KS; ++s2)
          f[s2] = load8(reinterpret_cast<const bf16*>(tile + hl::row8_frag_off(16 * rb, 32 * s2, lane, C::kRowK)));
      };
      auto block = [&](int ib, int jb, const bf16x8* kf, const bf16x8* qf) {
        f32x4 pt = zero4();
#pragma unroll
        for (int s2 = 0; s2 < KS; ++s2) pt = mfma16x16x32(kf[s2], qf[s2], pt);
        const int i = 16 * ib + li;
        const float gi = gp[rec::kG + i];
        const f32x4 gj = *reinterpret_cast<const f32x4*>(gp + rec::kG + 16 * jb + 4 * grp);
        bf16x4 pv;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * jb + 4 * grp + r;
          pv[r] = (bf16)((jb < ib || j <= i) ? pt[r] * fast_exp(gi - gj[r]) : 0.f);
        }
        *reinterpret_cast<bf16x4*>(lp + hl::pair_frag_off(16 * ib, 16 * jb, lane, 128)) = pv;
      };
      bf16x8 fa[KS], fb[KS], fc[KS], fd[KS];
      if (wq == 0) {  // (3, 0), (3, 1), (3, 2)
        frags(tq, 3, fa); frags(tk, 0, fb); frags(tk, 1, fc); frags(tk, 2, fd);
        block(3, 0, fb, fa); block(3, 1, fc, fa); block(3, 2, fd, fa);
      } else if (wq == 1) {  // (2, 0), (2, 1), (2, 2)
        frags(tq, 2, fa); frags(tk, 0, fb); frags(tk, 1, fc); frags(tk, 2, fd);
        block(2, 0, fb, fa); block(2, 1, fc, fa); block(2, 2, fd, fa);
      } else if (wq == 2) {  // (3, 3), (1, 0)
        frags(tq, 3, fa); frags(tk, 3, fb); frags(tq, 1, fc); frags(tk, 0, fd);
        block(3, 3, fb, fa); block(1, 0, fd, fc);
      } else {  // (1, 1), (0, 0)
        frags(tq, 1, fa); frags(tk, 1, fb); frags(tq, 0, fc); frags(tk, 0, fd);
        block(1, 1, fb, fa); block(0, 0, fd, fc);
      }
    }
    lds_barrier();  // M: scores, S pairs and v_new pairs of chunk c are in LDS

    if (state_wave) {
      issue_av(c + 2 < sp.n ? c + 2 : sp.n - 1, s);
      bf16x8 vh[2];
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const f32x4 fa = *reinterpret_cast<const f32x4*>(gp + rec::kEgl + 32 * s2 + 4 * grp);
        const f32x4 fb = *reinterpret_cast<const f32x4*>(gp + rec::kEgl + 32 * s2 + 16 + 4 * grp);
        vh[s2] = pair_bf16(vn[2 * s2] * fa, vn[2 * s2 + 1] * fb);
      }
      const float decay = gp[rec::kEg + kBT - 1];
#pragma unroll
      for (int kb = 0; kb < C::KB; ++kb) {
        S[kb] *= decay;
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) S[kb] = mfma16x16x32(kT_frag(tk, kb, s2, lane, C::kRowK), vh[s2], S[kb]);
      }
      wait_vmcnt<C::kWait>();  // this wave's DMA of chunk c + 1 is in
    } else {
      bf16x8 sb[KB2];
#pragma unroll
      for (int s2 = 0; s2 < KB2; ++s2) sb[s2] = ls[s2 * 64];
      const bf16x8 vb16[2] = {lv[0], lv[64]};
      bf16* ob = o0 + c * kBT * H * V;
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        f32x4 acc = rows_times_S(tq, ib, sb);  // q S
        acc *= *reinterpret_cast<const f32x4*>(gp + rec::kEg + 16 * ib + 4 * grp);
        f32x4 loc = zero4();
#pragma unroll
        for (int s2 = 0; s2 <= ib / 2; ++s2) {
          const bf16x4 lo = *reinterpret_cast<const bf16x4*>(lp + hl::pair_frag_off(16 * ib, 32 * s2, lane, 128));
          bf16x4 hi = {};
          if (2 * s2 + 1 <= ib) hi = *reinterpret_cast<const bf16x4*>(lp + hl::pair_frag_off(16 * ib, 32 * s2 + 16, lane, 128));
          loc = mfma16x16x32(concat(lo, hi), vb16[s2], loc);
        }
        store_rows(ob, ib, (acc + loc) * scale);
      }
    }
  }
  wait_vmcnt<0>();  // no DMA may still target this workgroup's LDS when it exits

  if (state_wave && ht && seg == nseg - 1) {
#pragma unroll
    for (int kb = 0; kb < C::KB; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) ht[st_base + (int64_t)(16 * kb + 4 * grp + r) * V + ncol] = S[kb][r];
  }
}

// Segments of a call: `out` of the output kernel, each of `per` transition
// segments of `len` chunks (the last may be shorter, none is empty).
struct Plan {
  int64_t out, per, len;
  int64_t segs(int64_t NT) const { return (NT + len - 1) / len; }
};

// The plan of least estimated time, in us on MI355X (only the ratios matter):
// a launch of workgroups that each walk n chunks takes a start that grows with
// the share of the CUs in use, and n periods; one CU holds one workgroup of
// either kernel (LDS), so more workgroups than CUs run in rounds.  Measured at
// K = V = 128: period 2.0-2.1 (outputs), 2.3-2.4 (transitions), 0.9 per combine
// step; whole forwards, unsegmented -> best of ten plans -> this rule's choice:
// 16 heads: 16 chunks 42 -> 36 -> 36 us, 32 chunks 77 -> 48 -> 48, 128 chunks
// 276 -> 107 -> 107; 32 heads, 32 chunks 84 -> 66; 4 heads, 64 chunks 140 -> 55.
// Two segments never gain (the transitions of the first alone take as long as
// its outputs), and neither do 128 workgroups or more without segments (64
// heads, 32 chunks: 86 unsegmented, 96 at best), so a plan has to save 5 %.
inline Plan plan_segments(int64_t BH, int64_t NT, int64_t nvt) {
  const int64_t cu = std::max<int64_t>(device_cu_count(), 1);
  auto launch = [&](int64_t wgs, double start, double period, int64_t chunks) {
    const double share = std::min(1.0, (double)wgs / cu);
    return (double)((wgs + cu - 1) / cu) * (start + 5.0 * share + period * chunks);
  };
  Plan best = {1, 1, std::max<int64_t>(NT, 1)};
  double t_best = 0.95 * launch(BH * nvt, 3.0, 2.02, NT);
  for (int64_t out = 3; out <= 32 && out <= NT; ++out) {
    for (int64_t per = 1; per <= 4 && out * per <= NT; ++per) {
      const int64_t len = (NT + out * per - 1) / (out * per);
      const int64_t nt = (NT + len - 1) / len;  // transition segments
      const int64_t no = (nt + per - 1) / per;  // output segments
      if (no < 3) continue;
      const double t = launch(BH * (nt - 1), 4.0, 2.4, len) + 3.0 + 0.9 * (nt - 2) +
                       launch(BH * nvt * no, 3.0, 2.1, len * per);
      if (t < t_best) {
        t_best = t;
        best = {no, per, len};
      }
    }
  }
  return best;
}

struct Workspace {
  int64_t records, pbuf, sbuf, bytes;
};
inline Workspace workspace_of(int64_t B, int64_t T, int64_t H, int64_t K, int64_t V, const Plan& p) {
  const int64_t NT = T / kBT, BH = B * H, nt = p.out > 1 ? p.segs(NT) : 1;
  Workspace w;
  w.records = 0;
  w.pbuf = BH * NT * rec::kBytes;
  w.sbuf = w.pbuf + (nt > 1 ? (nt - 2) * BH * K * K * 4 : 0);
  w.bytes = w.sbuf + (nt > 1 ? (nt - 1) * BH * K * V * 4 : 0);
  return w;
}

template <int K, int V>
hipError_t launch_rec(const void* q, const void* k, const void* v, const void* beta, const void* gate,
                      int gate_mode, const void* h0, void* o, void* ht, char* ws, const Plan& p, float scale,
                      int64_t B, int64_t T, int64_t H, hipStream_t s) {
  const int64_t NT = T / kBT, BH = B * H;
  const Workspace w = workspace_of(B, T, H, K, V, p);
  if (NT > 0) {
    const hipError_t e = build_records(K, k, beta, gate, gate_mode, ws + w.records, B, T, H, s);
    if (e != hipSuccess) return e;
  }
  if (p.out > 1) {
    const int64_t nt = p.segs(NT);
    hipLaunchKernelGGL((chunk_transition_kernel<K, V>), dim3((unsigned)(BH * (nt - 1))), dim3(rec::TCfg<K, V>::kThreads),
                       0, s, (const bf16*)k, (const bf16*)v, ws + w.records, (const float*)h0, ws + w.pbuf, ws + w.sbuf,
                       T, H, NT, BH, p.len);
    hipLaunchKernelGGL((chunk_combine_kernel<K, V>), dim3((unsigned)(BH * (V / 16))), dim3(4 * K), 0, s, ws + w.pbuf,
                       ws + w.sbuf, BH, nt);
  }
  hipLaunchKernelGGL((chunk_output_kernel<K, V>), dim3((unsigned)(BH * (V / kTileV) * p.out)), dim3(rec::kOThreads), 0,
                     s, (const bf16*)q, (const bf16*)k, (const bf16*)v, ws + w.records, (const float*)h0, ws + w.sbuf,
                     (bf16*)o, (float*)ht, scale, T, H, NT, BH, p.out, p.len * p.per, p.per);
  return hipGetLastError();
}

}  // namespace
}  // namespace thm

extern "C" int64_t thm_chunk_gated_delta_rule_workspace(int64_t B, int64_t T, int64_t H, int64_t K, int64_t V) {
  using namespace thm;
  if (B < 0 || T < 0 || H <= 0 || T % kBT || (K != 64 && K != 128) || (V != 64 && V != 128)) return THM_ERR_BAD_SHAPE;
  if (B == 0 || T == 0) return 0;
  if (B > (INT64_C(1) << 31) / H || B * (T / kBT) > (INT64_C(1) << 31) / H) return THM_ERR_BAD_SHAPE;
  return workspace_of(B, T, H, K, V, plan_segments(B * H, T / kBT, V / kTileV)).bytes;
}

extern "C" int thm_chunk_gated_delta_rule_fwd(const void* q, const void* k, const void* v, const void* beta,
                                              const void* gate, const void* h0, void* o, void* ht,
                                              void* workspace, int64_t workspace_bytes, float scale, int64_t B,
                                              int64_t T, int64_t H, int64_t K, int64_t V, int32_t chunk_size,
                                              int32_t qkv_dtype, int32_t gate_dtype, int32_t gate_kind,
                                              void* stream) {
  using namespace thm;
  if (chunk_size != kBT) return THM_ERR_BAD_ARGUMENT;
  if (gate_kind != THM_GATE_IDENTITY && gate_kind != THM_GATE_LOGSIGMOID && gate_kind != THM_GATE_CUMULATIVE)
    return THM_ERR_BAD_ARGUMENT;
  if (B < 0 || T < 0 || H <= 0 || K <= 0 || V <= 0 || T % kBT) return THM_ERR_BAD_SHAPE;
  if (qkv_dtype != THM_DTYPE_BF16) return THM_ERR_BAD_DTYPE;  // bf16 only
  if (gate && gate_dtype != THM_DTYPE_F32 && (gate_dtype != THM_DTYPE_BF16 || gate_kind == THM_GATE_CUMULATIVE))
    return THM_ERR_BAD_DTYPE;
  if ((K != 64 && K != 128) || (V != 64 && V != 128)) return THM_ERR_UNSUPPORTED;
  if (B == 0) return THM_OK;
  if (T == 0 && !ht) return THM_OK;
  if (T > 0 && (!q || !k || !v || !beta || !o)) return THM_ERR_NULL_POINTER;
  const void* p16[] = {q, k, v, workspace};
  for (const void* p : p16)
    if ((uintptr_t)p % 16) return THM_ERR_MISALIGNED;
  const void* p4[] = {h0, ht, beta};
  for (const void* p : p4)
    if ((uintptr_t)p % 4) return THM_ERR_MISALIGNED;
  if (((uintptr_t)gate % (gate_dtype == THM_DTYPE_F32 ? 4 : 2)) || ((uintptr_t)o % 8)) return THM_ERR_MISALIGNED;
  if (B > (INT64_C(1) << 31) / H) return THM_ERR_BAD_SHAPE;
  if (T > 0 && B * (T / kBT) > (INT64_C(1) << 31) / H) return THM_ERR_BAD_SHAPE;
  const Plan plan = plan_segments(B * H, T / kBT, V / kTileV);
  // The largest grids: records (one tile per workgroup), transitions, outputs.
  if (!launch_fits(B * (T / kBT) * H, 256) || !launch_fits(B * H * (V / kTileV) * plan.out * plan.per, 512))
    return THM_ERR_BAD_SHAPE;
  // 32-bit lane offsets within one chunk's token block.
  if (kBT * H * (K > V ? K : V) * 2 > (INT64_C(1) << 31)) return THM_ERR_UNSUPPORTED;
  const int64_t need = workspace_of(B, T, H, K, V, plan).bytes;
  if (workspace_bytes < need) return THM_ERR_BAD_ARGUMENT;
  if (need > 0 && !workspace) return THM_ERR_NULL_POINTER;
  int mode = rec::kGateNone;
  if (gate)
    mode = gate_kind == THM_GATE_CUMULATIVE ? rec::kGateCumulative
                                            : rec::kGatePerToken | (gate_kind == THM_GATE_LOGSIGMOID ? rec::kGateLogsigmoid : 0) |
                                                  (gate_dtype == THM_DTYPE_BF16 ? rec::kGateBf16 : 0);
  hipStream_t s = (hipStream_t)stream;
  char* const ws = (char*)workspace;
  hipError_t e;
  if (K == 64 && V == 64) e = launch_rec<64, 64>(q, k, v, beta, gate, mode, h0, o, ht, ws, plan, scale, B, T, H, s);
  else if (K == 64 && V == 128) e = launch_rec<64, 128>(q, k, v, beta, gate, mode, h0, o, ht, ws, plan, scale, B, T, H, s);
  else if (K == 128 && V == 64) e = launch_rec<128, 64>(q, k, v, beta, gate, mode, h0, o, ht, ws, plan, scale, B, T, H, s);
  else e = launch_rec<128, 128>(q, k, v, beta, gate, mode, h0, o, ht, ws, plan, scale, B, T, H, s);
  return (int)e;
}
