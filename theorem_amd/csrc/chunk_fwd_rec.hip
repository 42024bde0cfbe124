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
//      each of several segments of the sequences (segments.h, the transition
//      and combine kernels; how many, seg_plan.h);
//   3. the output kernel, one workgroup per (b, head, segment, 64-column
//      V-tile).
//
// Segments (segments.h) cost less than twice the recurrence's own work,
// against a serial chain shorter by their number: B = 1, T = 8192, H = 16,
// K = V = 128 (32 workgroups of 128 chunks without them) 274 -> 116 us for the
// whole forward.
#include "h_layout.h"
#include "mfma.h"
#include "rec_cfg.h"
#include "segments.h"
#include "vmem.h"

namespace thm {

// wy_build_A.hip
hipError_t build_records(int64_t K, const void* k, const void* beta, const void* gate, int gate_mode,
                         void* records, int64_t B, int64_t T, int64_t H, hipStream_t s);

namespace {

using rec::kBT;
using rec::kTileV;
using namespace seg;

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
                    const char* __restrict__ sbuf, const uint32_t* __restrict__ redo, bf16* __restrict__ o,
                    float* __restrict__ ht, float scale, int64_t T, int64_t H, int64_t NT, int64_t BH, int64_t nseg, int64_t len, int64_t t_per_seg) {
  using C = rec::OCfg<K>;
  constexpr int NVT = V / kTileV, KB2 = C::KB / 2;
  __shared__ __attribute__((aligned(1024))) char lds[C::kLds];

  const hl::BhTile bt = hl::xcd_tile(blockIdx.x, BH * nseg, NVT);
  const int64_t seg = bt.bh / BH, bh = bt.bh - seg * BH;
  const int64_t b = bh / H, hh = bh - b * H;
  const int v0 = (int)bt.vt * kTileV;
  Span sp = span_of(seg, len, NT);
  const bool whole = nseg > 1 && redo_columns<V>(redo, bh, v0, kTileV);

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
      const int x = C::a_block(wq, i);
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
    issue_av(sp.c0 + 1 < NT ? 1 : 0, 1);  // (past a segment of one chunk, for `whole`)
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
  if (whole) {
    if (seg > 0) return;  // (uniform over the workgroup)
    sp.n = NT;
  }

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

  if (state_wave && ht && sp.c0 + sp.n == NT) {
#pragma unroll
    for (int kb = 0; kb < C::KB; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) ht[st_base + (int64_t)(16 * kb + 4 * grp + r) * V + ncol] = S[kb][r];
  }
}

inline Plan plan_of(int64_t B, int64_t T, int64_t H, int64_t K, int64_t V) {
  return plan_fwd(B * H, T / kBT, K, V, device_cu_count());
}

struct Workspace {
  int64_t records, pbuf, sbuf, redo, bytes;
};
inline Workspace workspace_of(int64_t B, int64_t T, int64_t H, int64_t K, int64_t V, const Plan& p) {
  const int64_t NT = T / kBT, BH = B * H;
  Workspace w;
  w.records = 0;
  w.pbuf = BH * NT * rec::kBytes;
  w.sbuf = w.pbuf + p_bytes(p, BH, NT, K);
  w.redo = w.sbuf + s_bytes(p, BH, NT, K, V);
  w.bytes = w.redo + redo_bytes(p, BH, V);
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
    hipLaunchKernelGGL((chunk_transition_kernel<K, V, false, true>), dim3((unsigned)(BH * (nt - 1))),
                       dim3(rec::TCfg<K, V, false>::kThreads), 0, s, (const bf16*)k, (const bf16*)nullptr, (const bf16*)v,
                       (const float*)nullptr, ws + w.records, (const float*)h0, ws + w.pbuf, ws + w.sbuf, T, H, NT, BH,
                       p.len);
    hipLaunchKernelGGL((chunk_combine_kernel<K, V>), dim3((unsigned)(BH * (V / 16))), dim3(4 * K), 0, s, ws + w.pbuf,
                       ws + w.sbuf, (uint32_t*)(ws + w.redo), BH, nt);
  }
  hipLaunchKernelGGL((chunk_output_kernel<K, V>), dim3((unsigned)(BH * (V / kTileV) * p.out)), dim3(rec::kOThreads), 0,
                     s, (const bf16*)q, (const bf16*)k, (const bf16*)v, ws + w.records, (const float*)h0, ws + w.sbuf,
                     (const uint32_t*)(ws + w.redo), (bf16*)o, (float*)ht, scale, T, H, NT, BH, p.out, p.len * p.per, p.per);
  return hipGetLastError();
}

}  // namespace
}  // namespace thm

extern "C" int64_t thm_chunk_gated_delta_rule_workspace(int64_t B, int64_t T, int64_t H, int64_t K, int64_t V) {
  using namespace thm;
  if (B < 0 || T < 0 || H <= 0 || T % kBT || (K != 64 && K != 128) || (V != 64 && V != 128)) return THM_ERR_BAD_SHAPE;
  if (B == 0 || T == 0) return 0;
  if (B > (INT64_C(1) << 31) / H || B * (T / kBT) > (INT64_C(1) << 31) / H) return THM_ERR_BAD_SHAPE;
  return workspace_of(B, T, H, K, V, plan_of(B, T, H, K, V)).bytes;
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
  const Plan plan = plan_of(B, T, H, K, V);
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
