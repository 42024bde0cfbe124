// Blocked inversion of the WY matrix of one 64-token chunk (gfx950), shared by
// the A-builder (wy_build_A.hip) and the fused WY forward (wy_fwd.hip).
//
// With L = sign M strictly lower triangular, M[i][j] = beta_i (k_i . k_j)
// e^{g_i - g_j}, the chunk's A = (I + L)^{-1} is block lower triangular in
// 16 x 16 blocks:
//   X_ii = (I + L_ii)^{-1}                        (forward substitution)
//   X_ij = -X_ii sum_{m=j}^{i-1} L_im X_mj        (i > j, a column j per wave)
// Lower blocks (i, j), j <= i < 4, are stored packed (blk(i, j)) in LDS with
// row pitch kBP floats.  The math follows the reference's `_build_A`
// (kernels/recompute_w_u/reference.py:48-91: a torch matmul for M and
// solve_triangular for the inverse).
#pragma once

#include "h_layout.h"
#include "mfma.h"

namespace thm {
namespace wy {

constexpr int kBT = 64;
constexpr int kBP = hl::kWyPitch;  // LDS pitch (floats) of a 16x16 block (h_layout.h)
constexpr int kBlk = hl::kWyBlk;   // floats per block
constexpr int kLdsFloats = 10 * kBlk + 10 * kBlk;  // L, X

// Packed index of lower block (i, j), j <= i < 4.
__host__ __device__ constexpr int blk(int i, int j) { return i * (i + 1) / 2 + j; }

__device__ __forceinline__ f32x4 mfma16x16x4f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// acc += P X for a 16x16 block P in LDS (pitch kBP) and X in accumulator form
// (lane (g, l): rows 4g + r of column l in x[r]): at k-step q lane (g, l) feeds
// P[l][4g + q] and X[4g + q][l] = x[q], so an accumulator is the next product's
// B operand as it stands and P is one 16-byte row read per lane.
__device__ __forceinline__ f32x4 block_row4(const float* P) {
  return *reinterpret_cast<const f32x4*>(P + hl::wy_row_off(lane_id()));
}
__device__ __forceinline__ f32x4 block_mm(f32x4 p, f32x4 x, f32x4 acc) {
#pragma unroll
  for (int q = 0; q < 4; ++q) acc = mfma16x16x4f32(p[q], x[q], acc);
  return acc;
}

__device__ __forceinline__ void block_put(float* D, f32x4 acc) {
  const int lane = lane_id();
#pragma unroll
  for (int r = 0; r < 4; ++r) D[hl::wy_put_off(lane, r)] = acc[r];
}

// L blocks of one chunk from k fragments fh[tb][s] = k[16 tb + li][32 s + 8 grp .. + 7]
// (fp32 k: bf16 hi fh + lo fl, three products): wave wv forms the lower blocks
// p = wv, wv + 4, wv + 8 of the packed order (compile-time block indices, so
// the fragments stay in registers); sb, sg hold beta and g of the chunk.
template <int SIGN, int KS, bool kSplit>
__device__ __forceinline__ void form_L(const bf16x8 (&fh)[4][KS], const bf16x8 (&fl)[4][kSplit ? KS : 1],
                                       const float* sb, const float* sg, float* Lb, int wv) {
  const int lane = lane_id(), grp = lane >> 4, li = lane & 15;
#pragma unroll
  for (int p = 0; p < 10; ++p) {
    if ((p & 3) != wv) continue;  // wave-uniform
    constexpr int kIb[10] = {0, 1, 1, 2, 2, 2, 3, 3, 3, 3};
    const int ib = kIb[p], jb = p - ib * (ib + 1) / 2;
    f32x4 acc = zero4();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      acc = mfma16x16x32(fh[ib][s], fh[jb][s], acc);
      if constexpr (kSplit) {
        acc = mfma16x16x32(fh[ib][s], fl[jb][s], acc);
        acc = mfma16x16x32(fl[ib][s], fh[jb][s], acc);
      }
    }
    const int j = 16 * jb + li;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * ib + 4 * grp + r;
      const float l = (float)SIGN * sb[i] * acc[r] * fast_exp(sg[i] - sg[j]);
      Lb[p * kBlk + hl::wy_put_off(lane, r)] = (jb < ib || j < i) ? l : 0.f;
    }
  }
}

// form_L for bf16 k with the fragments read from LDS per block (frag(tb, s)
// returns k[16 tb + li][32 s + 8 grp .. + 7]) instead of held in registers
// for the whole chunk: the same products in the same order, ~40 fewer VGPRs
// at K = 128 (the A-builder's pipelined kernel, 4 workgroups per CU).
template <int SIGN, int KS, typename Frag>
__device__ __forceinline__ void form_L_lds(Frag frag, const float* sb, const float* sg, float* Lb, int wv) {
  const int lane = lane_id(), grp = lane >> 4, li = lane & 15;
#pragma unroll
  for (int p = 0; p < 10; ++p) {
    if ((p & 3) != wv) continue;  // wave-uniform
    constexpr int kIb[10] = {0, 1, 1, 2, 2, 2, 3, 3, 3, 3};
    const int ib = kIb[p], jb = p - ib * (ib + 1) / 2;
    bf16x8 fi[KS], fj[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      fi[s] = frag(ib, s);
      fj[s] = frag(jb, s);
    }
    f32x4 acc = zero4();
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = mfma16x16x32(fi[s], fj[s], acc);
    const int j = 16 * jb + li;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * ib + 4 * grp + r;
      const float l = (float)SIGN * sb[i] * acc[r] * fast_exp(sg[i] - sg[j]);
      Lb[p * kBlk + hl::wy_put_off(lane, r)] = (jb < ib || j < i) ? l : 0.f;
    }
  }
}

// Column J of X below the diagonal, X_{J+1,J} .. X_{3,J}, by one wave:
// T = sum_m L_im X_mJ, X_iJ = -X_ii T.  T and the X_mJ stay in accumulators,
// which are the next products' B operands; only L_im and X_ii come from LDS
// (row reads with no dependence on the chain, so they run ahead of it).
template <int J>
__device__ __forceinline__ void invert_column(const float* Lb, float* Xb) {
  if constexpr (J < 3) {
    f32x4 x[4];
    const float* D = Xb + blk(J, J) * kBlk;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[J][r] = D[hl::wy_put_off(lane_id(), r)];
    f32x4 l[4][3], xi[4];
#pragma unroll
    for (int i = J + 1; i < 4; ++i) {
      xi[i] = block_row4(Xb + blk(i, i) * kBlk);
#pragma unroll
      for (int m = J; m < i; ++m) l[i][m] = block_row4(Lb + blk(i, m) * kBlk);
    }
#pragma unroll
    for (int i = J + 1; i < 4; ++i) {
      f32x4 t = zero4();
#pragma unroll
      for (int m = J; m < i; ++m) t = block_mm(l[i][m], x[m], t);
      x[i] = -block_mm(xi[i], t, zero4());
      block_put(Xb + blk(i, J) * kBlk, x[i]);
    }
  }
}

// X = (I + L)^{-1} from the L blocks (all four waves, `role` a permutation of
// them; ends with a barrier):
//   diagonal blocks: role 3, lane (d, c) owns column c of X_dd (16-row
//   forward substitution of all four blocks at once), then one barrier;
//   off-diagonal blocks: role j < 3 forms column j of X (invert_column, 9, 5
//   and 2 products), exact fp32 multiplies; one barrier at the end.
// The products' latency chain costs, not their count.  With T and X_mj passed
// through LDS between products -> handed over in accumulators -> the four
// substitutions in one wave (a quarter of their issue slots; HIP events):
// fused WY at config 4 254 -> 246 -> 230 us, at K = V = 64 190 -> 179 -> 168;
// A-builder at config 4 (its roles also rotated over the SIMDs) 112 -> 112 ->
// 101, at 2048 tiles of K = 128 20.6 -> 20.0 -> 19.0, at 48 tiles 9.4 -> 9.0
// -> 8.1.  Error against float64 unchanged.
__device__ __forceinline__ void invert_L(const float* Lb, float* Xb, int role) {
  if (role == 3) {
    const int lane = lane_id(), d = lane >> 4, col = lane & 15;
    const float* L = Lb + blk(d, d) * kBlk;
    float* X = Xb + blk(d, d) * kBlk;
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float a0 = (r == col) ? 1.f : 0.f, a1 = 0.f;
#pragma unroll
      for (int s = 0; s < r; ++s) {
        if (s & 1) a1 = fmaf(-L[r * kBP + s], x[s], a1);
        else a0 = fmaf(-L[r * kBP + s], x[s], a0);
      }
      x[r] = a0 + a1;
      X[r * kBP + col] = x[r];
    }
  }
  lds_barrier();
  if (role == 0) invert_column<0>(Lb, Xb);
  else if (role == 1) invert_column<1>(Lb, Xb);
  else if (role == 2) invert_column<2>(Lb, Xb);
  lds_barrier();
}

}  // namespace wy
}  // namespace thm
