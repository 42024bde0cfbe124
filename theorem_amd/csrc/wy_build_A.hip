// WY matrix of the Gated DeltaNet chunk forward for MI355X (gfx950):
//   per chunk c of 64 tokens:  M[i][j] = beta_i (k_i . k_j) e^{g_i - g_j}  (j < i),
//                              A_c = (I + sign M)^{-1}
// sign = -1 is the reference's (I - M)^{-1} (kernels/recompute_w_u/reference.py:48-91,
// `_build_A`, a torch matmul + solve_triangular); sign = +1 is the gated delta
// rule's (I + M)^{-1}.  A [B, T, H, 64] fp32 holds row r of A_c at token c*64 + r.
//
// One workgroup (4 wavefronts) per (b, chunk, head) tile, head fastest.  With
// L = sign M (strictly lower) and 16x16 blocks L_ij, X = (I + L)^{-1} is block
// lower triangular:
//   X_ii = (I + L_ii)^{-1}                        (forward substitution)
//   X_ij = -X_ii sum_{m=j}^{i-1} L_im X_mj        (i > j, a column j per wave)
//   1. k k^T on v_mfma_f32_16x16x32_bf16: lane (g, j) holds features
//      8g .. 8g+7 of token j of a 16-token block, so the A fragment of block ib
//      and the B fragment of block jb are the same kind of 16-byte row load
//      (fp32 k: bf16 hi + lo, three products).  The 10 lower blocks are spread
//      over the 4 waves; every wave loads the tile's k (the repeats hit L2).
//   2. L blocks (scaled by beta_i e^{g_i - g_j}, strict lower part) go to LDS.
//   3. One wave inverts the four diagonal blocks: lane (d, c) owns column c of
//      block d and runs the 16-row substitution.
//   4. The other three waves take a block column of X each, its two to nine
//      16x16 products on v_mfma_f32_16x16x4_f32 (exact fp32 multiplies): T = sum
//      L_im X_mj, then X_ij = -X_ii T, each product's accumulators being the
//      next one's B operand (wy_blocks.h invert_L).
//   5. All 256 threads write A_c: 16-byte stores, 4 full 256-byte rows per
//      wavefront instruction.
// With per-token log decays (thm_wy_build_A_gates) the tile's first wave also
// forms and writes their cumulative sums, which it needs anyway: no launch of
// their own (4.9 us at B = 2, T = 2048, H = 8).
// HBM traffic per tile: k, beta, g read once, A written once.
//
// The record form (REC, bf16 k, sign +1; thm_chunk_gated_delta_rule_fwd) takes
// the gate as the caller has it (per-token log decay or its chunk-local
// cumulative sum) and writes, instead of A rows, one contiguous record per
// tile (rec_cfg.h): the ten lower 16 x 16 blocks of A as bf16 hi + lo in the
// lane order of the recurrence kernels' MFMA operands, the gates, their
// factors and beta.  That is 11 KiB against the 16 KiB of A rows (whose upper
// blocks are zero), 1 KiB runs instead of 256-byte rows H x 256 bytes apart,
// no cumsum launch, and nothing left to convert in the recurrence's serial
// chain.
#include <type_traits>

#include "gate.h"
#include "h_layout.h"
#include "rec_cfg.h"
#include "wy_blocks.h"

namespace thm {
namespace {

using wy::blk;
using wy::kBlk;
using wy::kBP;
constexpr int kBT = wy::kBT;
constexpr int kABThreads = 256;

// A_c rows of the inverted blocks Xb: thread (r = q / 16, chunk j4 = q % 16)
// writes A[r][4 j4 .. + 3]; 16-byte stores, 4 full 256-byte rows per
// wavefront instruction.
__device__ __forceinline__ void store_A(const float* Xb, float* out, int64_t H) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int it = 0; it < kBT * 16 / kABThreads; ++it) {
    const int q = tid + it * kABThreads;
    const int r = q >> 4, j0 = (q & 15) * 4;
    const int ib = r >> 4, jb = j0 >> 4;
    f32x4 v = zero4();
    if (jb <= ib) {
      const float* X = Xb + blk(ib, jb) * kBlk + (r & 15) * kBP + (j0 & 15);
      v[0] = X[0]; v[1] = X[1]; v[2] = X[2]; v[3] = X[3];
    }
    *reinterpret_cast<f32x4*>(out + (int64_t)r * H * kBT + j0) = v;
  }
}

// The tile's record from the inverted blocks Xb and sb, sg (beta, g).
__device__ __forceinline__ void store_rec(const float* Xb, const float* sb, const float* sg, char* out, int wv) {
  const int lane = lane_id();
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int p = wv + 4 * i;
    if (p < rec::kBlocks) {  // wave-uniform
      *reinterpret_cast<u32x4*>(out + p * rec::kBlockBytes + 16 * lane) = hi_lo4(wy::block_row4(Xb + p * kBlk));
    }
  }
  if (wv == 3) {
    float* const gp = reinterpret_cast<float*>(out + rec::kGateOff);
    const float g = sg[lane];
    gp[rec::kG + lane] = g;
    gp[rec::kEg + lane] = fast_exp(g);
    gp[rec::kEgl + lane] = fast_exp(sg[kBT - 1] - g);
    gp[rec::kBeta + lane] = sb[lane];
  }
}

// Raw gate value of one token-head (row = its index in [B, T, H]); 0 without a gate.
__device__ __forceinline__ float load_gate(const void* p, int mode, int64_t row) {
  if (mode == rec::kGateNone) return 0.f;
  if (mode & rec::kGateBf16) return (float)reinterpret_cast<const bf16*>(p)[row];
  return reinterpret_cast<const float*>(p)[row];
}
// The chunk's cumulative gates from its raw values, one token per lane.
__device__ __forceinline__ float form_gate(float x, int mode) {
  if (mode & rec::kGateLogsigmoid) x = logsigmoid(x);
  return mode & rec::kGatePerToken ? wave_inclusive_sum(x) : x;
}

template <typename IT, int K, int SIGN, bool REC>
__global__ void __launch_bounds__(kABThreads)
wy_build_A_kernel(const IT* __restrict__ k, const float* __restrict__ beta,
                  const void* __restrict__ g, int gate_mode, void* __restrict__ out, float* __restrict__ g_out,
                  int64_t T, int64_t H, int64_t NT) {
  constexpr bool kSplit = std::is_same<IT, float>::value;
  constexpr int KS = K / 32;  // contraction steps
  __shared__ __attribute__((aligned(16))) float Lb[10 * kBlk];  // L = sign M, lower blocks (diagonal blocks: strict lower part)
  __shared__ __attribute__((aligned(16))) float Xb[10 * kBlk];  // X = A_c, lower blocks
  __shared__ float sb[kBT], sg[kBT];

  const TileCoord tc = tile_coord(blockIdx.x, H, NT, T);
  const int64_t h = tc.hh;
  const int64_t tok0 = tc.tok0;
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: branches on it stay scalar
  const int lane = tid & 63;
  const int grp = lane >> 4, li = lane & 15;

  // 1. k fragments: fh[tb][s] = k[tok0 + 16 tb + li][32 s + 8 grp .. + 7].
  bf16x8 fh[4][KS], fl[4][kSplit ? KS : 1];
  {
    float v[8];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      const IT* row = k + ((tok0 + 16 * tb + li) * H + h) * K + 8 * grp;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if constexpr (kSplit) {
          load8f(row + 32 * s, v);
          split_bf16x8(v, fh[tb][s], fl[tb][s]);
        } else {
          fh[tb][s] = load8(row + 32 * s);
        }
      }
    }
  }
  if (tid < kBT) {
    const int64_t row = (tok0 + tid) * H + h;
    sb[tid] = beta[row];
    const float gc = form_gate(load_gate(g, gate_mode, row), gate_mode);
    sg[tid] = gc;
    if (g_out) g_out[row] = gc;
  }
  lds_barrier();

  // 2. L blocks; 3.-4. X = (I + L)^{-1}.
  wy::form_L<SIGN, KS, kSplit>(fh, fl, sb, sg, Lb, wv);
  lds_barrier();
  wy::invert_L(Lb, Xb, wv);

  // 5. A_c rows, or the record.
  if constexpr (REC) store_rec(Xb, sb, sg, reinterpret_cast<char*>(out) + rec::offset(tc.b * H + h, tc.c, NT), wv);
  else store_A(Xb, reinterpret_cast<float*>(out) + (tok0 * H + h) * kBT, H);
}

// ---------------------------------------------------------------------------
// bf16 k on grids of at least two tiles per persistent workgroup:
// software-pipelined, as the fused WY kernel (wy_fwd.hip).  Workgroups walk
// the tiles t, t + G, ... and issue the next tile's k rows (16-byte row-major
// loads), beta and g into registers before computing the current tile, so the
// loads are in flight through form_L and the inversion; the k tile is staged
// in LDS and the MFMA fragments are read from there.  The arithmetic is the
// one-tile kernel's, so A is bit-identical.
// Workgroups per CU: 4.  The inversion's latency chain, not memory, sets this
// kernel's time, so the more tiles a CU inverts at once the better (times at
// config 4 with an earlier inversion, whose off-diagonal products went through
// LDS: without the inversion a quarter of the time; wy_blocks.h has today's):
//   * the k loads go through one 32-bit per-lane offset on a wave-uniform
//     base (h_layout.h o_blk_lane / o_blk_step; 64-bit addresses spilled at
//     3 workgroups): 2 -> 3 per CU, 140 -> 116 us;
//   * the X blocks share the k tile's LDS (31.9 KB per workgroup at K = 128
//     instead of 44.9) and form_L reads its k fragments per block
//     (wy::form_L_lds; 114 VGPRs at K = 128, no scratch): 3 -> 4 per CU,
//     105.7 -> 96.3 us.  5 per CU spilled (140 us).
// A is bit-identical throughout.
template <int K>
constexpr int ab_pipe_wgs_per_cu() { return 4; }

template <int K, int SIGN, bool REC>
__global__ void __launch_bounds__(kABThreads, ab_pipe_wgs_per_cu<K>())
wy_build_A_pipe_kernel(const bf16* __restrict__ k, const float* __restrict__ beta,
                       const void* __restrict__ g, int gate_mode, void* __restrict__ out, int64_t T, int64_t H,
                       int64_t NT, int64_t tiles) {
  constexpr int KS = K / 32;
  // bf16 elements per k row: a 32-byte pad (h_layout.h tr_pitch), under which
  // the 16-byte fragment reads of 16 rows are conflict-free on gfx950.
  constexpr int kPitch = hl::tr_pitch(2 * K) / 2;
  constexpr int kCPR = K / 8;                         // 16-byte chunks per k row
  constexpr int kLoads = kBT * kCPR / kABThreads;     // per thread
  static_assert(kBT * kCPR % kABThreads == 0, "staging split");
  // The k tile is read only up to the barrier after form_L and restaged
  // after the barrier that follows the store of A, so the inversion's X blocks
  // share its LDS.
  constexpr int kKBytes = kBT * kPitch * 2, kXBytes = 10 * kBlk * 4;
  __shared__ __attribute__((aligned(16))) char kxt[kKBytes > kXBytes ? kKBytes : kXBytes];
  bf16* const ks = reinterpret_cast<bf16*>(kxt);
  float* const Xb = reinterpret_cast<float*>(kxt);
  __shared__ __attribute__((aligned(16))) float Lb[10 * kBlk];
  __shared__ float sb[kBT], sg[kBT];

  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: branches on it stay scalar
  const int lane = tid & 63;
  const int grp = lane >> 4, li = lane & 15;

  // XCD-aware walk (h_layout.h xcd_tile_order, a bijection of the tiles;
  // with a grid that is a multiple of 8, 1024 on MI355X, sequence index t runs
  // on XCD t % 8): the 16 heads of a (b, chunk) share
  // one XCD's L2, so each 64-byte line of beta and g is fetched once, not once
  // per XCD.  Measured traffic 1.108 -> 1.00 of the algorithmic bytes, at
  // +1.4 % time (115.2 -> 116.8 us at config 4, A bit-identical).
  const int64_t BNT = tiles / H;
  auto coord = [&](int64_t tile) { return tile_coord(hl::xcd_tile_order((uint32_t)tile, H, BNT), H, NT, T); };
  u32x4 kr[kLoads];
  float br = 0.f, gr = 0.f;
  const uint32_t k_off = hl::o_blk_lane(tid, K, H * K);
  auto prefetch = [&](int64_t tile) {
    const TileCoord tc = coord(tile);
    const int64_t h = tc.hh, tok0 = tc.tok0;
    const char* const kb = reinterpret_cast<const char*>(k + (tok0 * H + h) * K);
#pragma unroll
    for (int it = 0; it < kLoads; ++it) kr[it] = ldg16_nt(kb + hl::o_blk_step(it, K, H * K) + k_off);
    if (tid < kBT) {
      const int64_t row = (tok0 + tid) * H + h;
      br = beta[row];
      gr = load_gate(g, gate_mode, row);
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int it = 0; it < kLoads; ++it) {
      const int q = tid + it * kABThreads;
      const int j = q / kCPR, col = (q - j * kCPR) * 8;
      *reinterpret_cast<u32x4*>(ks + j * kPitch + col) = kr[it];
    }
    if (tid < kBT) {
      sb[tid] = br;
      sg[tid] = form_gate(gr, gate_mode);
    }
  };

  // Wave w of every workgroup sits on SIMD w, and the roles of the inversion
  // differ in work: rotated over the workgroups of a CU (launch order i,
  // i + 256, ...), each SIMD gets one of each.
  const int role = (wv + (int)(blockIdx.x * ab_pipe_wgs_per_cu<K>() / gridDim.x)) & 3;

  int64_t t = blockIdx.x;
  if (t >= tiles) return;  // whole workgroup
  prefetch(t);
  stage();
  lds_barrier();
  for (;;) {
    const int64_t tn = t + gridDim.x;
    if (tn < tiles) prefetch(tn);  // in flight while tile t computes
    const TileCoord tc = coord(t);
    wy::form_L_lds<SIGN, KS>([&](int tb, int s) { return load8(ks + (16 * tb + li) * kPitch + 32 * s + 8 * grp); },
                             sb, sg, Lb, wv);
    lds_barrier();  // every wave's k fragment reads are done: X may overwrite ks
    wy::invert_L(Lb, Xb, role);  // ends with a barrier
    if constexpr (REC) store_rec(Xb, sb, sg, reinterpret_cast<char*>(out) + rec::offset(tc.b * H + tc.hh, tc.c, NT), wv);
    else store_A(Xb, reinterpret_cast<float*>(out) + (tc.tok0 * H + tc.hh) * kBT, H);

    if (tn >= tiles) break;
    lds_barrier();  // every wave is done with tile t's LDS
    stage();
    lds_barrier();
    t = tn;
  }
}

template <typename IT, int K, int SIGN, bool REC>
hipError_t launch_A(const void* k, const void* beta, const void* g, int gate_mode, void* out, int64_t B,
                    int64_t T, int64_t H, hipStream_t s, float* g_out = nullptr) {
  const int64_t NT = T / kBT;
  const int64_t tiles = B * NT * H;
  if constexpr (std::is_same<IT, bf16>::value) {
    const int64_t pgrid = (int64_t)device_cu_count() * ab_pipe_wgs_per_cu<K>();
    if (pgrid > 0 && tiles >= 2 * pgrid) {
      hipLaunchKernelGGL((wy_build_A_pipe_kernel<K, SIGN, REC>), dim3((unsigned)pgrid), dim3(kABThreads), 0, s,
                         (const bf16*)k, (const float*)beta, g, gate_mode, out, T, H, NT, tiles);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((wy_build_A_kernel<IT, K, SIGN, REC>), dim3((unsigned)tiles), dim3(kABThreads), 0, s,
                     (const IT*)k, (const float*)beta, g, gate_mode, out, g_out, T, H, NT);
  return hipGetLastError();
}

template <typename IT, int K>
hipError_t launch_A_sign(const void* k, const void* beta, const void* g, void* A, int64_t B, int64_t T, int64_t H,
                         int sign, hipStream_t s) {
  const int mode = g ? rec::kGateCumulative : rec::kGateNone;
  return sign < 0 ? launch_A<IT, K, -1, false>(k, beta, g, mode, A, B, T, H, s)
                  : launch_A<IT, K, 1, false>(k, beta, g, mode, A, B, T, H, s);
}

}  // namespace

__attribute__((visibility("hidden"))) hipError_t build_records(int64_t K, const void* k, const void* beta,
                                                               const void* gate, int gate_mode, void* records,
                                                               int64_t B, int64_t T, int64_t H, hipStream_t s) {
  return K == 64 ? launch_A<bf16, 64, 1, true>(k, beta, gate, gate_mode, records, B, T, H, s)
                 : launch_A<bf16, 128, 1, true>(k, beta, gate, gate_mode, records, B, T, H, s);
}

}  // namespace thm

extern "C" int thm_wy_build_A(const void* k, const void* beta, const void* g, void* A, int64_t B,
                              int64_t T, int64_t H, int64_t K, int32_t chunk_size,
                              int32_t k_dtype, int32_t sign, void* stream) {
  using namespace thm;
  if (chunk_size != kBT) return THM_ERR_BAD_ARGUMENT;
  if (sign != 1 && sign != -1) return THM_ERR_BAD_ARGUMENT;
  if (B < 0 || T < 0 || H <= 0 || K <= 0 || T % kBT) return THM_ERR_BAD_SHAPE;
  if (k_dtype != THM_DTYPE_F32 && k_dtype != THM_DTYPE_BF16) return THM_ERR_BAD_DTYPE;
  if (K != 64 && K != 128) return THM_ERR_UNSUPPORTED;
  if (B == 0 || T == 0) return THM_OK;  // empty: nothing is read or written
  if (!k || !beta || !A) return THM_ERR_NULL_POINTER;
  if (((uintptr_t)k % 16) || ((uintptr_t)A % 16)) return THM_ERR_MISALIGNED;
  if (((uintptr_t)beta % 4) || (g && ((uintptr_t)g % 4))) return THM_ERR_MISALIGNED;
  if (B * (T / kBT) > (INT64_C(1) << 31) / H) return THM_ERR_BAD_SHAPE;
  if (!launch_fits(B * (T / kBT) * H, kABThreads)) return THM_ERR_BAD_SHAPE;
  // 32-bit per-lane offsets of the pipelined kernel's k loads: 64 tokens x H heads.
  if (kBT * H * K * 2 >= (INT64_C(1) << 32)) return THM_ERR_BAD_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  hipError_t e;
  if (k_dtype == THM_DTYPE_F32)
    e = (K == 64) ? launch_A_sign<float, 64>(k, beta, g, A, B, T, H, sign, s)
                  : launch_A_sign<float, 128>(k, beta, g, A, B, T, H, sign, s);
  else
    e = (K == 64) ? launch_A_sign<bf16, 64>(k, beta, g, A, B, T, H, sign, s)
                  : launch_A_sign<bf16, 128>(k, beta, g, A, B, T, H, sign, s);
  return (int)e;
}

extern "C" int thm_wy_build_A_gates(const void* k, const void* beta, const void* a, void* A, void* g, int64_t B,
                                    int64_t T, int64_t H, int64_t K, int32_t chunk_size, int32_t k_dtype,
                                    int32_t a_dtype, int32_t gate_kind, int32_t sign, void* stream) {
  using namespace thm;
  if (chunk_size != kBT) return THM_ERR_BAD_ARGUMENT;
  if (sign != 1 && sign != -1) return THM_ERR_BAD_ARGUMENT;
  if (gate_kind != THM_GATE_IDENTITY && gate_kind != THM_GATE_LOGSIGMOID) return THM_ERR_BAD_ARGUMENT;
  if (B < 0 || T < 0 || H <= 0 || K <= 0 || T % kBT) return THM_ERR_BAD_SHAPE;
  if (k_dtype != THM_DTYPE_F32) return THM_ERR_BAD_DTYPE;  // fp32 k only: the one-tile kernel
  if (a_dtype != THM_DTYPE_F32 && a_dtype != THM_DTYPE_BF16) return THM_ERR_BAD_DTYPE;
  if (K != 64 && K != 128) return THM_ERR_UNSUPPORTED;
  if (B == 0 || T == 0) return THM_OK;
  if (!k || !beta || !a || !A || !g) return THM_ERR_NULL_POINTER;
  if (((uintptr_t)k % 16) || ((uintptr_t)A % 16)) return THM_ERR_MISALIGNED;
  if (((uintptr_t)beta % 4) || ((uintptr_t)g % 4) || ((uintptr_t)a % (a_dtype == THM_DTYPE_F32 ? 4 : 2)))
    return THM_ERR_MISALIGNED;
  if (B * (T / kBT) > (INT64_C(1) << 31) / H) return THM_ERR_BAD_SHAPE;
  if (!launch_fits(B * (T / kBT) * H, kABThreads)) return THM_ERR_BAD_SHAPE;
  if (kBT * H * K * 2 >= (INT64_C(1) << 32)) return THM_ERR_BAD_SHAPE;  // as thm_wy_build_A
  const int mode = rec::kGatePerToken | (gate_kind == THM_GATE_LOGSIGMOID ? rec::kGateLogsigmoid : 0) |
                   (a_dtype == THM_DTYPE_BF16 ? rec::kGateBf16 : 0);
  hipStream_t s = (hipStream_t)stream;
  float* const go = (float*)g;
  hipError_t e;
  if (K == 64)
    e = sign < 0 ? launch_A<float, 64, -1, false>(k, beta, a, mode, A, B, T, H, s, go)
                 : launch_A<float, 64, 1, false>(k, beta, a, mode, A, B, T, H, s, go);
  else
    e = sign < 0 ? launch_A<float, 128, -1, false>(k, beta, a, mode, A, B, T, H, s, go)
                 : launch_A<float, 128, 1, false>(k, beta, a, mode, A, B, T, H, s, go);
  return (int)e;
}
