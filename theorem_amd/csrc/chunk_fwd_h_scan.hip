// Gated DeltaNet inter-chunk state recurrence, reference form, on grids that
// leave the GPU idle (gfx950; called from chunk_fwd_h.hip), fp32 or bf16 k, v:
//   S <- e^{g_last} S + k_c^T (v_c e^{g_last - g_c});  h[c] = S
// (kernels/chunk_fwd_h/reference.py:50-97; replaces kernel.py:61-138 there.)
//
// Without w the chunks are independent up to the decay: the products k_c^T v_c
// of many chunks are formed side by side and only an elementwise scan stays
// serial, where a kernel that walks the chunks pays its load - LDS - MFMA
// chain in each (0.8 us a chunk).  What bounds it is the memory latency of a
// batch on small calls and the store of h on large ones.
//
// One 1024-thread workgroup per (b, head, TB x TB tile of the state), 16
// chunks a batch:
//   * wave w forms the tile's product of chunk c0 + w: lane (grp, li) loads
//     columns TB / 16 li .. of k and of v for the 16 tokens 16 grp + e
//     straight into MFMA operand registers (nothing is staged; any token order
//     serves as long as both operands share it), so with TB = 32 the tile is
//     2 x 2 products whose rows and columns interleave.  bf16: v e^{g_last - g}
//     rounded to bf16, v_mfma_f32_16x16x32_bf16; fp32:
//     v_mfma_f32_16x16x4_f32, exact fp32 products;
//   * the next batch's loads are issued, the products go to LDS (two buffers,
//     one barrier a batch), and every thread scans its element of the tile
//     over the batch's chunks and stores h.
#include <type_traits>

#include "h_layout.h"
#include "mfma.h"

namespace thm {
namespace {

constexpr int kBT = 64;
constexpr int kBatch = 16;  // chunks a batch, one per wave
constexpr int kScanThreads = 64 * kBatch;

template <typename IT, int N>
struct Cols {
  typedef IT type __attribute__((ext_vector_type(N)));
};
template <typename IT>
struct Cols<IT, 1> {
  typedef IT type;
};

template <typename IT, int TB>
__global__ void __launch_bounds__(kScanThreads)
chunk_fwd_h_scan_kernel(const IT* __restrict__ k, const IT* __restrict__ v, const float* __restrict__ g,
                        const float* __restrict__ h0, float* __restrict__ h, float* __restrict__ ht, int64_t T,
                        int64_t H, int64_t NT, int64_t BH, int64_t heads, int K, int V) {
  constexpr int CPL = TB / 16;  // columns per lane
  constexpr int E = TB * TB;
  constexpr bool kF32 = std::is_same<IT, float>::value;
  using L = typename Cols<IT, CPL>::type;
  __shared__ __attribute__((aligned(16))) float prod[2][kBatch][E];
  __shared__ float decay[2][kBatch];
  __shared__ __attribute__((aligned(16))) float fac[kBatch][kBT];

  // The tiles of one (b, head) share an XCD, whose L2 then serves the columns
  // of k and v that several tiles read.  `heads`: BH rounded up to whole rounds
  // of the XCDs (64 x 64, bf16, 48 chunks of 45 heads, us: walking 25.6, tiles
  // of a head spread over the XCDs 28.1; 64 chunks 33.2, 36.7, together 20.8).
  const int nv = V / TB;
  const hl::BhTile bt = hl::xcd_tile(blockIdx.x, heads, (K / TB) * nv);
  if (bt.bh >= BH) return;  // (uniform over the workgroup)
  const int64_t b = bt.bh / H, hh = bt.bh - b * H;
  const int kt = (int)bt.vt / nv, vt = (int)bt.vt - kt * nv;
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, grp = lane >> 4, li = lane & 15;

  const int64_t tsk = H * K * (int64_t)sizeof(IT), tsv = H * V * (int64_t)sizeof(IT);  // bytes between tokens
  const char* const k0 = reinterpret_cast<const char*>(k + (b * T * H + hh) * K + kt * TB);
  const char* const v0 = reinterpret_cast<const char*>(v + (b * T * H + hh) * V + vt * TB);
  const float* const g0 = g ? g + b * T * H + hh : nullptr;
  const uint32_t koff = (uint32_t)(16 * grp * tsk + CPL * li * (int)sizeof(IT));
  const uint32_t voff = (uint32_t)(16 * grp * tsv + CPL * li * (int)sizeof(IT));

  L kr[16], vr[16];
  float gr = 0.f;
  auto load = [&](int64_t c) {
    const char* kb = k0 + c * kBT * tsk;
    const char* vb = v0 + c * kBT * tsv;
#pragma unroll
    for (int e = 0; e < 16; ++e) kr[e] = *reinterpret_cast<const L*>(kb + e * tsk + koff);
#pragma unroll
    for (int e = 0; e < 16; ++e) vr[e] = *reinterpret_cast<const L*>(vb + e * tsv + voff);
    if (g) gr = g0[(c * kBT + lane) * H];
  };
  auto col = [](const L& x, int c) -> IT {
    if constexpr (CPL == 1) return x;
    else return x[c];
  };

  // This thread's element of the tile, in the order of the accumulators:
  // position ((4 c + r) 64 + lane) CPL + c' holds row CPL (4 grp + r) + c,
  // column CPL li + c'.
  const bool scans = tid < E;
  const int el = (tid / CPL) & 63, ecr = tid / (64 * CPL);
  const int erow = CPL * (4 * (el >> 4) + (ecr & 3)) + (ecr >> 2), ecol = CPL * (el & 15) + tid % CPL;
  const int64_t eoff = (int64_t)(kt * TB + erow) * V + vt * TB + ecol;
  float S = scans && h0 ? h0[bt.bh * K * V + eoff] : 0.f;
  float* hp = h + (b * NT * H + hh) * K * V + eoff;
  const int64_t hstep = H * K * V;

  if (wv < NT) load(wv);
  for (int64_t c0 = 0; c0 < NT; c0 += kBatch) {
    const int f = (int)(c0 / kBatch) & 1;
    const int64_t c = c0 + wv;
    if (c < NT) {
      if (g) {
        const float gl = __shfl(gr, 63);
        fac[wv][lane] = fast_exp(gl - gr);
        if (lane == 0) decay[f][wv] = fast_exp(gl);
      } else {
        fac[wv][lane] = 1.f;
        if (lane == 0) decay[f][wv] = 1.f;
      }
      wave_lds_sync();
      float fv[16];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(&fac[wv][16 * grp + 4 * i]);
#pragma unroll
        for (int r = 0; r < 4; ++r) fv[4 * i + r] = x[r];
      }
      f32x4 acc[CPL][CPL];
#pragma unroll
      for (int a = 0; a < CPL; ++a)
#pragma unroll
        for (int d = 0; d < CPL; ++d) acc[a][d] = zero4();
      if constexpr (kF32) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
          for (int a = 0; a < CPL; ++a)
#pragma unroll
            for (int d = 0; d < CPL; ++d)
              acc[a][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(col(kr[e], a), col(vr[e], d) * fv[e], acc[a][d], 0, 0, 0);
      } else {
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          bf16x8 ka[CPL], vb[CPL];
#pragma unroll
          for (int a = 0; a < CPL; ++a)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              ka[a][e] = col(kr[8 * s2 + e], a);
              vb[a][e] = (bf16)((float)col(vr[8 * s2 + e], a) * fv[8 * s2 + e]);
            }
#pragma unroll
          for (int a = 0; a < CPL; ++a)
#pragma unroll
            for (int d = 0; d < CPL; ++d) acc[a][d] = mfma16x16x32(ka[a], vb[d], acc[a][d]);
        }
      }
      if (c + kBatch < NT) load(c + kBatch);
#pragma unroll
      for (int a = 0; a < CPL; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float* p = &prod[f][wv][((4 * a + r) * 64 + lane) * CPL];
          if constexpr (CPL == 1) *p = acc[a][0][r];
          else *reinterpret_cast<f32x2*>(p) = f32x2{acc[a][0][r], acc[a][1][r]};
        }
    }
    // Also keeps buffer f until every thread has scanned it: it is written
    // again two batches on, after the next barrier.
    lds_barrier();
    if (scans) {
      const int64_t left = NT - c0;
      auto step = [&](int i) {
        S = decay[f][i] * S + prod[f][i][tid];
        *hp = S;
        hp += hstep;
      };
      if (left >= kBatch) {
#pragma unroll
        for (int i = 0; i < kBatch; ++i) step(i);
      } else {
        for (int i = 0; i < (int)left; ++i) step(i);
      }
    }
  }
  if (scans && ht) ht[bt.bh * K * V + eoff] = S;
}

template <typename IT, int TB>
hipError_t launch_scan(const void* k, const void* v, const void* g, const void* h0, void* h, void* ht, int64_t B,
                       int64_t T, int64_t H, int64_t K, int64_t V, hipStream_t s) {
  const int64_t BH = B * H, tiles = (K / TB) * (V / TB), whole = (BH + 7) / 8 * 8;
  const int64_t slots = device_cu_count() * (int64_t)(BH * tiles <= device_cu_count() ? 1 : 2);
  const int64_t heads = BH > 8 && whole * tiles <= slots ? whole : BH;  // (fewer heads would leave XCDs idle)
  hipLaunchKernelGGL((chunk_fwd_h_scan_kernel<IT, TB>), dim3((unsigned)(heads * tiles)), dim3(kScanThreads), 0, s,
                     (const IT*)k, (const IT*)v, (const float*)g, (const float*)h0, (float*)h, (float*)ht, T, H, T / kBT,
                     BH, heads, (int)K, (int)V);
  return hipGetLastError();
}

}  // namespace

// Tile side for a call, or 0: the kernels that walk the chunks.  A workgroup
// fills a CU (16 waves, and with 32 x 32 tiles 132 KB of LDS), so the tile is
// the smallest that leaves one per CU; MI355X, us, walking -> 16 -> 32 (bf16;
// fp32 in brackets):
//   6 heads of 64 x 64, 16 chunks       9.2 -> 4.6 -> 5.1    (14.6 -> 5.4 -> 8.6)
//   16 heads of 64 x 64, 128 chunks    58 -> 33 -> 40        (100 -> 35 -> 70)
//   8 heads of 128 x 128, 128 chunks   84 -> 54 -> 35        (181 -> 66 -> 70)
//   16 heads of 128 x 128, 128 chunks  83 -> 109 -> 42       (185 -> 128 -> 75)
// Two 32 x 32 workgroups per CU gain on long sequences at K = 128 (a walking
// workgroup takes all K rows of 64 columns, so its chunk costs more there),
// three nowhere; walking -> 32, 64 chunks:
//   128 x 128, 20 heads   44.6 -> 37.1    (100 -> 70)     32 heads  43.5 -> 41.7  (97 -> 74)
//   128 x 64, 45 heads    43.8 -> 37.8    (93 -> 71)      64 heads  44.3 -> 44.9  (127 -> 98)
//   64 x 128, 45 heads, tiles of a head apart, 43.6 -> 70.9; 64 heads 37.7 -> 43.9
// (where h takes most of the memory-side cache, 22 and 25 heads of 128 x 128 at
// 128 chunks, bf16, it loses: 85 -> 105 and 113 -> 136; 24 heads 149 -> 129).
// Four chunks or fewer are walked in the time of one batch (2 chunks of 62
// heads of 64 x 64: 3.4 -> 9.8 -> 4.1).
__attribute__((visibility("hidden"))) int h_scan_tile(int64_t BH, int64_t NT, int64_t K, int64_t V) {
  if (NT <= 4) return 0;
  const int64_t cu = device_cu_count(), n32 = BH * (K / 32) * (V / 32);
  if (4 * n32 <= cu) return 16;
  return n32 <= cu || (n32 <= 2 * cu && NT >= 32 && K == 128) ? 32 : 0;
}

__attribute__((visibility("hidden"))) hipError_t chunk_fwd_h_scan(bool f32, int tile, const void* k, const void* v,
                                                                  const void* g, const void* h0, void* h, void* ht,
                                                                  int64_t B, int64_t T, int64_t H, int64_t K,
                                                                  int64_t V, hipStream_t s) {
  if (f32)
    return tile == 16 ? launch_scan<float, 16>(k, v, g, h0, h, ht, B, T, H, K, V, s)
                      : launch_scan<float, 32>(k, v, g, h0, h, ht, B, T, H, K, V, s);
  return tile == 16 ? launch_scan<bf16, 16>(k, v, g, h0, h, ht, B, T, H, K, V, s)
                    : launch_scan<bf16, 32>(k, v, g, h0, h, ht, B, T, H, K, V, s);
}

}  // namespace thm
