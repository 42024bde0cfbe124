// Depthwise causal 1-D convolution, two extensions of causal_conv1d.hip for
// MI355X (gfx950), same arithmetic (acc = bias, then taps 0..W-1 in fp32 FMA,
// optional SiLU):
//
// 1. Channels-last layout: x, out [B, S, D] with D contiguous (the layout of a
//    [B, D, S] tensor that is a transposed view of [B, S, D]).  Vectors run
//    along D: a lane owns VEC channels (one 16-byte vector) and walks a segment
//    of timesteps, keeping the last W-1 input vectors of its channels in
//    registers; only the W-1 rows before each segment are read twice.  A
//    wavefront reads and writes 1 KiB of one row per step, and x and out are
//    streamed once.  Bound by memory at large sizes (5.6 TB/s) and by the
//    steps' arithmetic at smaller ones: [2, 5001, 4352] bf16 with SiLU 47.7 ->
//    37.4 us (whole lanes, whole segments, no IEEE division; 64-step segments
//    throughout and a step-by-step tail before).
//
// 2. Decode step (rolling state): for each (b, d), with state s[0..L_s) and
//    the new samples x[0..L):  window = s ++ x,
//      out[t] = act(bias + sum_k w[k] window[L_s - (W-1) + t + k]),  t < L,
//    and the state becomes the last L_s samples of the window (in place).
//    One lane per (b, d); a decode step moves a few bytes per channel, so this
//    is latency-, not bandwidth-, bound: one sample per sequence has a kernel
//    of its own (causal_conv1d_step_kernel).
#include <algorithm>

#include "common.h"

namespace thm {
namespace {

constexpr int kClThreads = 256;
constexpr int kClSeg = 64;  // timesteps per lane, at most

// Time steps whose loads are in flight ahead of use (16 KiB or less per wave;
// 16 steps of bf16 lanes take 193 VGPRs against 134, 38.5 against 37.4 us at
// [2, 5001, 4352], and 8 steps of fp32 lanes 94 against 84 at [4, 2500, 5120]).
template <typename XT>
constexpr int cl_depth() { return sizeof(XT) == 2 ? 8 : 16; }

__device__ __forceinline__ float conv_param(const void* p, int64_t i, int is_bf16) {
  return is_bf16 ? (float)reinterpret_cast<const bf16*>(p)[i] : reinterpret_cast<const float*>(p)[i];
}

template <typename XT, int VEC>
__device__ __forceinline__ void cl_load(const XT* p, float* v) {
  if constexpr (VEC * sizeof(XT) == 16) {
    unpack16(ldg16_nt(p), v, XT{});
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) v[i] = to_f32(p[i]);
  }
}

template <typename XT, int VEC>
__device__ __forceinline__ void cl_store(XT* p, const float* v) {
  if constexpr (VEC * sizeof(XT) == 16) {
    stg16_nt(p, pack16(v, XT{}));
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) p[i] = from_f32<XT>(v[i]);
  }
}

// One lane per (b, segment, channel group), channel group fastest, so a
// wavefront's lanes stay full whatever the channel count.  BLOCKS: segments of
// `seg` steps, a multiple of cl_depth, in blocks of cl_depth steps whose loads
// are in flight a block ahead of use.  The last segment of a sequence starts early enough to be
// whole and writes only the steps that are its own, so a ragged length costs
// no step-by-step tail (whose loads each wait for memory).  Otherwise: steps
// one by one (scalar lanes, and sequences shorter than a block).
template <typename XT, typename WT, int VEC, int W, bool SILU, bool BLOCKS>
__global__ void __launch_bounds__(kClThreads)
causal_conv1d_cl_kernel(const XT* __restrict__ x, const void* __restrict__ weight,
                        const void* __restrict__ bias, XT* __restrict__ out, int64_t seqlen,
                        int64_t dim, int seg, uint32_t groups, uint32_t segs, uint32_t items) {
  const uint32_t item = blockIdx.x * kClThreads + threadIdx.x;
  if (item >= items) return;  // no barriers follow
  const uint32_t bs = item / groups, cg = item - bs * groups;
  const uint32_t b = bs / segs;
  const int64_t d0 = (int64_t)cg * VEC;
  const int64_t own = (int64_t)(bs - b * segs) * seg;  // first step this lane writes
  const int64_t tend = (own + seg < seqlen) ? own + seg : seqlen;
  const int64_t t0 = BLOCKS ? tend - seg : own;

  const XT* __restrict__ xb = x + b * seqlen * dim + d0;
  XT* __restrict__ ob = out + b * seqlen * dim + d0;
  constexpr int kDepth = cl_depth<XT>();
  u32x4 pf[kDepth];
  if constexpr (BLOCKS) {
#pragma unroll
    for (int i = 0; i < kDepth; ++i) pf[i] = ldg16_nt(xb + (t0 + i) * dim);
  }
  // win[k] = input at t - (W-1) + k for k < W-1 (zero before t = 0): loaded
  // from a clamped row, then zeroed, so every load is issued before any use.
  float win[W > 1 ? W - 1 : 1][VEC];
#pragma unroll
  for (int k = 0; k < W - 1; ++k) {
    const int64_t t = t0 - (W - 1) + k;
    cl_load<XT, VEC>(xb + (t >= 0 ? t : 0) * dim, win[k]);
    if (t < 0) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) win[k][v] = 0.f;
    }
  }
  // Weights and bias (bias absent: read the weights, then zero).
  const WT* __restrict__ wp = reinterpret_cast<const WT*>(weight);
  const WT* __restrict__ bp = bias ? reinterpret_cast<const WT*>(bias) : wp;
  float wk[W][VEC], bv[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
#pragma unroll
    for (int k = 0; k < W; ++k) wk[k][v] = to_f32(wp[(d0 + v) * W + k]);
    bv[v] = to_f32(bp[d0 + v]);
  }
  if (!bias) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) bv[v] = 0.f;
  }

  const int skip = (int)(own - t0);  // steps of the previous segment's lane
  XT* op = ob + t0 * dim;
  auto step = [&](int j, const float* cur) {
    float res[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      float acc = bv[v];
#pragma unroll
      for (int k = 0; k < W - 1; ++k) acc = __builtin_fmaf(wk[k][v], win[k][v], acc);
      acc = __builtin_fmaf(wk[W - 1][v], cur[v], acc);
      res[v] = acc;
    }
    if constexpr (SILU) silu<XT, VEC>(res);
    if (!BLOCKS || j >= skip) cl_store<XT, VEC>(op, res);
    op += dim;
#pragma unroll
    for (int k = 0; k + 1 < W - 1; ++k)
#pragma unroll
      for (int v = 0; v < VEC; ++v) win[k][v] = win[k + 1][v];
    if constexpr (W > 1) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) win[W - 2][v] = cur[v];
    }
  };

  if constexpr (BLOCKS) {
    const XT* xp = xb + (t0 + kDepth) * dim;
    int j = 0;
    for (; j + kDepth < seg; j += kDepth) {
#pragma unroll
      for (int i = 0; i < kDepth; ++i) {
        float cur[VEC];
        unpack16(pf[i], cur, XT{});
        pf[i] = ldg16_nt(xp);
        xp += dim;
        step(j + i, cur);
      }
    }
#pragma unroll
    for (int i = 0; i < kDepth; ++i) {
      float cur[VEC];
      unpack16(pf[i], cur, XT{});
      step(j + i, cur);
    }
  } else {
    const int n = (int)(tend - t0);
    for (int j = 0; j < n; ++j) {
      float cur[VEC];
      cl_load<XT, VEC>(xb + (t0 + j) * dim, cur);
      step(j, cur);
    }
  }
}

template <typename XT, typename WT, int VEC, bool BLOCKS>
hipError_t launch_cl_w(int width, int seg, const void* x, const void* weight, const void* bias, void* out,
                       int64_t batch, int64_t seqlen, int64_t dim, int act, hipStream_t s) {
  const int64_t groups = dim / VEC, segs = (seqlen + seg - 1) / seg;
  const int64_t items = batch * segs * groups;
  const dim3 grid((unsigned)((items + kClThreads - 1) / kClThreads));
#define THM_CL_LAUNCH(WV, SL)                                                                             \
  hipLaunchKernelGGL((causal_conv1d_cl_kernel<XT, WT, VEC, WV, SL, BLOCKS>), grid, dim3(kClThreads), 0, s,   \
                     (const XT*)x, weight, bias, (XT*)out, seqlen, dim, seg, (uint32_t)groups,             \
                     (uint32_t)segs, (uint32_t)items)
  switch (width) {
#define THM_CL_W(WV)                                     \
  case WV:                                               \
    if (act == THM_ACT_SILU) THM_CL_LAUNCH(WV, true);    \
    else THM_CL_LAUNCH(WV, false);                       \
    break;
    THM_CL_W(1)
    THM_CL_W(2)
    THM_CL_W(3)
    THM_CL_W(4)
    THM_CL_W(5)
    THM_CL_W(6)
    THM_CL_W(7)
    THM_CL_W(8)
#undef THM_CL_W
#undef THM_CL_LAUNCH
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Steps per lane: waves take a start of about four steps (the window, the
// taps) and their own steps, on a SIMD one after another in whole waves, and a
// SIMD needs two to cover their loads; the last segment repeats steps of the
// one before it.  So a length that leaves the SIMDs two waves each beats a
// shorter one with four, and both beat two and a half.  us at segments of
// 8 / 16 / 32 / 64 (two waves per SIMD at the marked one):
//   bf16 [8, 8192, 4096] 209 / 214 / 196 / 190, [2, 5001, 4352] 42 / 39 / 37 /
//     44, [1, 1000, 4352] 8.1 / 9.4 / 14 / 24, [4, 2048, 4096] 33 / 31 / 27 /
//     27*, [4, 5001, 2048] 39 / 33 / 36 / 44, [8, 2500, 6144] 102 / 94 / 100 /
//     104;
//   fp32 [4, 2048, 4096] - / 61 / 62 / 51*, [1, 8192, 2048] - / 29 / 27* / 29,
//     [1, 5001, 4352] - / 39 / 37 / 40, [4, 5001, 2048] - / 69 / 70 / 77, [8,
//     257, 6144] - / 25 / 25 / 27, [8, 1000, 6144] - / 82 / 81 / 87 (taken: 64).
inline int cl_segment(int64_t batch, int64_t seqlen, int64_t groups, int depth) {
  const int64_t simds = 4 * (int64_t)std::max(device_cu_count(), 1);
  int best = depth;
  int64_t least = INT64_MAX;
  for (int seg = kClSeg; seg >= depth; seg /= 2) {
    const int64_t items = batch * ((seqlen + seg - 1) / seg) * groups;
    if (seg > seqlen || (seg < kClSeg && !launch_fits((items + kClThreads - 1) / kClThreads, kClThreads))) continue;
    const int64_t waves = (items + kWave - 1) / kWave;
    const int64_t cost = std::max<int64_t>((waves + simds - 1) / simds, 2) * (seg + 4);
    if (cost < least) {
      least = cost;
      best = seg;
    }
  }
  return best;
}

template <typename XT, typename WT>
hipError_t launch_cl(bool vec_ok, int width, const void* x, const void* weight, const void* bias, void* out,
                     int64_t batch, int64_t seqlen, int64_t dim, int act, hipStream_t s) {
  constexpr int VEC = 16 / (int)sizeof(XT);
  if (!vec_ok) return launch_cl_w<XT, WT, 1, false>(width, kClSeg, x, weight, bias, out, batch, seqlen, dim, act, s);
  constexpr int kDepth = cl_depth<XT>();
  if (seqlen < kDepth) return launch_cl_w<XT, WT, VEC, false>(width, kClSeg, x, weight, bias, out, batch, seqlen, dim, act, s);
  const int seg = cl_segment(batch, seqlen, dim / VEC, kDepth);
  return launch_cl_w<XT, WT, VEC, true>(width, seg, x, weight, bias, out, batch, seqlen, dim, act, s);
}

template <typename XT>
__global__ void __launch_bounds__(256)
causal_conv1d_update_kernel(const XT* __restrict__ x, XT* __restrict__ state,
                            const void* __restrict__ weight, const void* __restrict__ bias,
                            XT* __restrict__ out, int64_t rows, int64_t dim, int64_t seqlen,
                            int64_t state_len, int width, int w_is_bf16, int act) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // b * dim + d
  if (row >= rows) return;
  const int64_t d = row % dim;
  float wk[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) wk[k] = (k < width) ? conv_param(weight, d * width + k, w_is_bf16) : 0.f;
  const float b0 = bias ? conv_param(bias, d, w_is_bf16) : 0.f;
  XT* __restrict__ st = state + row * state_len;
  const XT* __restrict__ xr = x + row * seqlen;
  XT* __restrict__ orow = out + row * seqlen;
  // window = st ++ xr;  window index i is st[i] for i < L_s, else xr[i - L_s].
  auto at = [&](int64_t i) { return to_f32(i < state_len ? st[i] : xr[i - state_len]); };
  for (int64_t t = 0; t < seqlen; ++t) {
    float acc = b0;
    const int64_t base = state_len - (width - 1) + t;
    for (int k = 0; k < width; ++k) acc = __builtin_fmaf(wk[k], at(base + k), acc);
    if (act == THM_ACT_SILU) silu<XT, 1>(&acc);
    orow[t] = from_f32<XT>(acc);
  }
  // New state: the last L_s window samples, written front to back (the
  // source index i + seqlen is never below the destination i).
  for (int64_t i = 0; i < state_len; ++i) st[i] = i + seqlen < state_len ? st[i + seqlen] : xr[i + seqlen - state_len];
}

// One new sample per row and a state of W - 1 + OFF samples (OFF 0 or 1: what a
// decode loop keeps): the state, the taps and the sample are loaded whole and
// all at once, where the general kernel's loop waits for each tap in turn.
// [64, 4096] bf16, W = 4, kernel trace: 5.6 -> 2.5 us.
template <typename XT, typename WT, int W, int OFF>
__global__ void __launch_bounds__(256)
causal_conv1d_step_kernel(const XT* __restrict__ x, XT* __restrict__ state, const void* __restrict__ weight,
                          const void* __restrict__ bias, XT* __restrict__ out, uint32_t rows, uint32_t dim, int act) {
  constexpr int L = W - 1 + OFF;
  const uint32_t row = blockIdx.x * 256 + threadIdx.x;  // b * dim + d
  if (row >= rows) return;
  const uint32_t d = row % dim;
  XT win[L + 1];  // the state, then the new sample
  WT wk[W];
  XT* const st = state + (int64_t)row * L;
  if constexpr (L > 0) __builtin_memcpy(win, st, L * sizeof(XT));
  __builtin_memcpy(wk, reinterpret_cast<const WT*>(weight) + (int64_t)d * W, W * sizeof(WT));
  win[L] = x[row];
  float acc = bias ? to_f32(reinterpret_cast<const WT*>(bias)[d]) : 0.f;
#pragma unroll
  for (int k = 0; k < W; ++k) acc = __builtin_fmaf(to_f32(wk[k]), to_f32(win[OFF + k]), acc);
  if (act == THM_ACT_SILU) silu<XT, 1>(&acc);
  out[row] = from_f32<XT>(acc);
  if constexpr (L > 0) __builtin_memcpy(st, win + 1, L * sizeof(XT));
}

template <typename XT, typename WT, int OFF>
hipError_t launch_step(int width, const void* x, void* state, const void* weight, const void* bias, void* out,
                       int64_t rows, int64_t dim, int act, hipStream_t s) {
  const dim3 grid((unsigned)((rows + 255) / 256));
  switch (width) {
#define THM_STEP_W(WV)                                                                                              \
  case WV:                                                                                                          \
    hipLaunchKernelGGL((causal_conv1d_step_kernel<XT, WT, WV, OFF>), grid, dim3(256), 0, s, (const XT*)x, (XT*)state, \
                       weight, bias, (XT*)out, (uint32_t)rows, (uint32_t)dim, act);                                 \
    break;
    THM_STEP_W(1)
    THM_STEP_W(2)
    THM_STEP_W(3)
    THM_STEP_W(4)
    THM_STEP_W(5)
    THM_STEP_W(6)
    THM_STEP_W(7)
    THM_STEP_W(8)
#undef THM_STEP_W
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename XT>
hipError_t launch_update(const void* x, void* state, const void* weight, const void* bias, void* out,
                         int64_t batch, int64_t dim, int64_t seqlen, int64_t state_len, int width,
                         int wb, int act, hipStream_t s) {
  const int64_t rows = batch * dim;
  if (seqlen == 1 && state_len == width - 1)
    return wb ? launch_step<XT, bf16, 0>(width, x, state, weight, bias, out, rows, dim, act, s)
              : launch_step<XT, float, 0>(width, x, state, weight, bias, out, rows, dim, act, s);
  if (seqlen == 1 && state_len == width)
    return wb ? launch_step<XT, bf16, 1>(width, x, state, weight, bias, out, rows, dim, act, s)
              : launch_step<XT, float, 1>(width, x, state, weight, bias, out, rows, dim, act, s);
  const dim3 grid((unsigned)((rows + 255) / 256));
  hipLaunchKernelGGL((causal_conv1d_update_kernel<XT>), grid, dim3(256), 0, s, (const XT*)x,
                     (XT*)state, weight, bias, (XT*)out, rows, dim, seqlen, state_len, width, wb, act);
  return hipGetLastError();
}

}  // namespace
}  // namespace thm

extern "C" int thm_causal_conv1d_fwd_channels_last(const void* x, const void* weight,
                                                   const void* bias, void* out, int64_t batch,
                                                   int64_t seqlen, int64_t dim, int32_t width,
                                                   int32_t x_dtype, int32_t w_dtype,
                                                   int32_t activation, void* stream) {
  using namespace thm;
  if (batch < 0 || dim <= 0 || seqlen < 0) return THM_ERR_BAD_SHAPE;
  if (x_dtype != THM_DTYPE_F32 && x_dtype != THM_DTYPE_BF16) return THM_ERR_BAD_DTYPE;
  if (w_dtype != THM_DTYPE_F32 && w_dtype != THM_DTYPE_BF16) return THM_ERR_BAD_DTYPE;
  if (width < 1 || width > 8) return THM_ERR_UNSUPPORTED;
  if (activation != THM_ACT_NONE && activation != THM_ACT_SILU) return THM_ERR_BAD_ARGUMENT;
  if (batch == 0 || seqlen == 0) return THM_OK;
  if (!x || !weight || !out) return THM_ERR_NULL_POINTER;
  const int64_t xe = (x_dtype == THM_DTYPE_F32) ? 4 : 2;
  const int64_t we = (w_dtype == THM_DTYPE_F32) ? 4 : 2;
  if (((uintptr_t)x % xe) || ((uintptr_t)out % xe) || ((uintptr_t)weight % we) ||
      (bias && ((uintptr_t)bias % we)))
    return THM_ERR_MISALIGNED;
  if (batch > (INT64_C(1) << 40) / dim || batch * dim > (INT64_C(1) << 46) / seqlen)
    return THM_ERR_BAD_SHAPE;
  const int vec = (int)(16 / xe);
  const bool vec_ok = ((uintptr_t)x % 16 == 0) && ((uintptr_t)out % 16 == 0) && (dim % vec == 0);
  const int64_t groups = vec_ok ? dim / vec : dim;
  // (Below 2^32 lanes, so the kernel's 32-bit indices hold; cl_segment keeps
  // shorter segments to it too.)
  if (!launch_fits(batch * ((seqlen + kClSeg - 1) / kClSeg) * ((groups + kClThreads - 1) / kClThreads), kClThreads))
    return THM_ERR_BAD_SHAPE;
  const int wb = (w_dtype == THM_DTYPE_BF16);
  hipStream_t s = (hipStream_t)stream;
  auto run = [&](auto xt) {
    using XT = decltype(xt);
    return wb ? launch_cl<XT, bf16>(vec_ok, width, x, weight, bias, out, batch, seqlen, dim, activation, s)
              : launch_cl<XT, float>(vec_ok, width, x, weight, bias, out, batch, seqlen, dim, activation, s);
  };
  const hipError_t e = x_dtype == THM_DTYPE_F32 ? run(float{}) : run(bf16{});
  return (int)e;
}

extern "C" int thm_causal_conv1d_update(const void* x, void* conv_state, const void* weight,
                                        const void* bias, void* out, int64_t batch, int64_t dim,
                                        int64_t seqlen, int64_t state_len, int32_t width,
                                        int32_t x_dtype, int32_t w_dtype, int32_t activation,
                                        void* stream) {
  using namespace thm;
  if (batch < 0 || dim <= 0 || seqlen < 0 || state_len < 0) return THM_ERR_BAD_SHAPE;
  if (x_dtype != THM_DTYPE_F32 && x_dtype != THM_DTYPE_BF16) return THM_ERR_BAD_DTYPE;
  if (w_dtype != THM_DTYPE_F32 && w_dtype != THM_DTYPE_BF16) return THM_ERR_BAD_DTYPE;
  if (width < 1 || width > 8) return THM_ERR_UNSUPPORTED;
  if (state_len < width - 1) return THM_ERR_BAD_SHAPE;  // the window must cover the taps
  if (activation != THM_ACT_NONE && activation != THM_ACT_SILU) return THM_ERR_BAD_ARGUMENT;
  if (batch == 0 || seqlen == 0) return THM_OK;  // nothing new: the state is unchanged
  if (!x || !weight || !out || (state_len > 0 && !conv_state)) return THM_ERR_NULL_POINTER;
  const int64_t xe = (x_dtype == THM_DTYPE_F32) ? 4 : 2;
  const int64_t we = (w_dtype == THM_DTYPE_F32) ? 4 : 2;
  if (((uintptr_t)x % xe) || ((uintptr_t)out % xe) || ((uintptr_t)conv_state % xe) ||
      ((uintptr_t)weight % we) || (bias && ((uintptr_t)bias % we)))
    return THM_ERR_MISALIGNED;
  if (batch > (INT64_C(1) << 38) / dim || !launch_fits((batch * dim + 255) / 256, 256)) return THM_ERR_BAD_SHAPE;
  const int wb = (w_dtype == THM_DTYPE_BF16);
  hipStream_t s = (hipStream_t)stream;
  const hipError_t e =
      (x_dtype == THM_DTYPE_F32)
          ? launch_update<float>(x, conv_state, weight, bias, out, batch, dim, seqlen, state_len, width, wb, activation, s)
          : launch_update<bf16>(x, conv_state, weight, bias, out, batch, dim, seqlen, state_len, width, wb, activation, s);
  return (int)e;
}
