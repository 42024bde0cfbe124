// What the units of chunk_fwd_h share (chunk_fwd_h.hip: bf16 inputs and the
// entry points; chunk_fwd_h_f32.hip: fp32 inputs).
#pragma once

#include "common.h"
#include "seg_plan.h"

namespace thm {
namespace {

constexpr int kBT = 64;
constexpr int kHBV = 64;  // V-tile width

// Grids of at least this many workgroups are bandwidth-bound: fp32 inputs then
// prefetch two chunks ahead (chunk_fwd_h_reg.h DEEP), bf16 inputs take the DMA
// pipeline of chunk_fwd_h.hip.
constexpr int64_t kHDmaMinGrid = 256;

__device__ __forceinline__ const char* cptr(const void* p, int64_t byte_off) {
  return reinterpret_cast<const char*>(p) + byte_off;
}

}  // namespace

// fp32 inputs, chunk_fwd_h_f32.hip (out, per, len: seg::Plan).
__attribute__((visibility("hidden"))) hipError_t chunk_fwd_h_f32(
    bool delta, int64_t K, int64_t V, const void* k, const void* w, const void* vu, const void* g, const void* h0,
    void* h, void* vnew, void* ht, char* ws, int64_t out, int64_t per, int64_t len, int64_t B, int64_t T, int64_t H,
    hipStream_t s);
}  // namespace thm
