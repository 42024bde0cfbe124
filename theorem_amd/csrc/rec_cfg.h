// Chunk records of the chunked Gated DeltaNet forward, and the layout of the
// kernels that read them (chunk_fwd_rec.hip, segments.h).  Plain constants and
// index maps, also compiled by the host-side check of their addressing
// (tests/csrc/dma_check.cpp).
//
// A record holds what the recurrence of one (b, head, chunk) needs besides
// the k, q and v rows, written by wy_build_A.hip's record form:
//   blocks 0..9: the lower 16 x 16 blocks (ib, jb <= ib) of A = (I + M)^{-1}
//     in the order ib (ib + 1) / 2 + jb, 1 KiB each, lane-major: lane
//     (grp, li) holds A[16 ib + li][16 jb + 4 grp .. + 3] as 4 bf16 hi then
//     4 bf16 lo (hi + lo = A to ~2^-16), half of an MFMA A operand in paired
//     contraction order;
//   then 256 floats, one per token each: the cumulative gates g, e^g,
//     e^{g_last - g} and beta.
// Records lie by (b, head), chunks in sequence, so a recurrence reads one
// contiguous stream.
#pragma once

#include <stdint.h>

#include "h_layout.h"

namespace thm {
namespace rec {

constexpr int kBT = 64;
constexpr int kBlocks = 10;
constexpr int kBlockBytes = 1024;
constexpr int kGateOff = kBlocks * kBlockBytes;
constexpr int kBytes = kGateOff + 1024;
// Float offsets in the gate part.
constexpr int kG = 0, kEg = 64, kEgl = 128, kBeta = 192;

// Gate input of the builder: none, or per-token log decays (optionally through
// log(sigmoid)) or their chunk-local cumulative sums, fp32 or bf16.
constexpr int kGateNone = 0, kGateCumulative = 1, kGatePerToken = 2, kGateLogsigmoid = 4, kGateBf16 = 8;

// Block (ib, jb <= ib) of a record.
THM_HD constexpr int block(int ib, int jb) { return ib * (ib + 1) / 2 + jb; }

// Byte offset of the record of chunk c of sequence bh = b H + head.
THM_HD constexpr int64_t offset(int64_t bh, int64_t c, int64_t NT) { return (bh * NT + c) * kBytes; }

// ---------------------------------------------------------------------------
// Output kernel: 4 state and 4 output wavefronts per (b, head, segment,
// 64-column V-tile); see chunk_fwd_rec.hip.
constexpr int kTileV = 64;
constexpr int kOThreads = 512;

template <int K>
struct OCfg {
  static constexpr int kRowK = K * 2, kTileK = kBT * kRowK;
  static constexpr int kRowV = kTileV * 2, kTileVB = kBT * kRowV;
  static constexpr int kStage = 2 * kTileK + kTileVB + kBytes;  // k, q, v tile, record
  static constexpr int KB = K / 16;
  static constexpr int kPBytes = kBT * kBT * 2;           // scores, bf16
  static constexpr int kSBytes = 4 * (KB / 2) * 64 * 16;  // S handed over as bf16 B-operand pairs
  static constexpr int kVBytes = 4 * 2 * 64 * 16;         // v_new handed over the same way
  static constexpr int kLds = 2 * kStage + kPBytes + kSBytes + kVBytes;
  static constexpr int kKDma = kTileK / 1024 / 4;         // 1 KiB DMA instructions per state wave per k / q tile
  static constexpr int kADma = (kBlocks + 3) / 4;         // ... of A blocks (the last repeat block 9)
  static constexpr int kVDma = kTileVB / 1024 / 4;
  // The block that DMA instruction i of state wave wq loads.
  THM_HD static constexpr int a_block(int wq, int i) { return wq + 4 * i < kBlocks ? wq + 4 * i : kBlocks - 1; }
  // Issue schedule as the A form of pipe_cfg.h FCfg: chunk x's k, q and gates
  // in phase 1 of chunk x - 1, its A blocks and v after the mid-chunk barrier
  // of chunk x - 2.  So after the k / q DMA of a chunk exactly one A / v set is
  // issued before the wait for it.
  static constexpr int kAvDma = kADma + kVDma;
  static constexpr int kWait = kAvDma;
  static_assert(kStage % 1024 == 0 && kLds <= 160 * 1024, "LDS budget");
};

// Transition kernel: one wavefront per 16 kCT columns of [P | Q], K + V in all.
// Stage: the k tile, the v tiles and the record; WU: k, u, w tiles and the gates.
template <int K, int V, bool WU>
struct TCfg {
  static constexpr int kCT = 2;  // 16-column tiles per wave
  static constexpr int kWaves = (K + V) / (16 * kCT), kThreads = 64 * kWaves;
  static constexpr int kPWaves = K / (16 * kCT);
  static constexpr int kRowK = K * 2, kTileK = kBT * kRowK;
  static constexpr int kRowV = kTileV * 2, kTileVB = kBT * kRowV;
  static constexpr int kNVT = V / kTileV;
  static constexpr int kStage = kTileK + kNVT * kTileVB + (WU ? kTileK + 1024 : kBytes);
  static constexpr int kStages = 3;
  static constexpr int kLds = kStages * kStage;
  // 1 KiB DMA instructions of a chunk, in the order of the stage, spread over
  // the waves round by round: every wave issues kDma, or one fewer where the
  // last round does not reach it.
  static constexpr int kKInstr = kTileK / 1024, kRInstr = (WU ? kTileK : kBytes) / 1024, kVInstr = kNVT * kTileVB / 1024;
  static constexpr int kInstr = kKInstr + kVInstr + kRInstr;
  // Instruction j = wave + i kWaves fills KiB j of the stage: its source (k, v
  // or the third) and the lane's offset there, tokens tsk (k, w) and tsv bytes apart.
  THM_HD static constexpr bool from_k(int j) { return j < kKInstr; }
  THM_HD static constexpr bool from_v(int j) { return j >= kKInstr && j < kKInstr + kVInstr; }
  THM_HD static constexpr uint32_t src_off(int j, int lane, int64_t tsk, int64_t tsv) {
    constexpr int kPer = kTileVB / 1024;  // instructions per v tile
    const int x = from_k(j) ? j : from_v(j) ? j - kKInstr : j - kKInstr - kVInstr;
    return from_k(j)   ? hl::dma_src_off(x * 64 + lane, kRowK, tsk)
           : from_v(j) ? hl::dma_src_off((x % kPer) * 64 + lane, kRowV, tsv) + (uint32_t)((x / kPer) * kRowV)
           : WU        ? hl::dma_src_off(x * 64 + lane, kRowK, tsk)
                       : (uint32_t)(x * 1024 + lane * 16);
  }
  // Byte offsets in a stage: the v tile of columns 64 t .., the record or w tile, the gates.
  static constexpr int kOffV = kTileK, kOffR = kTileK + kNVT * kTileVB, kOffG = kInstr * 1024 - (WU ? 0 : 1024);
  static constexpr int kDma = (kInstr + kWaves - 1) / kWaves;
  static constexpr int kWait = (kStages - 2) * kDma;
  static_assert(kStage % 1024 == 0 && kLds <= 160 * 1024, "LDS budget");
};

// Workspace blocks of the segmented form, fp32 in 1 KiB lane-major 16 x 16
// blocks: P (K x K) of segment s >= 1 and the state at the start of segment
// s + 1 (K x V; first Q of segment s), s < segments - 1.
// P's blocks are of A-operand lanes: lane (grp, li) holds row li, columns 4 grp
// .. + 3.  A lane that holds row 4 grp + li / 4, columns 4 (li % 4) .. + 3 (an
// accumulator after acc_to_row_quads) writes them at p_slot.
THM_HD constexpr int p_slot(int lane) { return 16 * (lane & 3) + 4 * (lane >> 4) + ((lane & 15) >> 2); }
THM_HD constexpr int64_t p_off(int64_t s, int64_t bh, int64_t BH, int64_t K) { return ((s - 1) * BH + bh) * K * K * 4; }
THM_HD constexpr int64_t s_off(int64_t s, int64_t bh, int64_t BH, int64_t K, int64_t V) { return (s * BH + bh) * K * V * 4; }

}  // namespace rec
}  // namespace thm
