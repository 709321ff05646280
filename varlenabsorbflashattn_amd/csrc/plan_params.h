// Tile sizes and key-split policy shared by the planner and the kernels.
#pragma once
#include <cstdint>

namespace vafa {

// Varlen: a forward / dQ workgroup covers one query tile (32 rows per wave)
// and a dK/dV workgroup one key tile (32 keys per wave).  The planner picks
// each per call between kVarlenTile (4-wave workgroups) and kVarlenWideTile
// (8-wave workgroups, D <= 128 only: at D=256 one wave per SIMD holds the
// registers); the fused K-major pass always uses kVarlenTile keys.
constexpr int kVarlenTile = 128;
constexpr int kVarlenWideTile = 256;
// Absorb: a forward workgroup covers up to kAbsorbRows (token, head) rows;
// a dX workgroup covers up to kAbsorbKTile keys of one sample (two 128-key
// sub-tiles on the matrix-core path), kAbsorbSmallKTile in launches of at most
// kAbsorbSmallKeys keys, whose dX grid would leave CUs idle (D_KV > 256:
// kAbsorbWideF below).  GPU time of
// forward + backward, us, at 512 / 256 / 128 keys: C4 (648k keys) 543 / 543 /
// 547, 1127 samples of <= 2048 keys (1.37M) 969 / 949 / 994, 256 and 64 C4
// samples (80k, 20k) 162 / 155 / 157 and 131 / 121 / 115, 512 C4 samples in
// fp32 (157k) 984 / 938 / 893.
constexpr int kAbsorbRows = 64;
constexpr int kAbsorbKTile = 256;
constexpr int kAbsorbSmallKTile = 128;
constexpr int64_t kAbsorbSmallKeys = 192 * 1024;

struct SplitPolicy {
  // Query tiles with at most `decode_rows` rows against >= decode_min_keys
  // keys are split into clamp(ceil(Lk/decode_chunk), min, max) chunks.
  int64_t decode_rows, decode_min_keys, decode_chunk, decode_min_split, decode_max_split;
  // Any other tile is split into ceil(Lk/long_chunk) chunks once
  // Lk > long_threshold (fa/interface.py:46-57 uses 4096 / 4096).
  int64_t long_threshold, long_chunk;
  int64_t align;          // chunk lengths are multiples of this many keys
  int64_t item_overhead;  // fixed per-item cost (keys-equivalent) for LPT
};

constexpr SplitPolicy kVarlenPolicy{16, 1024, 2048, 4, 16, 4096, 4096, 64, 64};
// vafa_plan_varlen_balanced: launches whose items cannot fill `cus` CUs evenly.
// 256-row (256-key) tiles become 128 where the longest walk exceeds a CU's
// share of the work.  Below 3/5 item per resident 128-row workgroup (two per
// CU; 4/5 at D = 256, one per CU) key ranges split beyond 3/2 of the average
// keys per workgroup, below two items each decode tiles into chunks of half of
// it (up to twice the splits), chunks of at least min_chunk keys before a range is
// divided evenly (513 keys end as 320 + 193), and only while the fp32 partial rows
// stay within max_part_bytes.  GPU time, us, fixed rules ->
// balanced (self-attention lengths log-uniform in [1, 4096] unless stated, H =
// heads): 16 sequences D = 128 H = 4 forward + backward 262 -> 215, 8 sequences
// H = 16 227 -> 206, 16 sequences D = 256 H = 2 402 -> 341, fp32 D = 64 32
// sequences of <= 2048 H = 8 1148 -> 990 and H = 2 967 -> 505; 500 queries
// against 3 histories of <= 8611 keys 157 -> 77; decode of 4 x 24k keys H = 4
// 49 -> 33.  On launches that fill the chip the same splits lose: 64 sequences
// D = 128 H = 16 2071 -> 2289 with 2048-key chunks, 8 sequences 215 -> 270 with
// 1024.
struct VarlenBalance {
  int64_t cus, min_chunk, max_part_bytes;
};
constexpr VarlenBalance kVarlenBalance{256, 512, 32 << 20};
// Absorb forward key splits.  A chunk holds kAbsorbSlack2 / 2 times the
// average keys per resident forward workgroup (256 CUs x 3 on the MI355X), so
// large launches stay whole (splitting C5's <= 8192-key samples into 1024-key
// chunks cost 10%, C4's <= 2000-key samples at 1024 keys 4%), and a small
// launch splits down to long_chunk keys, where one workgroup's walk over the
// longest sample is the launch's whole time.  Chunks below kAbsorbWideChunk
// are taken only while kAbsorbFineSplits of them cover the range (each costs a
// prologue, an epilogue and a partial row set).  GPU time of the forward, us,
// with chunks of at least 1024 keys at 3x the average -> this rule: 16 C4
// samples 43.7 -> 31.5, 256 / 512 skewed (C5) samples 157 / 275 -> 139 / 236,
// 512 C4 samples in fp32 246 -> 235, C4 and C5 themselves unchanged; smallest
// chunk 128 / 256 / 512: 31.4 / 33.9 / 38.2 on the 16 samples.
constexpr SplitPolicy kAbsorbPolicy{0, 1 << 30, 128, 1, 16, 128, 128, 64, 32};
constexpr int64_t kAbsorbWideChunk = 1024;
constexpr int64_t kAbsorbFineSplits = 16;
constexpr int64_t kAbsorbSlots = 768;
constexpr int64_t kAbsorbSlack2 = 5;
// Absorb backward, dU pass: two resident workgroups per CU; a chunk holds
// kAbsorbDuSlack times the average keys per workgroup.  A split tile writes
// and re-reads 8 bytes of fp32 partials per (row, feature), so only ranges above
// 256 keys split (evenly: 257 keys into 192 + 65).  GPU time of forward + backward,
// us, whole ranges -> split:
// 64 / 256 / 700 C4 samples 158 / 201 / 257 -> 131 / 162 / 234, 512 and 64 C4
// samples in fp32 1318 -> 985 and 872 -> 548; all of C4 unchanged (544, whole
// at this slack; 553 at half of it).
constexpr SplitPolicy kAbsorbDuPolicy{0, 1 << 30, 256, 1, 16, 256, 256, 64, 32};
constexpr int64_t kAbsorbDuSlots = 512;
constexpr int64_t kAbsorbDuSlack = 2;
// D_KV > kAbsorbWideF: one workgroup per CU in every pass, and an item costs a
// prologue and an epilogue worth kAbsorbWideItem + D_H keys, which count towards
// the average.  Forward chunks hold 5/4 of the average keys per CU, but no more
// than 1024 or 1/256 of the keys (chunks of that size keep the tail of a large launch
// short); dU chunks twice the average; dX tiles of 128, 256 or 512 keys leave one
// per CU.  Forward / forward + backward, us, at whole ranges and 512-key dX tiles -> the
// rules of narrower features -> these, D_KV 512: 512 samples of 8 heads of 32 72 / 415 ->
// 79 / 455 -> 72 / 414; 512 of 8 heads of 128 145 / 604 -> 172 / 677 -> 145 / 598; 64
// and 256 of 16 heads of 128 121 / 610 -> 153 / 506 -> 116 / 451 and 182 / 764 -> 231 /
// 818 -> 182 / 730; 64 and 256 of 8 heads of 32 in fp32, whose products outweigh an
// item's cost, 379 / 2066 -> 97 / 426 -> 115 / 444 and 410 / 2171 -> 225 / 945 -> 241 /
// 1106 (the planner does not see the data type).
constexpr int64_t kAbsorbWideF = 256;
constexpr int64_t kAbsorbWideSlots = 256;
constexpr int64_t kAbsorbWideItem = 64;
// A segment without queries is cleared by items of at most kAbsorbClearKeys keys.
// In the longest-first order a key counts as kAbsorbClearCost rows: it is stored
// and not read, about half of what a tile of 32 rows moves.  One item for the whole
// range, 16 to 32 threads storing a key at a time, ended the launch alone: 256 samples
// (D_KV = 256) beside one of 20k / 200k keys without queries, forward + backward
// 603 / 5114 us -> 155 / 157.
constexpr int64_t kAbsorbClearKeys = 1024;
constexpr int64_t kAbsorbClearCost = 16;

// Varlen backward, fused K-major path (dQ, dK, dV in one kernel, fp32 dQ
// partials per key chunk summed in order): segments with at most kFusedMaxQ
// queries and at least kFusedMinK keys, at head dims up to kFusedMaxD.  Each
// chunk writes Lq*D*4 bytes of partial dQ (plus the read back in the sum) and
// saves the second read of its K/V rows that the query-major dQ kernel makes.
// Measured on the MI355X with one 128-key tile per item (64 segments x 8192
// keys, backward
// ms, two-kernel vs fused): H=4 D=64 Lq=1/8/16: 0.447/0.440/0.451 vs
// 0.379/0.387/0.394; Lq=32 0.443 vs 0.440; Lq=48/64 0.487/0.472 vs
// 0.519/0.561.  At D=128 the fused kernel holds one workgroup per CU (256
// VGPRs + 225 AGPRs, 117 KB of LDS) and lost at every Lq (1.57-1.59 vs
// 1.65-1.95 ms at H=8), so it serves D <= 64 only.
constexpr int kFusedMaxQ = 16;
constexpr int kFusedMinK = 1;
constexpr int kFusedMaxD = 64;
// A fused item walks up to kFusedTiles 128-key tiles of one segment (the
// query block staged once, dQ summed over the chunk in registers).  Measured
// on the MI355X, backward ms for 1 / 2 / 3 / 4 tiles per item: 64 x 16 queries
// x 8192 keys (H=4, D=64) 0.667 / 0.666 / 0.607 / 0.750; 256 x 8 x 2048 keys
// 0.644 / 0.663 / 0.638 / 0.780; 32 x 1 x 32768 keys (H=8) 2.47 / 2.41 /
// 2.37 / 2.44.
constexpr int kFusedTiles = 3;

// Workgroups are dispatched round-robin over this many XCDs (one L2 each):
// workgroup i runs on XCD i % kXcds.
constexpr int kXcds = 8;

// Absorb dX: a segment with at most this many (token, head) rows keeps all of
// them resident in one workgroup (absorb_dx_res_kernel); longer segments are
// streamed in 32-row blocks (absorb_dx_kernel).
constexpr int kDxResidentRows = 64;
// 16-bit backward: the segments of at most kDxResidentRows rows run on the
// merged kernel when they are all of the launch or hold at least this many X
// elements (keys x D_KV).  In a mixed launch the merged kernel runs ahead of the
// other two, whose CUs it leaves idle at its end, so the pass over X that it saves
// has to be worth a kernel's tail, however long the other segments are.  Forward +
// backward, us, not merged / merged at M elements (samples of <= 2048 keys, 8 heads):
// D_KV 256  M = 40M 480 / 508, 58M 598 / 622, 82M 556 / 558, 96M 383 / 381, 106M
// 362 / 343, 119M 1077 / 1045, 191M 956 / 888, 16 heads 45M 457 / 491, 80M 759 / 734,
// 32 heads 85M 2224 / 2194; D_KV 192  62M 424 / 434, 72M 301 /
// 315, 89M 385 / 366, 103M 368 / 358; D_KV 128  29M 365 / 403, 60M 287 / 301, 74M
// 270 / 289, 67M (of 307M) 1235 / 1219, 96M 555 / 538, 129M 497 / 476.
constexpr int64_t kAbsorbMergedElems = int64_t{72} << 20;

}  // namespace vafa
