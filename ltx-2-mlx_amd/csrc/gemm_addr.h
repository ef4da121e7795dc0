// Source addresses of the projection GEMMs' direct loads: plain integer
// arithmetic, constexpr so that the kernels and host code share it.
#pragma once

namespace ltx {

// XOR swizzle of a 128-byte LDS row that holds two 64-byte halves of 16x16
// fragment reads (chunk 4 half + q of rows r16): a lane-octet pair that is
// served together holds eight rows at q and eight at q ^ 1, and even rows keep
// chunk bit 0, so the pair covers all 64 banks.
constexpr int swz_pair(int row) { return row & 6; }

// A direct load fills 8 LDS rows of 128 bytes, lane j the 16-byte slot j & 7 of
// row j >> 3; the logical chunk that the lane loads (rows come in blocks of 8).
constexpr int pair_chunk(int lane) { return (lane & 7) ^ swz_pair(lane >> 3); }

// Past the last unit of K (stage, pair, ...) a ring loads the last one again.
constexpr int clamp_unit(int u, int units) { return u < units ? u : units - 1; }

// 64-byte stages in pairs: the pairs of `stages` stages, and what a lane's
// source offset goes back by in pair u.  In a last half pair (odd count) the
// lanes of the missing stage load the other stage's bytes, so that no load
// leaves its row: the buffer's record count does not bound the scalar offset,
// where the pair's advance along K sits.
constexpr int stage_pairs(int stages) { return (stages + 1) >> 1; }
constexpr bool half_pair(int u, int stages) { return (stages & 1) != 0 && u == stage_pairs(stages) - 1; }
constexpr int half_pair_back(int lane) { return (pair_chunk(lane) & 4) * 16; }

}  // namespace ltx
