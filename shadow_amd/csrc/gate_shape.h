// How the gated block's kernel (gate.hip) cuts a shape: host code without HIP, so that
// tests/test_gate_shape_cpu.py can go over shapes without a device.
#ifndef SHADOW_AMD_CSRC_GATE_SHAPE_H_
#define SHADOW_AMD_CSRC_GATE_SHAPE_H_

#include <cstdint>

namespace shdw {

constexpr uint32_t kGateMaxRows = 64;  // per workgroup: a lane of one wave each in the ordered sum
constexpr uint32_t kGateLanes = 256, kGateVectorBytes = 16;

// How a group's rows are summed by the wave that does it: a lane a row, which reads LDS as it adds, or the lanes shared out
// among the rows (gate_walk).
enum : int { kGateLaneARow = 1, kGateTogether = 2 };

// The walks that a form's shapes have (gate_shape below): several turns of four vectors are up to 512 numbers a row and eight
// rows or more; rows in chunks, of five vectors a lane and more, and of sixteen are long.
constexpr int gate_walks(int slots, bool whole, bool one) {
  return !whole || slots == 16 || (slots == 8 && one) ? kGateTogether : slots == 4 && !one ? kGateLaneARow : kGateLaneARow | kGateTogether;
}

// How a shape is cut.
struct GateShape {
  uint32_t log2_lanes, pieces, group, chunk, pitch;
  int slots, walk;
};

// Five workgroups on a CU: the tile and 3.5 KB of parameters, table and partial sums each
// (28.9 KB of 160), as many as the registers of eight vectors a lane leave room for
// (gate_waves).  Rows that do not fit whole go through LDS in chunks (four of the
// 112x112 planes' rows per CU instead of three, [16,64,112,112] 124 -> 81 us; with 18 KB
// eight 28x28 planes would be cut too, [32,512,28,28] 26.0 -> 28.1; both before gate_whole took them
// where BatchNorm, ReLU and a residual are there), unless there are no
// more than two workgroups per CU to hold.
constexpr uint32_t kGateTileBytes = 26000, kGateMaxTileBytes = 62000, kGateCus = 256;

// Lanes per row: as many as a row has vectors, up to a wave; the whole workgroup where
// a wave would take more than eight steps over a row, and where there are so few rows
// that a row per wave would leave CUs idle.  Rows per workgroup: what eight vectors per
// lane hold, fewer while that leaves under 1024 workgroups (four per CU).
inline GateShape gate_shape(uint32_t rows, uint32_t len) {
  const uint32_t nv = (len + 3) / 4;
  GateShape g{};
  g.log2_lanes = nv <= 16 ? 4 : nv <= 32 ? 5 : nv <= 512 ? 6 : 8;
  if (nv > 16 && rows < 1024) g.log2_lanes = 8;
  const uint32_t lanes = 1u << g.log2_lanes, turn_rows = kGateLanes >> g.log2_lanes;
  g.pieces = (nv + lanes - 1) / lanes;
  uint32_t turns = g.pieces <= 8 ? 8 / g.pieces : 1;
  if (turns * turn_rows > kGateMaxRows) turns = kGateMaxRows / turn_rows;
  while (turns > 1 && (rows + turns * turn_rows - 1) / (turns * turn_rows) < 1024u) --turns;
  const uint32_t used = turns * g.pieces;
  g.slots = used <= 1 ? 1 : used <= 4 ? 4 : used <= 8 ? 8 : 16;
  g.group = turns * turn_rows;
  // LDS holds equal chunks of the rows, as few as fit the tile; the pitch is an odd
  // number of vectors, so that the summing lanes meet different banks.
  for (uint32_t chunks = 1;; ++chunks) {
    g.chunk = (g.pieces + chunks - 1) / chunks;
    g.pitch = (g.chunk * lanes < nv ? g.chunk * lanes : nv) | 1u;
    const uint32_t bytes = g.group * g.pitch * kGateVectorBytes;
    if (bytes <= (rows <= 2 * kGateCus * g.group ? kGateMaxTileBytes : kGateTileBytes) || g.chunk == 1) break;
  }
  // Together, an addition takes 4.8 cycles instead of 8, but has its SIMD to itself meanwhile, and what a chunk's last
  // lanes lack is added as zeros.  So where rows are long for their number, or their walks few enough to have a SIMD
  // each.  A lane a row / together, us: groups of four, 6700 rows of 784 9.6 / 9.1, of 400 6.9 / 6.5, of 225 5.5 / 5.9, but
  // 4000 (1000 workgroups) 5.0 / 4.9; of eight, 13000 of 784 21.3 / 20.7, 10000 of 289 7.9 / 8.2; of twelve, 13000 of 225
  // 8.9 / 9.4; of sixteen, 30000 of 49 5.1 / 5.7, of 289 18.8 / 19.8.
  const uint32_t grid = (rows + g.group - 1) / g.group;
  const bool together = len >= 96 * g.group || (g.group <= 4 && grid <= 4 * kGateCus) || g.chunk != g.pieces;
  g.walk = together ? kGateTogether : kGateLaneARow;
  return g;
}

// How whole_squeeze_gate_kernel cuts rows of nv whole vectors: `pieces` vectors of one row a lane.
struct GateWhole {
  uint32_t log2_lanes, pieces, group, pitch;
};

constexpr uint32_t kGateWholePieces = 15, kGateWholeMinVectors = 96, kGateWholeFewRows = 1024;
constexpr uint32_t kGateWholeTileBytes = 33000;  // four workgroups a CU; a row of the whole workgroup may take kGateMaxTileBytes

// Of 16, 32, 64 and 256 lanes a row, the ones with the fewest vector instructions an element: about 16 an
// element of a lane's share, whether it holds something or not, and the walk's additions, of which
// one instruction serves all rows of a workgroup; but with less than 1024 workgroups as many lanes as gate_shape
// takes ([32,512,28,28] 22.4 us with 32 lanes, 23.8 with 64; [8,512,28,28] 9.2 and 8.0; [64,64,40,40] 13.1 with 64, 14.3 with
// 256; [2,256,28,28] 6.9 / 5.7 / 5.4 with 32 / 64 / 256).  false: no cut holds the rows, or many rows are so short
// that squeeze_gate_kernel's several rows a lane are faster ([64,512,14,14] 11.5 and 12.8 at best, [64,256,20,20] 11.5 and 11.2).
inline bool gate_whole(uint32_t rows, uint32_t len, GateWhole* out) {
  const uint32_t nv = len / 4, usual = gate_shape(rows, len).log2_lanes;
  if (nv < kGateWholeMinVectors && rows >= kGateWholeFewRows) return false;
  float least = 0.f;
  bool found = false;
  for (uint32_t log2_lanes = 4; log2_lanes <= 8; log2_lanes += log2_lanes == 6 ? 2 : 1) {
    const uint32_t lanes = 1u << log2_lanes, pieces = (nv + lanes - 1) / lanes, group = kGateLanes >> log2_lanes, pitch = nv | 1u;
    const uint32_t bytes = group * pitch * kGateVectorBytes;
    if (pieces > (log2_lanes == 8 ? kGateWholePieces : 8u) || bytes > (log2_lanes == 8 ? kGateMaxTileBytes : kGateWholeTileBytes)) continue;
    if ((rows + group - 1) / group < 1024u && log2_lanes != usual) continue;
    const float cost = 16.f * static_cast<float>(pieces * lanes) / static_cast<float>(nv) + 64.f / static_cast<float>(group);
    if (found && cost >= least) continue;
    found = true, least = cost;
    *out = GateWhole{log2_lanes, pieces, group, pitch};
  }
  return found;
}

// Whether a call is whole_squeeze_gate_kernel's, and its cut.  vec: whole, aligned vectors in every row.
inline bool gate_takes_whole(bool vec, bool stats, bool relu, bool residual, uint32_t rows, uint32_t len, GateWhole* out) {
  return vec && stats && relu && residual && gate_whole(rows, len, out);
}

}  // namespace shdw

#endif  // SHADOW_AMD_CSRC_GATE_SHAPE_H_
