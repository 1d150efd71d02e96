// How Softmax's tile kernel (softmax.hip) cuts a shape: host code without HIP, so that
// tests/test_softmax_shape_cpu.py can go over shapes without a device.
#ifndef SHADOW_AMD_CSRC_SOFTMAX_SHAPE_H_
#define SHADOW_AMD_CSRC_SOFTMAX_SHAPE_H_

#include <cstdint>

namespace shdw {

constexpr uint32_t kSoftmaxTileLanes = 256, kSoftmaxTileTable = 256;  // lanes of a workgroup, bytes of the exponential's table

// A shape's tiles: 1 << shift positions each, vectors a lane has room for (what fixes how many waves a SIMD
// holds), steps of rows that LDS holds at a time (two at least, an even number), all of them or a part.
struct SoftmaxTiles {
  int shift, slots;
  uint32_t grid, steps, pass_steps, lds_bytes;
  bool whole() const { return pass_steps >= steps; }
};

// Waves per SIMD that `slots` vectors a lane leave room for.
constexpr uint32_t softmax_tile_waves(int slots) { return slots == 8 ? 7 : slots == 10 ? 6 : 4; }

// LDS: `rows` of a tile, the exponentials' table, and a tile row for each of the four waves.
constexpr uint32_t softmax_tile_bytes(uint32_t rows, int shift) {
  return (rows << shift) * 4u + kSoftmaxTileTable + (4u << shift) * 4u;
}

// Positions: as many as a lane's sixteen vectors hold (64, 32 or 16), or half of them where that
// gives no more than three tiles a CU ([1,150,5184] 7.1 us with 64 positions, 5.7 with 32; [4,150,5184] 9.5, 8.7;
// [8,150,5184], 1296 tiles of 32, 12.0 and 12.5; [4,500,3025] 19.2 with 32, 16.1 with 16; [16,300,1444] 16.2, 16.8), and
// where a lane of 64 positions had more than ten vectors, as long as the chip holds seven a CU ([16,250,1444]
// 16.1 and 13.7, [16,250,3136] 22.5 in two passes, 19.8; [64,250,1444] 41.7 and 45.7).  Not tiles of 32 if the last one of a row
// of them has four positions or fewer: eight lanes of its waves have work, and for reasons not known such tiles
// finish last where there are few (64 / 32 / 16 positions: [40,80,100] 4.7 / 6.0 / 3.9 us, but with eight more positions 4.8 / 4.5 /
// 4.0, [40,200,97] 9.2 / 10.5 / 6.2, [6,150,164] 6.5 / 7.5 / 4.7, [200,200,100] 11.7 / 12.5 / 10.9).
//
// Vectors: the fewest of eight, ten and sixteen that do (of 64 positions, ten / eight vectors for 91 rows: [62,91,1605] 20.3 /
// 19.0 us, [123,91,1605] 35.2 / 31.5).
//
// Passes: one, unless LDS and not the registers holds the number of tiles a CU down and two passes of half the rows
// bring all tiles onto the chip at once, but for a fifth, or where one pass leaves room for no more than two a CU.  One / two:
// [49,150,1920], 1470 tiles, 25.9 / 19.8 us, [36,512,805] 36.5 / 27.4, [62,1000,405] 72.5 / 68.1; with a fifth left over [54,150,1920]
// 28.1 / 25.1, [62,150,1605] 29.6 / 28.4, but for 32 and 16 positions in rows that share sectors with the neighbouring
// tile's [68,320,805] 38.1 / 39.2, [62,640,405] 44.0 / 49.5; more rounds [158,150,1605] 59.3 / 63.6, [123,640,405] 72.9 / 82.0.
inline SoftmaxTiles softmax_tiles(int outer_num, int dim, int inner_num, bool sectors) {
  constexpr uint32_t kCus = 256, kCuLds = 160 * 1024, kFewTiles = 3 * kCus, kNarrowTiles = 7 * kCus;
  const auto tiles = [&](int shift) {
    return static_cast<uint32_t>(outer_num) * ((static_cast<uint32_t>(inner_num) + (1u << shift) - 1) >> shift);
  };
  const uint32_t d = static_cast<uint32_t>(dim);
  SoftmaxTiles t{};
  t.shift = d <= 256 ? 6 : d <= 512 ? 5 : 4;
  const uint32_t few = t.shift == 6 && d > 160 ? kNarrowTiles : kFewTiles, over = static_cast<uint32_t>(inner_num) % 32;
  if (t.shift > 4 && tiles(t.shift - 1) <= few) {
    --t.shift;
    if (t.shift == 5 && over >= 1 && over <= 4 && tiles(4) <= few) t.shift = 4;
  }
  t.grid = tiles(t.shift);
  const uint32_t step = kSoftmaxTileLanes / ((1u << t.shift) / 4);
  t.steps = (d + step - 1) / step;
  t.slots = t.steps <= 8 ? 8 : t.steps <= 10 ? 10 : 16;
  const uint32_t whole = (t.steps + 1) & ~1u, part = 2 * ((t.steps + 3) / 4), waves = softmax_tile_waves(t.slots);
  const auto bytes = [&](uint32_t pass_steps) { return softmax_tile_bytes(pass_steps * step < d ? pass_steps * step : d, t.shift); };
  const auto held = [&](uint32_t pass_steps) {
    const uint32_t fit = kCuLds / bytes(pass_steps);
    return fit < waves ? fit : waves;
  };
  const uint32_t one = held(whole), two = held(part), spare = t.shift == 6 || t.slots == 16 || sectors ? two * kCus / 5 : 0;
  t.pass_steps = t.grid > one * kCus && two > one && (t.grid <= two * kCus + spare || one <= 2) ? part : whole;
  t.lds_bytes = bytes(t.pass_steps);
  return t;
}

}  // namespace shdw

#endif  // SHADOW_AMD_CSRC_SOFTMAX_SHAPE_H_
