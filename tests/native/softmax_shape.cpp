// softmax_tiles (shadow_amd/csrc/softmax_shape.h) for tests/test_softmax_shape_cpu.py.
#include "../../shadow_amd/csrc/softmax_shape.h"

extern "C" void softmax_tiles(int outer, int dim, int inner, int sectors, unsigned* out) {
  const shdw::SoftmaxTiles t = shdw::softmax_tiles(outer, dim, inner, sectors != 0);
  const unsigned all[] = {static_cast<unsigned>(t.shift), static_cast<unsigned>(t.slots), t.grid, t.whole() ? 1u : 2u, t.lds_bytes};
  for (int k = 0; k < 5; ++k) out[k] = all[k];
}

// The first length of columns in [65, 1024] whose cut breaks what the kernel relies on, or 0.
extern "C" int softmax_tiles_scan(int outer, int inner, int sectors) {
  for (int dim = 65; dim <= 1024; ++dim) {
    const shdw::SoftmaxTiles t = shdw::softmax_tiles(outer, dim, inner, sectors != 0);
    const unsigned d = static_cast<unsigned>(dim), step = 1024u >> t.shift, rows = t.pass_steps * step < d ? t.pass_steps * step : d;
    const bool ok = t.shift >= 4 && t.shift <= 6 && (t.slots == 8 || t.slots == 10 || t.slots == 16) &&
                    t.grid == static_cast<unsigned>(outer) * ((static_cast<unsigned>(inner) + (1u << t.shift) - 1) >> t.shift) &&
                    t.steps * step >= d && t.steps <= static_cast<unsigned>(t.slots) &&                     // every row has a vector
                    t.pass_steps >= 2 && t.pass_steps % 2 == 0 && (t.whole() || 2 * t.pass_steps >= t.steps) &&  // one pass or two
                    t.lds_bytes == (rows << t.shift) * 4u + 256u + (16u << t.shift) && t.lds_bytes <= 68000u &&
                    (t.shift > 4 || t.slots > 8 || t.whole());                                              // the forms that are launched
    if (!ok) return dim;
  }
  return 0;
}
