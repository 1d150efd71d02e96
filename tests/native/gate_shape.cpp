// gate_shape (shadow_amd/csrc/gate_shape.h) for tests/test_gate_shape_cpu.py.
#include "../../shadow_amd/csrc/gate_shape.h"

extern "C" void gate_shape(unsigned rows, unsigned len, unsigned* out) {
  const shdw::GateShape g = shdw::gate_shape(rows, len);
  const unsigned all[] = {g.log2_lanes, g.pieces, g.group, g.chunk, g.pitch, static_cast<unsigned>(g.slots),
                          g.walk == shdw::kGateTogether};
  for (int k = 0; k < 7; ++k) out[k] = all[k];
}

// The first length in [1, last] whose cut breaks what the kernel relies on, or 0.
extern "C" unsigned gate_shape_scan(unsigned rows, unsigned last) {
  for (unsigned len = 1; len <= last; ++len) {
    const shdw::GateShape g = shdw::gate_shape(rows, len);
    const int walks = shdw::gate_walks(g.slots, g.chunk == g.pieces, ((g.group << g.log2_lanes) / 256u) == 1u);
    if ((g.walk & walks) == 0 || (g.walk == shdw::kGateTogether && g.group > 16)) return len;  // a wave walks sixteen rows at most
    const unsigned nv = (len + 3) / 4, lanes = 1u << g.log2_lanes, turn_rows = 256u >> g.log2_lanes;
    const unsigned turns = g.group / turn_rows, kept = g.chunk * lanes < nv ? g.chunk * lanes : nv;
    const bool ok = (g.slots == 1 || g.slots == 4 || g.slots == 8 || g.slots == 16) &&
                    turns >= 1 && g.group == turns * turn_rows && g.group <= shdw::kGateMaxRows &&
                    turns * g.pieces <= static_cast<unsigned>(g.slots) &&             // every vector has a slot
                    g.pieces * lanes >= nv && g.chunk >= 1 && g.chunk <= g.pieces &&  // every column a piece
                    g.pitch >= kept && g.pitch % 2 == 1 &&
                    g.group * g.pitch * 16u + 2560u <= 65536u &&                      // LDS of a workgroup
                    (g.slots >= 8 || g.chunk == g.pieces) &&                          // the forms that are launched
                    (g.log2_lanes <= 6 || g.group <= shdw::kGateMaxRows / 8);         // partial sums of a row's waves
    if (!ok) return len;
  }
  return 0;
}

extern "C" int gate_whole(unsigned rows, unsigned len, unsigned* out) {
  shdw::GateWhole g{};
  if (!shdw::gate_whole(rows, len, &g)) return 0;
  out[0] = 1u << g.log2_lanes, out[1] = g.pieces, out[2] = g.group;
  return 1;
}

// Whether a call with these parts and aligned operands is whole_squeeze_gate_kernel's.
extern "C" int gate_takes_whole(unsigned rows, unsigned len, int stats, int relu, int residual) {
  shdw::GateWhole g{};
  return shdw::gate_takes_whole(len % 4 == 0, stats != 0, relu != 0, residual != 0, rows, len, &g);
}

// The same for gate_whole, lengths of whole vectors.
extern "C" unsigned gate_whole_scan(unsigned rows, unsigned last) {
  for (unsigned len = 4; len <= last; len += 4) {
    const shdw::GateShape other = shdw::gate_shape(rows, len);
    if (other.chunk != other.pieces && other.group > 16) return len;  // rows in chunks: one wave walks all of them together
    shdw::GateWhole g{};
    if (!shdw::gate_whole(rows, len, &g)) continue;
    const unsigned nv = len / 4, lanes = 1u << g.log2_lanes;
    const bool ok = g.log2_lanes >= 4 && g.log2_lanes <= 8 && g.log2_lanes != 7 && g.group * lanes == 256 && g.group <= 16 &&
                    g.pieces >= 1 && g.pieces <= shdw::kGateWholePieces && (g.pieces - 1) * lanes < nv && nv <= g.pieces * lanes &&
                    g.pitch >= nv && g.pitch % 2 == 1 && g.group * g.pitch * 16u + 1280u <= 65536u;
    if (!ok) return len;
  }
  return 0;
}
