// A gated block of a network in one launch: normalisation, scale and ReLU of a
// feature map, the average of every plane, its sigmoid, the map times that gate,
// and the residual tail behind it (scale, sum, ReLU, plane mean).  Every step
// works inside one (n, c) plane, so a workgroup that holds whole planes in LDS
// runs the sequence with x and the residual read once and y written once; as
// operators, or as the launches the fusion pass had for the parts, the map
// crosses memory four times more.
//
// Arithmetic per element is exactly the operator sequence (parts that are absent
// are skipped, or done with a neutral operand that keeps every bit: x - 0, x * 1,
// x + (-0)).  The plane sum is fp32, front to back, or has its bits (ordered_sum.h), as Vision::Pooling
// adds; the mean at the end is fp64, rounded once after the divide.
//
// Rows of whole vectors behind BatchNorm and ReLU take whole_squeeze_gate_kernel, all others squeeze_gate_kernel.
//
// What bounds it: rows held in LDS and registers leave five to seven workgroups on a CU, with nine vectors a lane and more
// three, and two where a row takes more than 52 KB of LDS, whose loads, ordered sums and
// stores overlap each other's; the sums, dependent additions, take 2 ns each (long rows without signs
// less); and 30 to 60 vector instructions an element.  One block with its tail takes, per call: [32,512,28,28]
// (103 MB) 21.8 us (its five launches 78), [64,64,56,56] 24.6, [16,64,112,112] 32.3, [8,128,64,64] 10.9,
// [64,512,14,14] 11.5, [64,1024,7,7] 7.8, [16,64,55,55] 10.1, [16,64,111,113] 28.3.  With a lane for each row's sum that
// reads it from LDS, and one kernel for all: 25.3, 41.4, 70.1, 30.2, 11.4, 7.8, 24.2 and 70.1.
#include <hip/hip_runtime.h>

#include "../../include/shadow_hip.h"
#include "device_common.h"
#include "gate_shape.h"
#include "launch.h"
#include "libm_exact.h"
#include "ordered_sum.h"

#pragma clang fp contract(off)

namespace shdw {

// Per-row parameters, as the rows' lanes leave them in LDS.
struct alignas(16) GateRow {
  float m, d;
  double r;  // 1 / d
  float s, b, tail_s, tail_b, gate;
};

struct GateParams {
  const float *stat_mean, *stat_variance, *scale, *bias, *tail_scale, *tail_bias;
  float scale_factor, eps, plane;
  int relu;
  FastDiv channel;
};

enum { kNoResidual = 0, kOtherResidual = 1, kSameResidual = 2 };

// Waves per SIMD that the registers are held to: what a lane's vectors leave room for.  ONE as in squeeze_gate_kernel: seven
// for four vectors of one row are 72 registers; with 74, and a workgroup a CU less, 6700 rows of 784 (1675
// workgroups) take 13.5 us instead of 9.1, of 943 15.8 instead of 11.0.
constexpr int gate_waves(int slots, bool one) { return slots == 16 ? 4 : slots == 8 ? 5 : slots == 4 && one ? 7 : 6; }

// sum + row[0] + row[1] + ..., in that order, by a lane (gate_shape.h: where).
// Two sets of six vectors take turns: one is read while the other is added.  A last part of a vector reads the
// whole of it.
SHDW_DEVICE float add_in_order(float sum, const v4f* row, uint32_t cols) {
  constexpr uint32_t kSet = 6;
  const uint32_t n = cols / 4;
  uint32_t v = 0;
  const auto read = [&](v4f* q) {
#pragma unroll
    for (uint32_t k = 0; k < kSet; ++k) q[k] = row[v + k];
    v += kSet;
    __builtin_amdgcn_sched_barrier(0);  // requested here, not where they are first used
  };
  const auto add = [&](const v4f* q) {
#pragma unroll
    for (uint32_t k = 0; k < 4 * kSet; ++k) sum += q[k / 4][k % 4];
  };
  v4f a[kSet], b[kSet];
  if (n >= kSet) {
    read(a);
    while (v + 2 * kSet <= n) {
      read(b);
      add(a);
      read(a);
      add(b);
    }
    if (v + kSet <= n) {
      read(b);
      add(a);
      add(b);
    } else {
      add(a);
    }
  }
  const uint32_t left = cols - 4 * v, last = (cols - 1) / 4;
  if (left) {
#pragma unroll
    for (uint32_t k = 0; k < kSet; ++k) a[k] = row[min(v + k, last)];
#pragma unroll
    for (uint32_t k = 0; k < 4 * kSet; ++k) {
      if (k >= left) break;
      sum += a[k / 4][k % 4];
    }
  }
  return sum;
}

// sum + row[0] + row[1] + ... of 2^log2_rows rows of `cols` numbers, front to back, by a whole wave: as many lanes a
// row, a lane with 28 consecutive numbers of a chunk in registers, and the sum from lane to lane (4.8 cycles an
// addition; a lane a row that reads it from LDS takes 8, and 16 where four workgroups a CU are all there is).
// One long row without signs: side by side (ordered_sum.h).  The rows lie pitch vectors apart; of those past the last one
// the last is read.  All lanes of a row give and get its sum.
template <bool VEC>
SHDW_DEVICE float gate_walk(float sum, const v4f* tile, uint32_t pitch, uint32_t cols, uint32_t log2_rows, uint32_t nrows) {
  constexpr uint32_t kVectors = 7, kSpan = 4 * kVectors, kSideBySide = 36;  // lanes' worth: 1008 numbers
  const uint32_t lane = threadIdx.x % kWave, shift = 6 - log2_rows, per_row = 1u << shift, at = lane & (per_row - 1);
  const uint32_t nv = (cols + 3) / 4;
  const v4f* row = tile + min(lane >> shift, nrows - 1) * pitch;
  for (uint32_t v0 = 0; v0 < nv; v0 += kVectors * per_row) {
    float v[kSpan];
    const uint32_t first = v0 + at * kVectors;
    if (4 * (v0 + kVectors * per_row) <= cols) {
#pragma unroll
      for (uint32_t i = 0; i < kVectors; ++i) {
        const v4f q = row[first + i];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) v[4 * i + j] = q[j];
      }
    } else {
#pragma unroll
      for (uint32_t i = 0; i < kVectors; ++i) {
        const v4f q = row[min(first + i, nv - 1)];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)  // a sum that starts at +0 stays as it is
          v[4 * i + j] = (VEC ? first + i < nv : 4 * (first + i) + j < cols) ? q[j] : 0.f;
      }
    }
    const uint32_t turns = min(per_row, (nv - v0 + kVectors - 1) / kVectors);
    if (log2_rows == 0 && turns >= kSideBySide && __builtin_amdgcn_ballot_w64(any_sign(v) || !(sum >= 0.f)) == 0) {
      sum = wave_sum_in_order(v, sum);
      continue;
    }
    const auto turn = [&](float from) {
      sum = from;
#pragma unroll
      for (uint32_t k = 0; k < kSpan; ++k) sum += v[k];
    };
    turn(sum);
    uint32_t t = 1;
    for (; t + 4 <= turns; t += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) turn(lane_in_front(sum));
    }
    for (; t < turns; ++t) turn(lane_in_front(sum));
    sum = __shfl(sum, (lane & ~(per_row - 1)) + turns - 1);
  }
  return sum;
}

// L = 2^log2_lanes lanes share a row, so a workgroup takes 256 / L rows per turn and
// `pieces` steps of 4 L columns per row; slot i of a lane's SLOTS vectors is a piece of
// a turn, the same for all lanes, and slots from `used` on hold nothing.  Every vector is
// requested before anything else happens, and without a branch (a branch around a load has
// the compiler copy the registers of the loads before it, and wait for them): lanes with
// nothing to load take the row's or the group's last vector again.  WHOLE: the front's
// result stays in LDS; otherwise LDS holds `chunk` pieces of the rows at a time and the
// front is taken again on the way out.  ONE: one turn, a lane's vectors are of one row.  TOGETHER: the walk (gate_shape.h; both
// in one kernel, 30000 rows of 49 take 5.1 us instead of 5.0, and four vectors a lane 74 registers).  FULL: every slot
// holds something ([64,1024,7,7] with x as the residual 9.8 us, 11.2 with a test a slot; without the test where
// slots are empty [32,300,27,27] 14.8 instead of 13.9).
template <int SLOTS, bool VEC, bool WHOLE, bool ONE, bool TOGETHER, bool FULL, int RESIDUAL>
__global__ __launch_bounds__(kBlock, gate_waves(SLOTS, ONE)) void squeeze_gate_kernel(const float* x, const float* res, float* y, float* mean,
                                                              uint32_t rows, uint32_t len, uint32_t group,
                                                              uint32_t log2_lanes, uint32_t pieces, uint32_t chunk,
                                                              uint32_t pitch, uint32_t used_slots, GateParams p) {
  extern __shared__ v4f tile[];  // a chunk of the group's rows, pitch vectors apart
  __shared__ uint64_t tab[32];
  __shared__ GateRow row_params[kGateMaxRows];
  __shared__ double part[kGateMaxRows / 8][kBlock / kWave];  // rows split over the waves: at most 8
  const uint32_t used = FULL ? SLOTS : used_slots;
  const uint32_t lanes = 1u << log2_lanes, turn_rows = kBlock >> log2_lanes;
  uint32_t sub = threadIdx.x & (lanes - 1), lead = threadIdx.x >> log2_lanes;
  const uint32_t row0 = xcd_runs(blockIdx.x, gridDim.x, 2) * group;
  const uint32_t nrows = min(group, rows - row0);
  const uint32_t last = len < 4 ? 0 : len - 4;  // of a row's columns that a vector can start at

  const auto step = [&](uint32_t& k, uint32_t& turn_row) {
    if (++k == pieces && !ONE) k = 0, turn_row += turn_rows;
  };
  // addresses: one for the group, the same for all lanes, and a lane's 32-bit offset
  const auto vector = [&](const float* src, uint32_t k, uint32_t turn_row) {
    const float* from = src + static_cast<uint64_t>(row0) * len;
    const uint32_t offset = min(lead + turn_row, nrows - 1) * len + min(4 * (sub + k * lanes), last);
    if (VEC) return load4_stream(from + offset);
    if (len >= 4) return load4_stream_any(from + offset);
    const float* at = from + offset;
    return v4f{at[0], at[len > 1 ? 1 : 0], at[len > 2 ? 2 : 0], 0.f};
  };
  const auto request = [&](const float* src, v4f* to) {
    uint32_t k = 0, turn_row = 0;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      to[i] = vector(src, k, turn_row);
      step(k, turn_row);
    }
  };
  // A row's last vector was requested from where it ends inside the row: its elements to the front.
  const auto arrange = [&](v4f& v, uint32_t c) {
    if (VEC || len < 4) return;
    const uint32_t by = c - min(c, last);
    if (by & 1u) v = v4f{v[1], v[2], v[3], v[3]};
    if (by & 2u) v = v4f{v[2], v[3], v[3], v[3]};
  };
  // The rows' parameters are requested ahead of the rows (a wait for them is then no wait
  // for the rows), an absent one from an address that is there.
  const uint32_t own = row0 + min(threadIdx.x, nrows - 1), ch = own - fd_div(own, p.channel) * p.channel.d;
  const auto param = [&](const float* from) { return (from ? from : x)[ch]; };
  const float stat_mean = param(p.stat_mean), stat_variance = param(p.stat_variance), scale = param(p.scale);
  const float bias = param(p.bias), tail_scale = param(p.tail_scale), tail_bias = param(p.tail_bias);
  const uint64_t entry = libm::kExp2fTab[threadIdx.x & 31u];
  constexpr int kTurn = 4;  // vectors of the residual in flight where x keeps its registers
  v4f reg[SLOTS], other[kTurn];
  request(x, reg);
  if (threadIdx.x < nrows) {
    GateRow g{0.f, 1.f, 1.0, 1.f, -0.f, 1.f, -0.f, 0.f};
    if (p.stat_mean) {
      g.m = stat_mean * p.scale_factor;
      g.d = __builtin_sqrtf(__builtin_fabsf(stat_variance * p.scale_factor) + p.eps);
      g.r = reciprocal(g.d);
    }
    if (p.scale) g.s = scale;
    if (p.bias) g.b = bias;
    if (p.tail_scale) g.tail_s = tail_scale;
    if (p.tail_bias) g.tail_b = tail_bias;
    row_params[threadIdx.x] = g;
  }
  if (threadIdx.x < 32) tab[threadIdx.x] = entry;
  __syncthreads();

  // max(t, 0) stands for t > 0 ? t : 0: both make 0 of NaN and of -0, and t, a sum, is no signalling NaN
  const auto front = [&](v4f t, const GateRow& g) {
    if (p.stat_mean) {
#pragma unroll
      for (int j = 0; j < 4; ++j) t[j] = t[j] - g.m;
      t = quotients4(t, g.d, g.r);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      t[j] = t[j] * g.s;
      t[j] = t[j] + g.b;
    }
    if (p.relu) {
#pragma unroll
      for (int j = 0; j < 4; ++j) t[j] = __builtin_fmaxf(t[j], 0.f);
    }
    return t;
  };

  // The ordered sums: all in one wave, which issues one addition for all rows; a different
  // wave in neighbouring workgroups, so that the walks of a CU do not meet on one SIMD.
  const uint32_t log2_rows = group > 1 ? 32 - __builtin_clz(group - 1) : 0;
  const uint32_t walked = TOGETHER ? (threadIdx.x & (kWave - 1)) >> (6 - log2_rows) : threadIdx.x & (kWave - 1);
  const bool walks = threadIdx.x / kWave == ((blockIdx.x / kXcds) & 3u) && (TOGETHER || walked < nrows);
  GateRow g;
  float sum = 0.f;
  for (uint32_t k0 = 0; k0 < pieces; k0 += chunk) {
    if (!WHOLE && k0) __syncthreads();
    asm("" : "+v"(sub), "+v"(lead));
    // Read again for every chunk: of a row's parameters that stay the same the compiler takes the front of
    // all slots ahead of the chunks, and spills what does not fit (500 bytes a lane of sixteen
    // vectors: [16,64,112,112] 92 us instead of 72, [16,64,96,96] 75 instead of 54, when all blocks came here).
    if (ONE) g = row_params[min(lead, nrows - 1)];
    uint32_t k = 0, turn_row = 0;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const uint32_t r = lead + turn_row, v = sub + k * lanes;
      // for every vector where rows go in chunks: kept from piece to piece they do not fit beside the vectors
      if (!ONE && (k == 0 || !WHOLE)) g = row_params[min(r, nrows - 1)];
      if (i < used && (WHOLE || k - k0 < chunk)) {
        arrange(reg[i], 4 * v);
        const v4f t = front(reg[i], g);
        if (r < nrows && 4 * v < len) tile[r * pitch + v - k0 * lanes] = t;
      }
      step(k, turn_row);
    }
    // the residual travels while the rows are summed
    if (RESIDUAL == kOtherResidual && WHOLE) request(res, reg);
    __syncthreads();
    if (walks) {
      const uint32_t cols = WHOLE ? len : min(len - 4 * k0 * lanes, 4 * chunk * lanes);
      __builtin_amdgcn_s_setprio(3);  // nothing else of the workgroup moves meanwhile: 26.9 -> 26.4 us on [32,512,28,28]
      if (TOGETHER) sum = gate_walk<VEC>(sum, tile, pitch, cols, log2_rows, nrows);
      else sum = add_in_order(sum, tile + walked * pitch, cols);
      __builtin_amdgcn_s_setprio(0);
    }
    if (WHOLE) break;
  }
  if (walks && walked < nrows) row_params[walked].gate = libm::exact_sigmoidf(sum / p.plane, tab);
  __syncthreads();

  asm("" : "+v"(sub), "+v"(lead));  // the slots' offsets are taken again instead of kept
  if (ONE) g = row_params[min(lead, nrows - 1)];
  double total = 0.0;
  uint32_t k = 0, turn_row = 0;
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    if (i >= used) continue;
    const uint32_t r = lead + turn_row, v = sub + k * lanes, c = 4 * v;
    if (!ONE && (k == 0 || !WHOLE)) g = row_params[min(r, nrows - 1)];
    v4f t = WHOLE ? tile[min(r, nrows - 1) * pitch + min(v, pitch - 1)] : front(reg[i], g);
    if (RESIDUAL == kOtherResidual && !WHOLE && i % kTurn == 0) {
      uint32_t k_ahead = k, turn_ahead = turn_row;
#pragma unroll
      for (int n = 0; n < kTurn; ++n) {
        other[n] = vector(res, k_ahead, turn_ahead);
        step(k_ahead, turn_ahead);
      }
    }
    v4f q = RESIDUAL == kOtherResidual && !WHOLE ? other[i % kTurn] : reg[i];
    if (RESIDUAL == kOtherResidual) arrange(q, c);
    // Eltwise SUM with unit coefficients is Set(0), then y += 1 * input, input by input: behind
    // the ReLU neither the 0 in front nor which input comes first can be told from t + q.
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      t[j] = t[j] * g.gate;
      if (RESIDUAL != kNoResidual) {
        t[j] = t[j] * g.tail_s;
        t[j] = t[j] + g.tail_b;
        t[j] = __builtin_fmaxf(t[j] + q[j], 0.f);
      }
    }
    if (r < nrows && c < len) {
      float* to = y + static_cast<uint64_t>(row0) * len;
      const uint32_t offset = r * len + c;
      if (VEC) {
        store4_stream(to + offset, t);
      } else if (c + 4 <= len) {
        store4_stream_any(to + offset, t);
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (c + j < len) to[offset + j] = t[j];
      }
    }
    if (RESIDUAL != kNoResidual && mean) {
      const auto add = [&](int j) { total += static_cast<double>(t[j]); };
      if (k + 1 < pieces || VEC) {
        if (k + 1 < pieces || c < len) add(0), add(1), add(2), add(3);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (c + j < len) add(j);
      }
      if (k + 1 == pieces) {  // the row is complete: every lane of the wave is here
        total += dpp_f64<kDppXor1>(total);
        total += dpp_f64<kDppXor2>(total);
        total += dpp_f64<kDppHalfMirror>(total);
        total += dpp_f64<kDppMirror>(total);
        if (log2_lanes > 4) total += __shfl_xor(total, 16, kWave);
        if (log2_lanes > 5) total += __shfl_xor(total, 32, kWave);
        if (log2_lanes > 6) {
          if ((threadIdx.x & (kWave - 1)) == 0 && r < nrows) part[r][threadIdx.x / kWave] = total;
        } else if (sub == 0 && r < nrows) {
          mean[row0 + r] = static_cast<float>(total / static_cast<double>(static_cast<int>(len)));
        }
        total = 0.0;
      }
    }
    step(k, turn_row);
  }
  if (RESIDUAL != kNoResidual && mean && log2_lanes > 6) {
    __syncthreads();
    if (threadIdx.x < nrows) {
      double sum = 0.0;
      for (int w = 0; w < kBlock / kWave; ++w) sum += part[threadIdx.x][w];
      mean[row0 + threadIdx.x] = static_cast<float>(sum / static_cast<double>(static_cast<int>(len)));
    }
  }
}

// Rows of whole, aligned vectors that lie in LDS whole, with BatchNorm and ReLU in front and a residual behind:
// PIECES vectors of one row a lane.  Where a vector lies is worked out once for a lane, or is uniform, so that an element
// costs its arithmetic and little else, and the walk reads LDS ahead of its additions.  Against squeeze_gate_kernel, with
// 47 vector instructions an element and a lane of a wave for each row's walk: [32,512,28,28] 25.4 -> 22.6 us, [64,64,56,56]
// 41.4 -> 24.8, [8,128,64,64] 29.9 -> 10.8, [16,256,48,48] 32.6 -> 21.9, [16,64,40,40] 11.2 -> 8.8.
// Seven workgroups a CU with up to four vectors a lane: 14000 rows of 448 12.5 us as six, 8.5.
constexpr int whole_waves(int pieces) { return pieces <= 4 ? 7 : pieces <= 8 ? 5 : 3; }

template <int PIECES, int RESIDUAL>
__global__ __launch_bounds__(kBlock, whole_waves(PIECES)) void whole_squeeze_gate_kernel(
    const float* x, const float* res, float* y, float* mean, uint32_t rows, uint32_t len, uint32_t log2_lanes, uint32_t pitch,
    GateParams p) {
  extern __shared__ v4f tile[];  // the group's rows, pitch vectors apart
  __shared__ uint64_t tab[32];
  __shared__ GateRow row_params[kBlock / 16];
  __shared__ double part[kBlock / kWave];
  const uint32_t lanes = 1u << log2_lanes, group = kBlock >> log2_lanes;
  const uint32_t sub = threadIdx.x & (lanes - 1), lead = threadIdx.x >> log2_lanes;
  const uint32_t row0 = xcd_runs(blockIdx.x, gridDim.x, 2) * group;
  const uint32_t nrows = min(group, rows - row0), nv = len / 4, row = min(lead, nrows - 1);
  const bool live = lead < nrows, whole = sub + (PIECES - 1) * lanes < nv;
  const uint64_t start = static_cast<uint64_t>(row0) * len;
  // Bytes from the group's first element: a lane's offset, which a piece's uniform part is added to, and the last
  // piece's, where lanes past the row's end take its last vector.
  const uint32_t at = (row * nv + sub) * static_cast<uint32_t>(sizeof(v4f));
  const uint32_t at_last = (row * nv + min(sub + (PIECES - 1) * lanes, nv - 1)) * static_cast<uint32_t>(sizeof(v4f));
  const auto place = [&](int k) { return k + 1 < PIECES ? static_cast<size_t>(k * lanes) * sizeof(v4f) + at : static_cast<size_t>(at_last); };
  const auto request = [&](const float* src, v4f (&to)[PIECES]) {
    const char* from = reinterpret_cast<const char*>(src + start);
#pragma unroll
    for (int k = 0; k < PIECES; ++k) to[k] = load4_stream(reinterpret_cast<const float*>(from + place(k)));
  };
  const uint32_t own = row0 + min(threadIdx.x, nrows - 1), ch = own - fd_div(own, p.channel) * p.channel.d;
  const auto param = [&](const float* from) { return (from ? from : x)[ch]; };  // an absent one from an address that is there
  const float stat_mean = p.stat_mean[ch], stat_variance = p.stat_variance[ch], scale = param(p.scale);
  const float bias = param(p.bias), tail_scale = param(p.tail_scale), tail_bias = param(p.tail_bias);
  const uint64_t entry = libm::kExp2fTab[threadIdx.x & 31u];
  v4f reg[PIECES];
  request(x, reg);
  if (threadIdx.x < nrows) {
    GateRow g{stat_mean * p.scale_factor, 1.f, 1.0, 1.f, -0.f, 1.f, -0.f, 0.f};
    g.d = __builtin_sqrtf(__builtin_fabsf(stat_variance * p.scale_factor) + p.eps);
    g.r = reciprocal(g.d);
    if (p.scale) g.s = scale;
    if (p.bias) g.b = bias;
    if (p.tail_scale) g.tail_s = tail_scale;
    if (p.tail_bias) g.tail_b = tail_bias;
    row_params[threadIdx.x] = g;
  }
  if (threadIdx.x < 32) tab[threadIdx.x] = entry;
  __syncthreads();

  v4f* const mine = tile + lead * pitch + sub;
  {
    const GateRow g = row_params[row];
#pragma unroll
    for (int k = 0; k < PIECES; ++k) {
      v4f t = reg[k];
#pragma unroll
      for (int j = 0; j < 4; ++j) t[j] = t[j] - g.m;
      t = quotients4(t, g.d, g.r);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        t[j] = t[j] * g.s;
        t[j] = __builtin_fmaxf(t[j] + g.b, 0.f);  // as in squeeze_gate_kernel
      }
      if (live && (k + 1 < PIECES || whole)) mine[k * lanes] = t;
    }
  }
  // the residual travels while the rows are summed
  if (RESIDUAL == kOtherResidual) request(res, reg);
  __syncthreads();
  if (threadIdx.x / kWave == ((blockIdx.x / kXcds) & 3u)) {  // as in squeeze_gate_kernel
    __builtin_amdgcn_s_setprio(3);
    const uint32_t log2_rows = 8 - log2_lanes, walked = (threadIdx.x & (kWave - 1)) >> (6 - log2_rows);
    const float sum = gate_walk<true>(0.f, tile, pitch, len, log2_rows, nrows);
    if (walked < nrows) row_params[walked].gate = libm::exact_sigmoidf(sum / p.plane, tab);  // all lanes of a row the same
    __builtin_amdgcn_s_setprio(0);
  }
  __syncthreads();

  const float gate = row_params[row].gate, tail_s = row_params[row].tail_s, tail_b = row_params[row].tail_b;
  char* const to = reinterpret_cast<char*>(y + start);
  double total = 0.0;
  const auto finish = [&](int k) {
    v4f t = mine[k * lanes];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      t[j] = t[j] * gate;
      t[j] = t[j] * tail_s;
      t[j] = t[j] + tail_b;
      t[j] = __builtin_fmaxf(t[j] + reg[k][j], 0.f);  // as in squeeze_gate_kernel
    }
    store4_stream(reinterpret_cast<float*>(to + place(k)), t);
    if (mean) {
#pragma unroll
      for (int j = 0; j < 4; ++j) total += static_cast<double>(t[j]);
    }
  };
  if (live) {
#pragma unroll
    for (int k = 0; k + 1 < PIECES; ++k) finish(k);
    if (whole) finish(PIECES - 1);
  }
  if (!mean) return;
  total += dpp_f64<kDppXor1>(total);
  total += dpp_f64<kDppXor2>(total);
  total += dpp_f64<kDppHalfMirror>(total);
  total += dpp_f64<kDppMirror>(total);
  if (log2_lanes > 4) total += __shfl_xor(total, 16, kWave);
  if (log2_lanes > 5) total += __shfl_xor(total, 32, kWave);
  if (log2_lanes > 6) {  // the workgroup's one row
    if ((threadIdx.x & (kWave - 1)) == 0) part[threadIdx.x / kWave] = total;
    __syncthreads();
    total = ((part[0] + part[1]) + part[2]) + part[3];
  }
  if (sub == 0 && live) mean[row0 + lead] = static_cast<float>(total / static_cast<double>(static_cast<int>(len)));
}

}  // namespace shdw

using namespace shdw;

namespace {

uint32_t used_slots(const GateShape& g) { return (g.group << g.log2_lanes) / kBlock * g.pieces; }

template <int SLOTS, bool VEC, bool WHOLE, bool ONE, bool TOGETHER>
void launch_gate_form(const GateShape& g, uint32_t rows, uint32_t len, const float* x, const float* res, float* y, float* mean,
                      const GateParams& p, hipStream_t st) {
  const uint32_t grid = (rows + g.group - 1) / g.group, used = used_slots(g);
  const size_t lds = static_cast<size_t>(g.group) * g.pitch * sizeof(v4f);
  const auto launch = [&](auto kernel) {
    kernel<<<grid, kBlock, lds, st>>>(x, res, y, mean, rows, len, g.group, g.log2_lanes, g.pieces, g.chunk, g.pitch, used, p);
  };
#define SHDW_LAUNCH(R)                                                                        \
  if (used == SLOTS) launch(squeeze_gate_kernel<SLOTS, VEC, WHOLE, ONE, TOGETHER, true, R>);  \
  else launch(squeeze_gate_kernel<SLOTS, VEC, WHOLE, ONE, TOGETHER, SLOTS == 1, R>)
  if (!res) {
    SHDW_LAUNCH(kNoResidual);
  } else if (res == x) {
    SHDW_LAUNCH(kSameResidual);
  } else {
    SHDW_LAUNCH(kOtherResidual);
  }
#undef SHDW_LAUNCH
}

template <int SLOTS, bool VEC, bool WHOLE, bool ONE>
void launch_gate(const GateShape& g, uint32_t rows, uint32_t len, const float* x, const float* res, float* y, float* mean,
                 const GateParams& p, hipStream_t st) {
  constexpr int kWalks = gate_walks(SLOTS, WHOLE, ONE);
  if constexpr (kWalks == (kGateLaneARow | kGateTogether)) {
    if (g.walk == kGateTogether) launch_gate_form<SLOTS, VEC, WHOLE, ONE, true>(g, rows, len, x, res, y, mean, p, st);
    else launch_gate_form<SLOTS, VEC, WHOLE, ONE, false>(g, rows, len, x, res, y, mean, p, st);
  } else {
    launch_gate_form<SLOTS, VEC, WHOLE, ONE, kWalks == kGateTogether>(g, rows, len, x, res, y, mean, p, st);
  }
}

// Four vectors a lane of every row and the rows' odd pitch stay below the tile: never cut.
static_assert((4 * kBlock + kGateMaxRows) * sizeof(v4f) <= kGateTileBytes, "rows of up to four vectors a lane lie whole in LDS");
static_assert(kBlock == kGateLanes && sizeof(v4f) == kGateVectorBytes, "gate_shape.h counts in these");

template <int SLOTS, bool VEC, bool ONE>
void launch_gate(const GateShape& g, uint32_t rows, uint32_t len, const float* x, const float* res, float* y, float* mean,
                 const GateParams& p, hipStream_t st) {
  if (g.chunk == g.pieces) launch_gate<SLOTS, VEC, true, ONE>(g, rows, len, x, res, y, mean, p, st);
  else launch_gate<SLOTS, VEC, false, ONE>(g, rows, len, x, res, y, mean, p, st);
}

template <bool VEC>
void launch_gate(const GateShape& g, uint32_t rows, uint32_t len, const float* x, const float* res, float* y, float* mean,
                 const GateParams& p, hipStream_t st) {
  const bool one = used_slots(g) == g.pieces;  // one and sixteen slots are of one turn in any case
  switch (g.slots) {
    case 1: launch_gate<1, VEC, true, true>(g, rows, len, x, res, y, mean, p, st); break;
    case 4:
      if (one) launch_gate<4, VEC, true, true>(g, rows, len, x, res, y, mean, p, st);
      else launch_gate<4, VEC, true, false>(g, rows, len, x, res, y, mean, p, st);
      break;
    case 8:
      if (one) launch_gate<8, VEC, true>(g, rows, len, x, res, y, mean, p, st);
      else launch_gate<8, VEC, false>(g, rows, len, x, res, y, mean, p, st);
      break;
    default: launch_gate<16, VEC, true>(g, rows, len, x, res, y, mean, p, st);
  }
}

template <int PIECES>
void launch_gate_whole(const GateWhole& g, uint32_t rows, uint32_t len, const float* x, const float* res, float* y, float* mean,
                       const GateParams& p, hipStream_t st) {
  const uint32_t grid = (rows + g.group - 1) / g.group;
  const size_t lds = static_cast<size_t>(g.group) * g.pitch * sizeof(v4f);
  const auto launch = [&](auto kernel) { kernel<<<grid, kBlock, lds, st>>>(x, res, y, mean, rows, len, g.log2_lanes, g.pitch, p); };
  if (res == x) launch(whole_squeeze_gate_kernel<PIECES, kSameResidual>);
  else launch(whole_squeeze_gate_kernel<PIECES, kOtherResidual>);
}

static_assert(kGateWholePieces == 15, "the switch covers up to 15 vectors a lane");

void launch_gate_whole(const GateWhole& g, uint32_t rows, uint32_t len, const float* x, const float* res, float* y, float* mean,
                       const GateParams& p, hipStream_t st) {
  switch (g.pieces) {
#define SHDW_PIECES(P) case P: launch_gate_whole<P>(g, rows, len, x, res, y, mean, p, st); break;
    SHDW_PIECES(1) SHDW_PIECES(2) SHDW_PIECES(3) SHDW_PIECES(4) SHDW_PIECES(5) SHDW_PIECES(6) SHDW_PIECES(7) SHDW_PIECES(8)
    SHDW_PIECES(9) SHDW_PIECES(10) SHDW_PIECES(11) SHDW_PIECES(12) SHDW_PIECES(13) SHDW_PIECES(14) SHDW_PIECES(15)
#undef SHDW_PIECES
  }
}

}  // namespace

extern "C" int shdw_hip_squeeze_gate(int n, int channel, int inner_num, const float* x, const float* stat_mean,
                                     const float* stat_variance, float scale_factor, float eps, const float* scale,
                                     const float* bias, int relu, const float* tail_scale, const float* tail_bias,
                                     const float* residual, int residual_first, float* y, float* mean, void* stream) {
  if (n < 0 || channel < 1 || inner_num < 1 || !x || !y || !stat_mean != !stat_variance) return SHDW_E_INVALID_ARGUMENT;
  if (residual ? !tail_scale && !tail_bias : tail_scale || tail_bias || mean) return SHDW_E_INVALID_ARGUMENT;
  if (n % inner_num != 0) return SHDW_E_INVALID_ARGUMENT;
  if (inner_num > SHDW_SQUEEZE_GATE_MAX_INNER) return SHDW_E_UNSUPPORTED;
  if (n == 0) return SHDW_OK;
  const uint32_t rows = static_cast<uint32_t>(n / inner_num), len = static_cast<uint32_t>(inner_num);
  const GateParams p{stat_mean, stat_variance, scale, bias, tail_scale, tail_bias, scale_factor, eps,
                     static_cast<float>(inner_num), relu, make_fastdiv(static_cast<uint32_t>(channel))};
  const bool vec = len % 4 == 0 && aligned16(x) && aligned16(y) && (!residual || aligned16(residual));
  if (GateWhole w; gate_takes_whole(vec, stat_mean != nullptr, relu != 0, residual != nullptr, rows, len, &w)) {
    launch_gate_whole(w, rows, len, x, residual, y, mean, p, static_cast<hipStream_t>(stream));
    return launch_status();
  }
  const GateShape g = gate_shape(rows, len);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (vec) launch_gate<true>(g, rows, len, x, residual, y, mean, p, st);
  else launch_gate<false>(g, rows, len, x, residual, y, mean, p, st);
  return launch_status();
}
