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
// x + (-0)).  The plane sum is fp32, front to back, by one lane, as Vision::Pooling
// adds; the mean at the end is fp64, rounded once after the divide.
//
// What bounds it: 25 KB of LDS a workgroup leave six on a CU, whose loads, ordered
// sums (784 dependent additions: 3 us) and stores overlap each other's.  A block on
// [32,512,28,28] takes 31 us (103 MB) where its five launches took 78; two such
// blocks behind a text model 239 -> 135 us a call, four on [1,256,14,14] 170 -> 108;
// four on [16,64,56,56] 241 -> 120, on [64,1024,7,7] 155 -> 77.  Long planes keep one
// row per workgroup and few workgroups per CU: four blocks on [16,64,112,112] 711 ->
// 501, on [64,64,112,112] level (1376, 1386).
#include <hip/hip_runtime.h>

#include "../../include/shadow_hip.h"
#include "device_common.h"
#include "launch.h"
#include "libm_exact.h"

#pragma clang fp contract(off)

namespace shdw {

// Per-row parameters, as the rows' lanes leave them in LDS.
struct GateRow {
  float m, d, s, b, tail_s, tail_b;
};

struct GateParams {
  const float *stat_mean, *stat_variance, *scale, *bias, *tail_scale, *tail_bias;
  float scale_factor, eps, plane;
  int relu, residual_first;
  FastDiv channel;
};

enum { kNoResidual = 0, kOtherResidual = 1, kSameResidual = 2 };

constexpr uint32_t kGateMaxRows = 64;  // per workgroup: a lane of one wave each in the ordered sum

// L = 2^log2_lanes lanes share a row, so a workgroup takes 256 / L rows per turn and
// `pieces` steps of 4 L columns per row; SLOTS >= turns * pieces vectors per lane, all
// requested before anything else happens.
template <int SLOTS, bool VEC, int RESIDUAL>
__global__ __launch_bounds__(kBlock) void squeeze_gate_kernel(const float* x, const float* res, float* y, float* mean,
                                                              uint32_t rows, uint32_t len, uint32_t group,
                                                              uint32_t log2_lanes, uint32_t pieces, uint32_t pitch,
                                                              GateParams p) {
  extern __shared__ __align__(16) float tile[];  // group rows of pitch floats
  __shared__ uint64_t tab[32];
  __shared__ GateRow row_params[kGateMaxRows];
  __shared__ float gate[kGateMaxRows];
  __shared__ double part[kGateMaxRows / 8][kBlock / kWave];  // rows split over the waves: at most 8
  const uint32_t lanes = 1u << log2_lanes, turn_rows = kBlock >> log2_lanes;
  const uint32_t sub = threadIdx.x & (lanes - 1), lead = threadIdx.x >> log2_lanes;
  const uint32_t row0 = xcd_runs(blockIdx.x, gridDim.x, 2) * group;
  const uint32_t nrows = min(group, rows - row0);

  v4f reg[SLOTS], other[RESIDUAL == kOtherResidual ? SLOTS : 1];
  auto request = [&](const float* src, v4f* to) {
    uint32_t r = lead, c = 4 * sub, k = 0;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      if (r < nrows && c < len) {
        const float* at = src + static_cast<uint64_t>(row0 + r) * len + c;
        if (VEC) {
          to[i] = load4_stream(at);
        } else if (c + 4 <= len) {
          to[i] = load4_stream_any(at);
        } else {
          to[i] = v4f{at[0], c + 1 < len ? at[1] : 0.f, c + 2 < len ? at[2] : 0.f, 0.f};
        }
      }
      if (++k == pieces) k = 0, c = 4 * sub, r += turn_rows;
      else c += 4 * lanes;
    }
  };
  request(x, reg);
  if (RESIDUAL == kOtherResidual) request(res, other);

  if (threadIdx.x < nrows) {
    const uint32_t row = row0 + threadIdx.x, c = row - fd_div(row, p.channel) * p.channel.d;
    GateRow g{0.f, 1.f, 1.f, -0.f, 1.f, -0.f};
    if (p.stat_mean) {
      g.m = p.stat_mean[c] * p.scale_factor;
      g.d = __builtin_sqrtf(__builtin_fabsf(p.stat_variance[c] * p.scale_factor) + p.eps);
    }
    if (p.scale) g.s = p.scale[c];
    if (p.bias) g.b = p.bias[c];
    if (p.tail_scale) g.tail_s = p.tail_scale[c];
    if (p.tail_bias) g.tail_b = p.tail_bias[c];
    row_params[threadIdx.x] = g;
  }
  if (threadIdx.x >= kBlock - 32) tab[threadIdx.x - (kBlock - 32)] = libm::kExp2fTab[threadIdx.x - (kBlock - 32)];
  __syncthreads();

  {
    uint32_t r = lead, c = 4 * sub, k = 0;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      if (r < nrows && c < len) {
        const GateRow g = row_params[r];
        v4f t = reg[i];
        if (p.stat_mean) {
#pragma unroll
          for (int j = 0; j < 4; ++j) t[j] = (t[j] - g.m) / g.d;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          t[j] = t[j] * g.s;
          t[j] = t[j] + g.b;
          if (p.relu) t[j] = t[j] > 0 ? t[j] : 0;
        }
        *reinterpret_cast<v4f*>(tile + r * pitch + c) = t;
      }
      if (++k == pieces) k = 0, c = 4 * sub, r += turn_rows;
      else c += 4 * lanes;
    }
  }
  __syncthreads();

  // The ordered sums, a lane per row: all in one wave, which issues one addition for
  // all rows; a different wave in neighbouring workgroups, so that the walks of a CU
  // do not meet on one SIMD.
  if (threadIdx.x / kWave == ((blockIdx.x / kXcds) & 3u) && (threadIdx.x & (kWave - 1)) < nrows) {
    const uint32_t r = threadIdx.x & (kWave - 1);
    const float* mine = tile + r * pitch;
    constexpr int kAhead = 16, kStep = 4 * kAhead;
    float sum = 0.f;
    uint32_t c = 0;
    for (; c + kStep <= len; c += kStep) {
      v4f q[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) q[k] = *reinterpret_cast<const v4f*>(mine + c + 4 * k);
#pragma unroll
      for (int k = 0; k < kStep; ++k) sum += q[k / 4][k % 4];
    }
    for (; c < len; ++c) sum += mine[c];
    gate[r] = libm::exact_sigmoidf(sum / p.plane, tab);
  }
  __syncthreads();

  double total = 0.0;
  uint32_t r = lead, c = 4 * sub, k = 0;
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    if (r < nrows && c < len) {
      const float g = gate[r], s = row_params[r].tail_s, b = row_params[r].tail_b;
      v4f t = *reinterpret_cast<const v4f*>(tile + r * pitch + c);
      const v4f q = RESIDUAL == kOtherResidual ? other[i] : reg[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        t[j] = t[j] * g;
        if (RESIDUAL != kNoResidual) {
          t[j] = t[j] * s;
          t[j] = t[j] + b;
          // Eltwise SUM with unit coefficients: Set(0), then y += 1 * input, input by input
          float u = 0.0f + (p.residual_first ? q[j] : t[j]);
          u = u + (p.residual_first ? t[j] : q[j]);
          t[j] = u > 0 ? u : 0;
          if (VEC || c + j < len) total += static_cast<double>(t[j]);
        }
      }
      float* at = y + static_cast<uint64_t>(row0 + r) * len + c;
      if (VEC) {
        store4_stream(at, t);
      } else if (c + 4 <= len) {
        store4_stream_any(at, t);
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (c + j < len) at[j] = t[j];
      }
    }
    if (++k == pieces) {
      if (RESIDUAL != kNoResidual && mean) {  // the row is complete: every lane of the wave is here
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
      k = 0, c = 4 * sub, r += turn_rows;
    } else {
      c += 4 * lanes;
    }
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

// How a shape is cut.
struct GateShape {
  uint32_t log2_lanes, pieces, group, pitch;
  int slots;
};

// Lanes per row: as many as a row has vectors, up to a wave; the whole workgroup where
// a wave would take more than eight steps over a row, and where there are so few rows
// that a row per wave would leave CUs idle.  Rows per workgroup: what eight vectors per
// lane hold, fewer while that leaves under 1024 workgroups (four per CU).
inline GateShape gate_shape(uint32_t rows, uint32_t len) {
  const uint32_t nv = (len + 3) / 4;
  GateShape g{};
  g.log2_lanes = nv <= 16 ? 4 : nv <= 32 ? 5 : nv <= 512 ? 6 : 8;
  if (nv > 16 && rows < 1024) g.log2_lanes = 8;
  const uint32_t lanes = 1u << g.log2_lanes, turn_rows = kBlock >> g.log2_lanes;
  g.pieces = (nv + lanes - 1) / lanes;
  g.slots = g.pieces <= 8 ? 8 : 16;
  uint32_t turns = static_cast<uint32_t>(g.slots) / g.pieces;
  if (turns * turn_rows > kGateMaxRows) turns = kGateMaxRows / turn_rows;
  while (turns > 1 && (rows + turns * turn_rows - 1) / (turns * turn_rows) < 1024u) --turns;
  g.group = turns * turn_rows;
  g.pitch = 4 * (nv | 1u);  // an odd number of 128-bit pieces: the summing lanes meet different banks
  return g;
}

}  // namespace shdw

using namespace shdw;

namespace {

template <int SLOTS, bool VEC>
void launch_gate(const GateShape& g, uint32_t rows, uint32_t len, const float* x, const float* res, float* y, float* mean,
                 const GateParams& p, hipStream_t st) {
  const uint32_t grid = (rows + g.group - 1) / g.group;
  const size_t lds = static_cast<size_t>(g.group) * g.pitch * sizeof(float);
#define SHDW_LAUNCH(R)                                                                                          \
  squeeze_gate_kernel<SLOTS, VEC, R><<<grid, kBlock, lds, st>>>(x, res, y, mean, rows, len, g.group, g.log2_lanes, \
                                                                g.pieces, g.pitch, p)
  if (!res) SHDW_LAUNCH(kNoResidual);
  else if (res == x) SHDW_LAUNCH(kSameResidual);
  else SHDW_LAUNCH(kOtherResidual);
#undef SHDW_LAUNCH
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
                     static_cast<float>(inner_num), relu, residual_first, make_fastdiv(static_cast<uint32_t>(channel))};
  const bool vec = len % 4 == 0 && aligned16(x) && aligned16(y) && (!residual || aligned16(residual));
  const GateShape g = gate_shape(rows, len);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (g.slots == 8) {
    if (vec) launch_gate<8, true>(g, rows, len, x, residual, y, mean, p, st);
    else launch_gate<8, false>(g, rows, len, x, residual, y, mean, p, st);
  } else {
    if (vec) launch_gate<16, true>(g, rows, len, x, residual, y, mean, p, st);
    else launch_gate<16, false>(g, rows, len, x, residual, y, mean, p, st);
  }
  return launch_status();
}
