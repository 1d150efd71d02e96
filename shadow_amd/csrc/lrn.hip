// LRN across channels (shadow/operators/kernels/lrn.cpp:9-60, lrn.cu).
//
// The reference walks the channels of one (batch, h, w) position with a running
// fp32 sum of squares -- the entering square is added, then the one that leaves
// the window is subtracted -- writes scale = k + sum * (alpha / size) into a
// scratch blob, and multiplies x by powf(scale, -beta) in a second pass.  The
// order of the additions and subtractions fixes the bits, so the walk stays: one
// lane per position, channel after channel.  What goes is the scratch blob and
// the second pass: the window's values wait in registers (windows of up to seven
// channels) or in LDS (a column of `size` floats per lane, no two lanes share a
// bank row), the centre of the window is multiplied as soon as its scale is
// known, x is read once and y written once.  Neighbouring lanes hold neighbouring
// positions, so every load and store of a wave is one run of 256 bytes.  y may be x: a lane
// has read every channel of a round, and all before it, when it writes the channels the
// round finishes, which lie behind them.
#include <hip/hip_runtime.h>

#include <climits>

#include "../../include/shadow_hip.h"
#include "device_common.h"
#include "launch.h"
#include "libm_exact.h"

#pragma clang fp contract(off)

namespace shdw {

// Windows of up to 63 channels: 63 KB of LDS for the 256 lanes of a workgroup, beside the tables.
constexpr int kLrnMaxSize = 63;

// Channels a lane takes per round: their loads go out together, the sum walks
// through them one by one, and only then come the powers, which do not depend on
// one another -- eight of them side by side, in their branch-free form, hide the
// latency of their table look-ups and fp64 chains, which the walk itself cannot
// (one power per step of the walk: 378 us on [64,256,56,56]; in rounds: 236 us; with the
// window in registers, the next round's loads under way and the tables in LDS: 140 us).
constexpr uint32_t kLrnRound = 8;

// The two tables of powf in LDS: read from there, the powers leave the vector
// memory counter alone, so that waiting for a table entry is not waiting for the
// next round's channels, which were asked for before it.
struct LrnTables {
  uint64_t exp2[32];
  libm::PowfLog2Entry log2[16];
};

// All lanes of the workgroup, before any of them leaves.
SHDW_DEVICE void lrn_stage_tables(LrnTables* t) {
  if (threadIdx.x < 32) t->exp2[threadIdx.x] = libm::kExp2fTab[threadIdx.x];
  if (threadIdx.x < 16) t->log2[threadIdx.x] = libm::kPowfLog2Tab[threadIdx.x];
  __syncthreads();
}

// powf(scale, y) for the scales of a round.  Where every scale of the wave lies in
// [2^-100, 2^100] and 0 < |y| <= 1.25 (`small_power`; LRN's scales are near k, its power
// -0.75), |y log2 scale| is below 126 and nothing of powf's special cases can apply:
// two comparisons on the round's extremes stand for the tests of each of the eight
// (a quarter of the instructions: [44,96,55,55] 39.1 -> 33.3 us, [64,256,56,56] 137 -> 118,
// held to five waves a SIMD; with the registers it likes, four, 38.1 and 118).  Otherwise the straight
// path with its range tests for all of them (any bits may go in, see powf_ordinary);
// then, if some lane holds a scale that is not a positive normal number, the whole
// function for those, one instance of its code.
SHDW_DEVICE void lrn_powers(const float (&scale)[kLrnRound], float y, bool small_power, const LrnTables* t,
                            float (&power)[kLrnRound]) {
  uint32_t lo = __float_as_uint(scale[0]), hi = lo;  // as bits: negative numbers and NaN lie above every positive one
#pragma unroll
  for (uint32_t j = 1; j < kLrnRound; ++j) {
    lo = min(lo, __float_as_uint(scale[j]));
    hi = max(hi, __float_as_uint(scale[j]));
  }
  if (small_power && __builtin_amdgcn_ballot_w64(!(lo >= __float_as_uint(0x1p-100f) && hi <= __float_as_uint(0x1p100f))) == 0) {
#pragma unroll
    for (uint32_t j = 0; j < kLrnRound; ++j)
      power[j] = libm::powf_ordinary<true>(__float_as_uint(scale[j]), y, 0u, t->exp2, t->log2);
    return;
  }
  asm volatile("");  // keeps the compiler from working out both forms side by side
  bool plain = true;
#pragma unroll
  for (uint32_t j = 0; j < kLrnRound; ++j) {
    power[j] = libm::powf_ordinary<false>(__float_as_uint(scale[j]), y, 0u, t->exp2, t->log2);
    plain = plain && libm::powf_is_ordinary(__float_as_uint(scale[j]), __float_as_uint(y));
  }
  if (__builtin_amdgcn_ballot_w64(!plain) == 0) return;
#pragma unroll 1
  for (uint32_t pick = 0; pick < kLrnRound; ++pick) {
    float s = scale[0];
#pragma unroll
    for (uint32_t j = 1; j < kLrnRound; ++j) s = pick == j ? scale[j] : s;
    if (libm::powf_is_ordinary(__float_as_uint(s), __float_as_uint(y))) continue;
    const float r = libm::exact_powf(s, y, libm::kExp2fTab);
#pragma unroll
    for (uint32_t j = 0; j < kLrnRound; ++j) power[j] = pick == j ? r : power[j];
  }
}

// ---- windows of 1, 3, 5 and 7 channels: the window lives in registers ----
// One, two or four waves of a workgroup own 64 positions and go through their channels in spans
// of a round each.  Every lane has the channels of its round at once, those of the next span
// on their way during the powers; the waves take turns at the walk, which is short (two dependent
// additions a channel), each handing the sum and the last SIZE channels to the next through
// LDS; then all of them work out their powers, which are most of the work, at the same time.
// Bound by the vector ALUs: the powers, fp64 for the most part.  With one wave
// walking all channels of its positions, and up to eight workgroups sharing the rounds of a
// position where there are few (each walking from the first channel on): [44,96,55,55]
// 36.9 -> 28.9 us (27.6 with what launch_windows cuts), [16,256,56,56] 48.6 -> 31.5, [64,256,56,56] 122 -> 92, [64,256,27,27] 50.0 ->
// 30.6, [1,96,55,55] 14.8 -> 8.8, [512,8,56,56] 48.0 -> 27.5, [100,40,56,56] 31.3 -> 24.0.  Rounds of 16
// and 24 channels: 37.8 and 37.6 on the first.
//
// Round c0 finishes channels c0 .. c0 + 7, for which the sum takes in channel c + post and
// lets go of channel c - post - 1: own[j] is channel c0 + post + j, prev[t] channel
// c0 + post - SIZE + t.  y may be x: what a span writes lies behind everything that later
// spans read, and inside a span all is read before the last of its barriers.
constexpr int kLrnWaves = kBlock / kWave;

template <int SIZE>
struct LrnHand {
  float accum[kWave], prev[SIZE][kWave];
};

// EDGE: the first segments and those that reach past the last channel, with the tests of the
// reference's three loops (the same for all lanes); the segments between them need none.
template <int SIZE, bool EDGE>
SHDW_DEVICE float lrn_walk(const float (&own)[kLrnRound], const float (&prev)[SIZE],
                           float (&scale)[kLrnRound], float accum, uint32_t c0, uint32_t channels,
                           float alpha_over_size, float k) {
  constexpr uint32_t post = (SIZE - 1) / 2;
#pragma unroll
  for (int j = 0; j < static_cast<int>(kLrnRound); ++j) {
    const uint32_t c = c0 + j;
    if (!EDGE || c + post < channels) accum += own[j] * own[j];
    if (!EDGE || (c > post && c < channels)) {
      const float leaving = j >= SIZE ? own[j >= SIZE ? j - SIZE : 0] : prev[j < SIZE ? j : 0];
      accum -= leaving * leaving;
    }
    scale[j] = k + accum * alpha_over_size;
  }
  return accum;
}

// WAVES: how many of the workgroup's four waves share the channels of 64 positions; the others have positions
// of their own (see the rule at launch_windows).
//
// STREAM: the stores carry the streams' hint; not where rows of positions start inside a vector, whose
// pieces of lines would leave one by one ([44,96,55,55] 32.6 us plain, 34.0 with it, [68,256,27,27] 35.0
// and 40.5; [64,256,56,56] 93.2 and 82.1, [256,64,14,14] 11.8 and 10.5, all with four waves a position).
template <int SIZE, int WAVES, bool STREAM>
SHDW_DEVICE void lrn_window(LrnTables& tables, LrnHand<SIZE>* hands, uint32_t block, uint32_t first, const float* x, float* y,
                            uint32_t positions, uint32_t step, uint32_t channels, float alpha_over_size, float neg_beta, float k,
                            const FastDiv& f_step) {
  constexpr int SEG = kLrnRound;
  static_assert(SIZE % 2 == 1 && SIZE <= SEG, "the window must fit into a round");
  constexpr uint32_t post = (SIZE - 1) / 2;
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t in_group = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  // in_group is below 4, which the compiler does not know: spelt out, [2,56,28,28] takes 6.1 us instead of 6.4
  const uint32_t share = WAVES == kLrnWaves ? 0u : in_group / WAVES, wave = WAVES == kLrnWaves ? in_group : in_group % WAVES;
  LrnHand<SIZE>& hand = hands[share];
  const uint32_t p = first + (block * (kLrnWaves / WAVES) + share) * kWave + lane, at = min(p, positions - 1);
  const uint32_t b = fd_div(at, f_step);
  const size_t base = static_cast<size_t>(b) * channels * step + (at - b * step);
  const float* in = x + base;
  float* out = y + base;
  float ahead[SEG];  // the next span's, on their way during the powers
  auto request = [&](uint32_t c0) {
#pragma unroll
    for (int j = 0; j < SEG; ++j) ahead[j] = in[static_cast<size_t>(min(c0 + post + j, channels - 1)) * step];
  };
  request(wave * SEG);
  for (uint32_t span = 0; span < channels; span += WAVES * SEG) {
    const uint32_t c0 = span + wave * SEG;
    float own[SEG], prev[SIZE], scale[SEG];
#pragma unroll
    for (int j = 0; j < SEG; ++j) own[j] = ahead[j];
    if (c0 == 0) {
#pragma unroll
      for (int t = 0; t < SIZE; ++t) prev[t] = t + static_cast<int>(post) >= SIZE ? in[static_cast<size_t>(t + post - SIZE) * step] : 0.f;
    }
    for (uint32_t turn = 0; turn < WAVES; ++turn) {
      if (wave == turn && c0 < channels) {  // the same for the whole wave
        float accum = 0.f;
        if (c0 == 0) {
#pragma unroll
          for (int t = SIZE - static_cast<int>(post); t < SIZE; ++t) accum += prev[t] * prev[t];
        } else {
          accum = hand.accum[lane];
#pragma unroll
          for (int t = 0; t < SIZE; ++t) prev[t] = hand.prev[t][lane];
        }
        if (c0 > post && c0 + post + SEG <= channels)
          accum = lrn_walk<SIZE, false>(own, prev, scale, accum, c0, channels, alpha_over_size, k);
        else
          accum = lrn_walk<SIZE, true>(own, prev, scale, accum, c0, channels, alpha_over_size, k);
        hand.accum[lane] = accum;
#pragma unroll
        for (int t = 0; t < SIZE; ++t) hand.prev[t][lane] = own[SEG - SIZE + t];
      }
      if (WAVES > 1) __syncthreads();
    }
    if (span + WAVES * SEG < channels) request(c0 + WAVES * SEG);
    if (c0 >= channels) continue;
    float power[SEG];
    lrn_powers(scale, neg_beta, neg_beta != 0.f && __builtin_fabsf(neg_beta) <= 1.25f, &tables, power);
#pragma unroll
    for (int j = 0; j < SEG; ++j) {
      const float centre = j >= static_cast<int>(post) ? own[j >= static_cast<int>(post) ? j - post : 0]
                                                       : prev[j < static_cast<int>(post) ? SIZE - post + j : 0];
      if (c0 + j < channels && p < positions) {
        float* to = out + static_cast<size_t>(c0 + j) * step;
        if (STREAM) __builtin_nontemporal_store(centre * power[j], to);
        else *to = centre * power[j];
      }
    }
  }
}

// `whole` workgroups of WAVES waves for 64 positions, and behind them, if there are more, workgroups of four waves
// for what positions are left.
template <int SIZE, int WAVES, bool STREAM>
__global__ __launch_bounds__(kBlock, 5) void lrn_window_kernel(const float* x, float* y, uint32_t positions, uint32_t step,
                                                               uint32_t channels, float alpha_over_size, float neg_beta,
                                                               float k, uint32_t whole, FastDiv f_step) {
  __shared__ LrnTables tables;
  __shared__ LrnHand<SIZE> hands[kLrnWaves / WAVES];
  lrn_stage_tables(&tables);
  if (WAVES == 2 && blockIdx.x >= whole) {
    lrn_window<SIZE, kLrnWaves, STREAM>(tables, hands, blockIdx.x - whole, whole * (kLrnWaves / WAVES * kWave), x, y, positions, step,
                                        channels, alpha_over_size, neg_beta, k, f_step);
    return;
  }
  // Runs of positions that start inside a line share it with the run before: the XCD's own neighbours then
  // ([44,96,55,55] 31.2 -> 29.8 us, [64,256,27,27] 34.1 -> 30.3; no gain where rows are whole vectors).
  const uint32_t block = STREAM ? blockIdx.x : xcd_contiguous(blockIdx.x, whole);
  lrn_window<SIZE, WAVES, STREAM>(tables, hands, block, 0, x, y, positions, step, channels, alpha_over_size, neg_beta, k, f_step);
}

// The channels of the round that starts at head0 (zeros past the last one).
SHDW_DEVICE void lrn_fetch(const float* in, uint32_t head0, uint32_t channels, uint32_t step,
                           float (&values)[kLrnRound]) {
#pragma unroll
  for (uint32_t j = 0; j < kLrnRound; ++j)
    values[j] = head0 + j < channels ? in[static_cast<size_t>(head0 + j) * step] : 0.f;
}

// ---- any window up to kLrnMaxSize channels: the window lives in LDS ----
__global__ __launch_bounds__(kBlock) void lrn_across_channels_kernel(
    const float* x, float* y, uint32_t positions, uint32_t step, uint32_t channels, FastDiv f_step,
    uint32_t size, float alpha_over_size, float neg_beta, float k) {
  extern __shared__ float window[];  // [size][kBlock]
  __shared__ LrnTables tables;
  lrn_stage_tables(&tables);
  const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
  if (p >= positions) return;  // no barrier below: a lane only meets its own column
  const uint32_t b = fd_div(p, f_step);
  const size_t base = static_cast<size_t>(b) * channels * step + (p - b * step);
  const float* in = x + base;
  float* out = y + base;
  float* mine = window + threadIdx.x;
  const uint32_t post = (size - 1) / 2;
  const uint32_t steps = channels + post;  // step `head` takes channel head in and finishes channel head - post
  float accum = 0.f;
  uint32_t slot_head = 0, slot_mid = 0;  // head % size and (head - post) % size
  float round[kLrnRound];
  const uint32_t rounds = (steps + kLrnRound - 1) / kLrnRound;  // shared out over gridDim.y as above
  const uint32_t first = blockIdx.y * rounds / gridDim.y * kLrnRound;
  const uint32_t end = (blockIdx.y + 1) * rounds / gridDim.y * kLrnRound;
  lrn_fetch(in, 0, channels, step, round);
  for (uint32_t head0 = 0; head0 < end; head0 += kLrnRound) {
    float entering[kLrnRound], scale[kLrnRound], centre[kLrnRound], power[kLrnRound];
#pragma unroll
    for (uint32_t j = 0; j < kLrnRound; ++j) entering[j] = round[j];
    lrn_fetch(in, head0 + kLrnRound, channels, step, round);  // the next round's, on their way during the powers
#pragma unroll
    for (uint32_t j = 0; j < kLrnRound; ++j) {
      const uint32_t head = head0 + j;
      scale[j] = 1.f;
      centre[j] = 0.f;
      if (head < steps) {  // the same for every lane
        if (head < channels) accum += entering[j] * entering[j];
        if (head >= size) {  // channel head - size lives where channel head goes
          const float leaving = mine[slot_head * kBlock];
          accum -= leaving * leaving;
        }
        if (head < channels) mine[slot_head * kBlock] = entering[j];
        slot_head = slot_head + 1 == size ? 0 : slot_head + 1;
        if (head >= post) {
          scale[j] = k + accum * alpha_over_size;
          centre[j] = mine[slot_mid * kBlock];
          slot_mid = slot_mid + 1 == size ? 0 : slot_mid + 1;
        }
      }
    }
    if (head0 < first) continue;  // in front of this workgroup's share: only the sum had to pass through
    lrn_powers(scale, neg_beta, neg_beta != 0.f && __builtin_fabsf(neg_beta) <= 1.25f, &tables, power);
#pragma unroll
    for (uint32_t j = 0; j < kLrnRound; ++j) {
      const uint32_t head = head0 + j;
      if (head >= post && head < steps) out[static_cast<size_t>(head - post) * step] = centre[j] * power[j];
    }
  }
}

}  // namespace shdw

using namespace shdw;

namespace {

// Two waves for 64 positions: the vector ALUs bound this, so the CU with the most workgroups does. Workgroups beyond
// the CUs' even share, if they are half a share or less, are cut in two, of four waves for 64 positions, so that no CU
// gets more than half of one on top: [44,96,55,55], 1040 workgroups, 29.8 -> 27.6 us, [44,96,56,56] 26.2 -> 22.8,
// [45,96,50,50] 24.8 -> 21.4, [33,64,64,64] 18.9 -> 17.1.
template <int SIZE, int WAVES>
void launch_windows(const float* x, float* y, uint32_t positions, uint32_t step, uint32_t channels, float alpha_over_size,
                    float neg_beta, float k, bool stream, hipStream_t st) {
  constexpr uint32_t kOwned = kLrnWaves / WAVES * kWave, kCus = 256;
  const uint32_t all = positions / kOwned + (positions % kOwned != 0), rest = all % kCus;
  const bool cut = WAVES == 2 && all > kCus && rest != 0 && rest <= kCus / 2 && channels > 4 * kLrnRound;
  const uint32_t whole = cut ? all - rest : all;
  const uint32_t grid = cut ? whole + (positions - whole * kOwned + kWave - 1) / kWave : all;
  const FastDiv f_step = make_fastdiv(step);
  if (stream) lrn_window_kernel<SIZE, WAVES, true><<<grid, kBlock, 0, st>>>(x, y, positions, step, channels, alpha_over_size, neg_beta, k, whole, f_step);
  else lrn_window_kernel<SIZE, WAVES, false><<<grid, kBlock, 0, st>>>(x, y, positions, step, channels, alpha_over_size, neg_beta, k, whole, f_step);
}

// One wave for 64 positions works without barriers and leaves no wave without a round, four finish soonest and
// share the SIMDs out most evenly: one from where on the SIMDs' shares of the runs of 64 (runs / 1024, rounded up)
// differ by an eighth at most, two from where on four are more than the chip holds at a time (5120), no more than
// there are rounds; and four where a walk over many channels would outlast the others.  With 1 / 2 / 4 waves,
// by runs: 23437 of 8 channels 26.6 / 37.1 / 58.6 us, 11718 of 16 24.7 / 26.4 / 41.5, 4687 of 40 25.1 / 26.6 / 32.1,
// 4000 of 96 42.1 / 44.1 / 46.5; 3332 of 64 28.4 / 26.3 / 26.9, 3136 of 40 18.5 / 18.3 / 20.7, 3136 of 64
// 29.6 / 26.7 / 27.0, of 96 42.1 / 39.4 / 36.2, of 256 103.6 / 92.8 / 88.5; 2079 of 96 34.4 / 28.7 / 30.0, 1400 of 96
// 27.4 / 19.7 / 20.9; 1200 of 96 26.3 / 19.1 / 16.0, 732 of 256 48.7 / 36.0 / 28.6.
template <int SIZE>
void launch_windows(const float* x, float* y, uint32_t positions, uint32_t step, uint32_t channels, float alpha_over_size,
                    float neg_beta, float k, bool stream, hipStream_t st) {
  constexpr uint32_t kResident = 5120, kEven = 3584;
  const uint32_t runs = (positions + kWave - 1) / kWave, rounds = (channels + kLrnRound - 1) / kLrnRound;
  if (rounds == 1 || (runs > kEven && rounds <= 16))
    launch_windows<SIZE, 1>(x, y, positions, step, channels, alpha_over_size, neg_beta, k, stream, st);
  else if (rounds == 2 || (runs > kResident / 4 && (runs <= kResident / 2 || rounds <= 8)))
    launch_windows<SIZE, 2>(x, y, positions, step, channels, alpha_over_size, neg_beta, k, stream, st);
  else
    launch_windows<SIZE, 4>(x, y, positions, step, channels, alpha_over_size, neg_beta, k, stream, st);
}

}  // namespace

extern "C" int shdw_hip_lrn(const int* in_shape, int size, float alpha, float beta, float k, const float* x,
                            float* y, void* stream) {
  if (!in_shape || size < 1 || size % 2 == 0) return SHDW_E_INVALID_ARGUMENT;
  long long count = 1;
  for (int d = 0; d < 4; ++d) {
    if (in_shape[d] < 0) return SHDW_E_INVALID_ARGUMENT;
    count *= in_shape[d];
    if (count > INT_MAX) return SHDW_E_UNSUPPORTED;
  }
  const int channels = in_shape[1], post = (size - 1) / 2;
  // fewer channels than lie behind the centre of a window: the reference's last
  // loop then writes in front of its scale blob
  if (channels < post) return SHDW_E_INVALID_ARGUMENT;
  if (count == 0) return SHDW_OK;
  if (!x || !y) return SHDW_E_INVALID_ARGUMENT;
  if (size > kLrnMaxSize) return SHDW_E_UNSUPPORTED;
  const uint32_t step = static_cast<uint32_t>(in_shape[2]) * static_cast<uint32_t>(in_shape[3]);
  const uint32_t positions = static_cast<uint32_t>(in_shape[0]) * step;
  const float alpha_over_size = alpha / size;  // float / int, as the reference forms it
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint32_t grid = grid_for(positions), chan = static_cast<uint32_t>(channels);
  const FastDiv f_step = make_fastdiv(step);
  if (size <= 7) {
    const bool stream = step % 4 == 0 && aligned16(y);
    if (size == 1) launch_windows<1>(x, y, positions, step, chan, alpha_over_size, -beta, k, stream, st);
    else if (size == 3) launch_windows<3>(x, y, positions, step, chan, alpha_over_size, -beta, k, stream, st);
    else if (size == 5) launch_windows<5>(x, y, positions, step, chan, alpha_over_size, -beta, k, stream, st);
    else launch_windows<7>(x, y, positions, step, chan, alpha_over_size, -beta, k, stream, st);
    return launch_status();
  }
  // A tensor with few positions has few waves, and each walks all the channels one round after
  // the other (72 us for 256 channels, however few the waves).  Up to eight workgroups then share
  // the rounds of a position, about 4096 waves in all and four rounds each at the least.  A window of nine
  // with 1 / 2 / 4 / 8 / 16 shares: [1,256,56,56] (49 waves) 72 / 56 / 49 / 45 / 43 us, [4,256,56,56] 72 / 57 / 50 / 48 / 49,
  // [16,256,56,56] (784) 82 / 71 / 67 / 78 / 105, [44,96,55,55] (2080) 44 / 42 / 49 / 64 / 95, [64,256,56,56] (3136)
  // 126 / 137 / 162; of 31 [44,96,55,55] 47 / 51 / 56, [16,256,56,56] 83 / 72 / 68.
  // In place a workgroup would overwrite what another still has to read: one share.
  const uint32_t waves = (positions + kWave - 1) / kWave;
  const uint32_t rounds = (chan + static_cast<uint32_t>(post) + kLrnRound - 1) / kLrnRound;
  uint32_t shares = (4096 + waves / 2) / waves;
  const uint32_t most = waves <= 512 ? 8u : 4u;
  shares = shares > most ? most : shares;
  shares = shares > rounds / 4 ? rounds / 4 : shares;
  if (x == y || shares < 1) shares = 1;
  const size_t lds = static_cast<size_t>(size) * kBlock * sizeof(float);
  lrn_across_channels_kernel<<<dim3(grid, shares), kBlock, lds, st>>>(x, y, positions, step, chan, f_step,
                                                        static_cast<uint32_t>(size), alpha_over_size, -beta, k);
  return launch_status();
}
