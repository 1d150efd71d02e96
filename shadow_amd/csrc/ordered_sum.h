// The fp32 running sum of a row, front to back, by a whole wave: the bits of
//   for (i = 0; i < n; ++i) sum += v[i];
// for terms that are not negative, without n additions that wait for one another.
//
// While a running sum stays between two powers of two, 2^e <= sum < 2^(e+1), it is a multiple
// of one unit u (its last place), and rounding sum + v to such a multiple depends on sum in one
// respect only: a tie goes to the even multiple.  A run of terms therefore adds one of two
// numbers of units to any such sum, one where its last bit is 0 and one where it is 1, and these
// two can be had by adding the terms to 2^e and to 2^e + u.  Read as an integer, a float's bits
// count units: the run takes the bits b to b + (b & 1 ? odd : even).  Two runs of the same e
// make one (the second's number is chosen by the first's last bit), so 64 lanes' runs make
// one in six steps.
//
// Each lane has a guess of the sum that reaches it, from the lanes' sums in any order: of that only
// e is used.  The true sum then goes through the lanes: over lanes of one e at once, from the
// guessed power of two on (checked: the sum in front of them and the sum behind them must both lie
// there, and as no term is negative every sum between them does), and by adding a lane's terms
// one after the other where the sum passes a power of two inside it, or where a guess was wrong.
// A row of n equal terms passes log2(n) powers of two, half of them in its first lane's terms.
//
// A guess is wrong where the sum passes a power of two within rounding of the end of a lane's terms (a row of 12544 in three
// thousand: every other call over 2048 of them): the true sum then passes it in the last lane of a run, or in the first.
// What is left of the run without that lane is joined anew, a few times a chunk.  One by one to the run's end, up to 63 lanes of
// 0.1 us, calls that had such a row took, averages of ReLU's output: 2048 x 3136 13.3 us instead of 7.5, 2048 x 12544 25.8 (17.7),
// softmax of [1000,4096] 14.2 (12.2).  Where the true sum passes it in the first lane of a run, the run in front still holds: with
// one row in 37 of that kind 1024 x 2048 took 7.5 us, and takes 4.3, 2048 x 3136 10.1 and 6.9.
#ifndef SHADOW_AMD_CSRC_ORDERED_SUM_H_
#define SHADOW_AMD_CSRC_ORDERED_SUM_H_

#include "device_common.h"

namespace shdw {

constexpr uint32_t kBinade = 1u << 23, kExponentBits = 0x7f800000u;

// What a lane's terms add to bits below a power of two, for even and odd ones; `first`: nothing in front of this
// lane is included (`even` and `odd` are of its own terms alone).
struct UnitRun {
  uint32_t even, odd, first;
};

template <int CTRL, int ROWS>
SHDW_DEVICE uint32_t moved_lane(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROWS, 0xf, false));
}

// The lanes named by the DPP control in front of this lane's own, unless nothing in front of this lane belongs to it
// (`first`); lanes without such a lane keep theirs.
template <int CTRL, int ROWS>
SHDW_DEVICE void join_units(UnitRun& r, bool first) {
  const uint32_t even = moved_lane<CTRL, ROWS>(r.even), odd = moved_lane<CTRL, ROWS>(r.odd);
  const uint32_t joined_even = even + (even & 1u ? r.odd : r.even);
  const uint32_t joined_odd = odd + (odd & 1u ? r.even : r.odd);
  r.even = first ? r.even : joined_even;
  r.odd = first ? r.odd : joined_odd;
}

template <int CTRL, int ROWS>
SHDW_DEVICE void join_run(UnitRun& r) {
  const uint32_t first = moved_lane<CTRL, ROWS>(r.first);
  join_units<CTRL, ROWS>(r, r.first != 0);
  r.first |= first;
}

template <int CTRL, int ROWS>
SHDW_DEVICE float add_lane(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, false));
}

constexpr int kDppShr1 = 0x111, kDppShr2 = 0x112, kDppShr4 = 0x114, kDppShr8 = 0x118;  // inside 16 lanes
constexpr int kDppBcast15 = 0x142, kDppBcast31 = 0x143;  // the last lane of 16, of 32, to the 16, 32 behind them

// All lanes' runs joined with the lanes that have met a start in a mask: two registers fewer than six of join_run, but
// 0.05 us more (with it everywhere 64 averages of 50176 take 29.0 us instead of 27.6).
SHDW_DEVICE void join_runs_masked(UnitRun& r, uint64_t starts) {
  const auto first = [&] { return __builtin_amdgcn_inverse_ballot_w64(starts); };
  join_units<kDppShr1, 0xf>(r, first());
  starts |= starts << 1 & 0xfffefffefffefffeull;
  join_units<kDppShr2, 0xf>(r, first());
  starts |= starts << 2 & 0xfffcfffcfffcfffcull;
  join_units<kDppShr4, 0xf>(r, first());
  starts |= starts << 4 & 0xfff0fff0fff0fff0ull;
  join_units<kDppShr8, 0xf>(r, first());
  starts |= starts << 8 & 0xff00ff00ff00ff00ull;
  join_units<kDppBcast15, 0xa>(r, first());
  starts |= (starts >> 15 & 0x0000000100000001ull) * 0xffff0000ull;
  join_units<kDppBcast31, 0xc>(r, first());
}

// Whether some element is negative, -0 or NaN.
template <int K>
SHDW_DEVICE bool any_sign(const float (&v)[K]) {
  uint32_t most = __float_as_uint(v[0]);
#pragma unroll
  for (int k = 1; k < K; ++k) most = max(most, __float_as_uint(v[k]));
  return most > kExponentBits;
}

// sum + v[0] + v[1] + ... of lane 0, then of lane 1, ...: the same sum in all lanes.  All 64 lanes call it, with
// the same sum; neither it nor any term is negative or NaN (infinities are fine).
template <int K>
SHDW_DEVICE float wave_sum_in_order(const float (&v)[K], float sum) {
  float own[4] = {v[0], v[1], v[2], v[3]};
  static_assert(K % 4 == 0 && K >= 4, "");
#pragma unroll
  for (int k = 4; k < K; ++k) own[k % 4] += v[k];
  const float mine = (own[0] + own[1]) + (own[2] + own[3]);
  float upto = mine;
  upto = add_lane<kDppShr1, 0xf>(upto);
  upto = add_lane<kDppShr2, 0xf>(upto);
  upto = add_lane<kDppShr4, 0xf>(upto);
  upto = add_lane<kDppShr8, 0xf>(upto);
  upto = add_lane<kDppBcast15, 0xa>(upto);
  upto = add_lane<kDppBcast31, 0xc>(upto);
  const float before = sum + lane_in_front(upto);
  const uint32_t power = __float_as_uint(before) & kExponentBits;
  const uint32_t guess = __float_as_uint(before) & ~1u;  // lane 0's is the sum's own, so its terms are added to the sum itself
  float from_even = __uint_as_float(guess), from_odd = __uint_as_float(guess | 1u);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    from_even += v[k];
    from_odd += v[k];
  }
  // passes: this lane's terms are added one by one; first: at, and behind, such a lane, and where e changes
  const uint32_t lane_id = threadIdx.x % kWave;
  const bool passes = lane_id == 0 || power == kExponentBits ||
                      max(__float_as_uint(from_even), __float_as_uint(from_odd)) - power >= kBinade;
  const uint32_t tag = passes ? 1u : power;  // of the powers none is 1
  const uint32_t tag_before = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(1, static_cast<int>(tag), kDppWaveShr1, 0xf, 0xf, false));
  const bool starts = passes || tag != tag_before;
  const uint64_t all_starts = __builtin_amdgcn_ballot_w64(starts);
  // lane 0 passes: its bit says that all lanes are done
  const uint64_t whole_runs = (all_starts & ~__builtin_amdgcn_ballot_w64(passes)) | 1u;
  UnitRun run{__float_as_uint(from_even) - guess, __float_as_uint(from_odd) - (guess | 1u), starts ? 1u : 0u};
  join_run<kDppShr1, 0xf>(run);
  join_run<kDppShr2, 0xf>(run);
  join_run<kDppShr4, 0xf>(run);
  join_run<kDppShr8, 0xf>(run);
  join_run<kDppBcast15, 0xa>(run);
  join_run<kDppBcast31, 0xc>(run);
  uint32_t bits = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(__float_as_int(sum)));
  const auto of_lane = [](uint32_t value, uint32_t lane) {
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(value), static_cast<int>(lane)));
  };
  bits = of_lane(bits & 1u ? __float_as_uint(from_odd) : __float_as_uint(from_even), 0);
  const auto add_one = [&](uint32_t lane) {
    float s = __uint_as_float(bits);
#pragma unroll
    for (int k = 0; k < K; ++k) s += v[k];
    bits = of_lane(__float_as_uint(s), lane);
  };
  // The lanes from `lane` on that make one run, if they do, at once; then the lane behind them, one by one.
  const uint64_t ends = all_starts >> 1 | 1ull << 63;  // lanes in front of a start, and the last
  uint32_t lane = 1;
  do {  // the same for all lanes; every turn is of one lane at least
    const uint32_t last = static_cast<uint32_t>(__builtin_ctzll(ends >> lane)) + lane;
    const uint32_t low = of_lane(power, lane), even = of_lane(run.even, last), odd = of_lane(run.odd, last);
    const uint32_t next = bits + (bits & 1u ? odd : even);
    // a run is known from its first lane on: not behind a lane whose guess was wrong
    if ((whole_runs >> lane & 1u) != 0) {
      if (bits - low >= kBinade || next - low >= kBinade) break;
      bits = next;
      lane = last + 1;
      // a run right behind a run: the sum that the first leaves is below the second's power of two, so the second's guess is wrong
      if ((whole_runs >> lane % kWave & 1u) != 0) break;
    }
    add_one(lane);
  } while (++lane < kWave);
  if (__builtin_expect(lane == kWave, 1)) return __uint_as_float(bits);

  // The same from `lane` on, the first of a run whose guess was wrong, with new starts.  Every turn is of one lane at
  // least, or is one of the joins.  What a lane adds is the same from any even, from any odd number of units that keeps it
  // inside its power of two: taken again, from the lowest, so that the loop above need not hold it.  Two registers, with
  // which the gated block's rows of four vectors a lane have 74 and a workgroup a CU less (gate.hip).
  const auto join = [&](uint64_t at) {
    float low_even = __uint_as_float(power), low_odd = __uint_as_float(power | 1u);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      low_even += v[k];
      low_odd += v[k];
    }
    UnitRun joined{__float_as_uint(low_even) - power, __float_as_uint(low_odd) - (power | 1u), 0};
    join_runs_masked(joined, at);
    return joined;
  };
  uint64_t new_starts = all_starts, new_whole = whole_runs;
  uint32_t joins_left = 3;
  while (lane < kWave) {
    const uint64_t new_ends = new_starts >> 1 | 1ull << 63;
    const uint32_t last = static_cast<uint32_t>(__builtin_ctzll(new_ends >> lane)) + lane;
    const uint32_t low = of_lane(power, lane), even = of_lane(run.even, last), odd = of_lane(run.odd, last);
    const uint32_t next = bits + (bits & 1u ? odd : even);
    const bool inside = bits - low < kBinade;
    if ((new_whole >> lane & 1u) != 0) {
      if (inside && next - low < kBinade) {
        bits = next;
        lane = last + 1;
        continue;
      }
      if (joins_left != 0 && last > lane) {
        --joins_left;
        const uint64_t start = 1ull << (inside ? last : lane + 1);
        new_starts |= start, new_whole |= start;
        run = join(new_starts);
        if (inside) continue;
      }
    }
    add_one(lane);
    ++lane;
  }
  return __uint_as_float(bits);
}

}  // namespace shdw

#endif  // SHADOW_AMD_CSRC_ORDERED_SUM_H_
