// A model of wave_sum_in_order (shadow_amd/csrc/ordered_sum.h), lane by lane, for tests/test_ordered_sum_cpu.py:
// a value of the kernel is an array of the 64 lanes' here, and a DPP move reads its neighbour's element.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <vector>

namespace {

constexpr int kLanes = 64;
constexpr uint32_t kBinade = 1u << 23, kExponentBits = 0x7f800000u;

uint32_t bits_of(float v) {
  uint32_t b;
  std::memcpy(&b, &v, 4);
  return b;
}
float float_of(uint32_t b) {
  float v;
  std::memcpy(&v, &b, 4);
  return v;
}

// The lane that a step of the scan over the lanes reads, or -1 where it has none and takes 0: row_shr 1, 2, 4 and 8
// inside 16 lanes, then lane 15 of each pair of 16 to the second, then lane 31 to the upper half.
int source(int step, int lane) {
  if (step < 4) return lane % 16 >= 1 << step ? lane - (1 << step) : -1;
  if (step == 4) return lane / 16 % 2 == 1 ? lane / 16 * 16 - 1 : -1;
  return lane >= 32 ? 31 : -1;
}

// Lanes that have met a start behind a step, of those that had in front of it, in a mask as join_runs_masked has them; the last
// step's are not asked for.
uint64_t met(int step, uint64_t starts) {
  switch (step) {
    case 0: return starts | (starts << 1 & 0xfffefffefffefffeull);
    case 1: return starts | (starts << 2 & 0xfffcfffcfffcfffcull);
    case 2: return starts | (starts << 4 & 0xfff0fff0fff0fff0ull);
    case 3: return starts | (starts << 8 & 0xff00ff00ff00ff00ull);
    default: return starts | (starts >> 15 & 0x0000000100000001ull) * 0xffff0000ull;
  }
}

struct Counts {
  long wrong = 0, one_by_one = 0, joins = 0;  // guesses that were off, lanes added one by one behind the first, runs joined anew
};

template <int K>
float wave_sum_in_order(const float (&v)[kLanes][K], float sum, Counts& n) {
  float upto[kLanes];
  for (int l = 0; l < kLanes; ++l) {
    float own[4] = {v[l][0], v[l][1], v[l][2], v[l][3]};
    for (int k = 4; k < K; ++k) own[k % 4] += v[l][k];
    upto[l] = (own[0] + own[1]) + (own[2] + own[3]);
  }
  for (int step = 0; step < 6; ++step) {
    float moved[kLanes];
    for (int l = 0; l < kLanes; ++l) moved[l] = source(step, l) < 0 ? 0.f : upto[source(step, l)];
    for (int l = 0; l < kLanes; ++l) upto[l] += moved[l];
  }
  uint32_t power[kLanes], own_even[kLanes], own_odd[kLanes], tag[kLanes];
  float from_even[kLanes], from_odd[kLanes];
  uint64_t all_starts = 0, all_passes = 0;
  for (int l = 0; l < kLanes; ++l) {
    const uint32_t before = bits_of(sum + (l ? upto[l - 1] : 0.f)), guess = before & ~1u;
    power[l] = before & kExponentBits;
    from_even[l] = float_of(guess), from_odd[l] = float_of(guess | 1u);
    for (int k = 0; k < K; ++k) from_even[l] += v[l][k], from_odd[l] += v[l][k];
    own_even[l] = bits_of(from_even[l]) - guess, own_odd[l] = bits_of(from_odd[l]) - (guess | 1u);
    const uint32_t most = std::max(bits_of(from_even[l]), bits_of(from_odd[l]));
    const bool passes = l == 0 || power[l] == kExponentBits || most - power[l] >= kBinade;
    tag[l] = passes ? 1u : power[l];
    const bool starts = passes || tag[l] != (l ? tag[l - 1] : 1u);
    all_starts |= static_cast<uint64_t>(starts) << l, all_passes |= static_cast<uint64_t>(passes) << l;
  }
  uint32_t even[kLanes], odd[kLanes];
  const auto join = [&](uint64_t starts) {
    for (int l = 0; l < kLanes; ++l) even[l] = own_even[l], odd[l] = own_odd[l];
    for (int step = 0; step < 6; ++step) {
      uint32_t e[kLanes], o[kLanes];
      for (int l = 0; l < kLanes; ++l) {
        const int s = source(step, l);
        e[l] = s < 0 ? 0 : even[s], o[l] = s < 0 ? 0 : odd[s];
      }
      for (int l = 0; l < kLanes; ++l) {
        const uint32_t joined_even = e[l] + (e[l] & 1u ? odd[l] : even[l]), joined_odd = o[l] + (o[l] & 1u ? even[l] : odd[l]);
        if (!(starts >> l & 1u)) even[l] = joined_even, odd[l] = joined_odd;
      }
      starts = met(step, starts);
    }
  };
  join(all_starts);
  uint32_t bits = bits_of(bits_of(sum) & 1u ? from_odd[0] : from_even[0]);
  const auto add_one = [&](int lane) {
    float s = float_of(bits);
    for (int k = 0; k < K; ++k) s += v[lane][k];
    bits = bits_of(s);
    ++n.one_by_one;
  };
  const uint64_t whole_runs = (all_starts & ~all_passes) | 1u, ends = all_starts >> 1 | 1ull << 63;
  int lane = 1;
  do {
    const int last = __builtin_ctzll(ends >> lane) + lane;
    const uint32_t low = power[lane], next = bits + (bits & 1u ? odd[last] : even[last]);
    if ((whole_runs >> lane & 1u) != 0) {
      if (bits - low >= kBinade || next - low >= kBinade) break;
      bits = next;
      lane = last + 1;
      if ((whole_runs >> lane % kLanes & 1u) != 0) break;
    }
    add_one(lane);
  } while (++lane < kLanes);
  uint64_t new_starts = all_starts, new_whole = whole_runs;
  int joins_left = 3;
  while (lane < kLanes) {
    const uint64_t new_ends = new_starts >> 1 | 1ull << 63;
    const int last = __builtin_ctzll(new_ends >> lane) + lane;
    const uint32_t low = power[lane], next = bits + (bits & 1u ? odd[last] : even[last]);
    const bool inside = bits - low < kBinade;
    if ((new_whole >> lane & 1u) != 0) {
      if (inside && next - low < kBinade) {
        bits = next;
        lane = last + 1;
        continue;
      }
      ++n.wrong;
      if (joins_left != 0 && last > lane) {
        --joins_left;
        for (int l = 0; l < kLanes; ++l) {  // again, from the lowest even and odd number of units of the lane's power of two
          float low_even = float_of(power[l]), low_odd = float_of(power[l] | 1u);
          for (int k = 0; k < K; ++k) low_even += v[l][k], low_odd += v[l][k];
          own_even[l] = bits_of(low_even) - power[l], own_odd[l] = bits_of(low_odd) - (power[l] | 1u);
        }
        const uint64_t start = 1ull << (inside ? last : lane + 1);
        new_starts |= start, new_whole |= start;
        join(new_starts);
        ++n.joins;
        if (inside) continue;
      }
    }
    add_one(lane);
    ++lane;
  }
  return float_of(bits);
}

// Terms and incoming sums of all kinds, none negative: even growth, ties in every addition, all sizes, subnormal
// ones, sums that overflow, zeros, infinities, and sums that stay within rounding of a power of two.
template <int K>
long scan(unsigned seed, long chunks, long* counts) {
  std::mt19937_64 gen(seed);
  const auto unit = [&] { return std::ldexp(static_cast<double>(gen() >> 11), -53); };
  const auto below = [&](int n) { return static_cast<int>(gen() % static_cast<unsigned>(n)); };
  Counts n;
  long bad = 0;
  for (long c = 0; c < chunks; ++c) {
    float v[kLanes][K];
    float sum = 0.f;
    switch (below(6)) {
      case 0: break;
      case 1: sum = static_cast<float>(std::ldexp(1.0, below(40) - 20)); break;
      case 2: sum = std::nextafterf(static_cast<float>(std::ldexp(1.0, below(40) - 20)), 0.f); break;
      case 3: sum = static_cast<float>(std::ldexp(unit(), below(200) - 100)); break;
      case 4: sum = float_of(static_cast<uint32_t>(below(1 << 24))); break;  // subnormal, or just not
      default: sum = below(8) ? static_cast<float>(unit()) : INFINITY;
    }
    const int kind = below(11), at = below(kLanes * K);
    const double scale = sum > 0.f && std::isfinite(sum) ? sum : 1.0, goal = std::ldexp(1.0, std::ilogb(scale) + 1);
    std::vector<double> head(at + 1);
    double total = 0;
    for (double& h : head) total += h = unit();
    for (double& h : head) h *= (goal - (std::isfinite(sum) ? sum : 0.f)) / total;
    for (int i = 0; i < kLanes * K; ++i) {
      double t = 0;
      switch (kind) {
        case 0: t = scale; break;
        case 1: t = std::max(0.0, unit() * 3 - 1); break;
        case 2: t = std::ldexp(scale, -below(26)); break;
        case 3: t = std::ldexp(unit(), below(81) - 40); break;
        case 4: t = std::ldexp(below(9), -149); break;
        case 5: t = unit() * 3e38; break;
        case 6: t = i < at ? 0 : unit(); break;
        case 7: t = i == at ? INFINITY : 0.1; break;
        case 8: t = i % kLanes == 0 ? 16777216.0 : 1; break;
        case 9: t = i <= at ? head[i] : std::ldexp(goal * unit(), -30); break;
        default: t = std::ldexp(scale, -24) * (below(4) ? 1 : 1.5);
      }
      v[i / K][i % K] = static_cast<float>(t);
    }
    float want = sum;
    for (int i = 0; i < kLanes * K; ++i) want += v[i / K][i % K];
    if (bits_of(want) != bits_of(wave_sum_in_order(v, sum, n))) ++bad;
  }
  counts[0] = n.wrong, counts[1] = n.one_by_one, counts[2] = n.joins;
  return bad;
}

// Uniform terms scaled so that their sum reaches a power of two just where a lane's terms end; counts[3]: the most lanes
// of a chunk that were added one by one.
template <int K>
long near(unsigned seed, long chunks, long* counts) {
  std::mt19937_64 gen(seed);
  Counts n;
  long bad = 0, most = 0;
  for (long c = 0; c < chunks; ++c) {
    double t[kLanes * K], total = 0;
    for (double& u : t) u = std::ldexp(static_cast<double>(gen() >> 11), -53);
    const int end = K * (3 + static_cast<int>(gen() % 58));
    for (int i = 0; i < end; ++i) total += t[i];
    const double factor = std::ldexp(1.0, std::ilogb(total)) / total;
    float v[kLanes][K], want = 0.f;
    for (int i = 0; i < kLanes * K; ++i) want += v[i / K][i % K] = static_cast<float>(t[i] * factor);
    const long before = n.one_by_one;
    if (bits_of(want) != bits_of(wave_sum_in_order(v, 0.f, n))) ++bad;
    most = std::max(most, n.one_by_one - before);
  }
  counts[0] = n.wrong, counts[1] = n.one_by_one, counts[2] = n.joins, counts[3] = most;
  return bad;
}

}  // namespace

// Chunks whose sum is not the running sum's to the bit; counts: guesses that were off, lanes added one by one, runs joined anew.
extern "C" long ordered_sum_scan(int terms, unsigned seed, long chunks, long* counts) {
  switch (terms) {
    case 16: return scan<16>(seed, chunks, counts);
    case 28: return scan<28>(seed, chunks, counts);
    case 32: return scan<32>(seed, chunks, counts);
  }
  return -1;
}

extern "C" long ordered_sum_near(int terms, unsigned seed, long chunks, long* counts) {
  switch (terms) {
    case 16: return near<16>(seed, chunks, counts);
    case 28: return near<28>(seed, chunks, counts);
    case 32: return near<32>(seed, chunks, counts);
  }
  return -1;
}
