// Shared device-side helpers for the gfx950 kernels: 128-bit vector access,
// exact division by launch-time constants, wave64 reductions.
#ifndef SHADOW_AMD_CSRC_DEVICE_COMMON_H_
#define SHADOW_AMD_CSRC_DEVICE_COMMON_H_

#include <hip/hip_runtime.h>

#include <cstdint>

// Shadow's CPU kernels are compiled for baseline x86-64: a*b+c is always a
// rounded multiply followed by a rounded add.  Keep the device code the same.
#pragma clang fp contract(off)

namespace shdw {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;
constexpr int kBlock = 256;  // 4 wave64 per workgroup
// Workgroup of the streaming kernels (one vector per lane, no LDS exchange, no
// barrier that matters): a single wave64.  A 256-lane workgroup is placed only
// when four wave slots of one CU are free at once; single waves fill the slots
// as they free up.  Measured on y = max(x, 0): 6.62 TB/s against 6.39 TB/s at
// 411 MB, 5.96 against 5.65 TB/s at 103 MB, 5.41 against 5.12 TB/s at 51 MB
// (128 lanes: no gain).
constexpr int kStream = 64;

#define SHDW_DEVICE __device__ __forceinline__

// Streaming accesses: whose cache lines one wave asks for, once.  Both directions
// carry the non-temporal hint; loads get it through these functions alone.
// Stores: a plain store leaves dirty lines in L2 that are written back when the
// kernel ends (broadcast of 67 MB of output 11.4 us with the hint, 13.0 to 19.2
// without; 103 MB copy 19.3 against 31.9).
// Loads: without the hint an operand that is new, or that the operator before has
// just written, arrives more slowly from 12 MB on, whatever the kernel: ReLU of 12.8 /
// 51 / 205 MB 5.1 / 17.0 / 62.6 us with it and 5.4 / 17.5 / 65.1 without, the sum of two of
// 51 MB 24.3 and 26.2, 7x7 averages of 205 MB 31.8 and 34.8, group norms of 205 MB 76.5 and
// 80.8; behind the kernel that wrote the operand the same (ReLU 16.9 and 17.8, sum 24.5 and
// 26.2).  Plain loads pay only where several operators read one tensor of up to 256 MB one
// after another (ReLU of 51 MB 15.6 against 16.6), which a kernel cannot know.
// load4 and load4_any below are for lines that are asked for more than once: operands that
// the kernel, or the call's next one, reads again (normalisation of 513 and more values in
// two walks, 103 MB: rows of 512 28.8 us plain, 32.9 with the hint, [16,4096,196] 73.7 and
// 86.7; SSDNormalize per item of [8,256,56,56] 18.6 and 20.3), and rows that start anywhere
// in a line where short pieces of them go to different waves (channel shuffle of 49-element
// rows, 103 MB: 20.9 us plain, 23.2 with the hint; the transposes in movers.hip; 3x3 pooling
// bands of 225-wide rows 122 and 133).
template <class T>
SHDW_DEVICE T load_stream(const T* p) {
  return __builtin_nontemporal_load(p);
}
SHDW_DEVICE v4f load4_stream(const float* p) { return load_stream(reinterpret_cast<const v4f*>(p)); }  // 128 bits
SHDW_DEVICE void store4_stream(float* p, v4f v) {
  __builtin_nontemporal_store(v, reinterpret_cast<v4f*>(p));
}
SHDW_DEVICE v4f load4(const float* p) { return *reinterpret_cast<const v4f*>(p); }

// The same for addresses that are only 4-byte aligned (Blas offsets, odd row
// lengths).  The hardware takes a 128-bit global access at any dword address
// and splits the ones that straddle a line; on aligned addresses it costs the
// same as the aligned form (61.7 us against 61.8 us for 411 MB), one dword off
// 73 us, where four 4-byte accesses per lane need 172 us.
typedef float v4f_unaligned __attribute__((ext_vector_type(4), aligned(4)));
SHDW_DEVICE v4f load4_stream_any(const float* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const v4f_unaligned*>(p));  // T would lose the alignment
}
SHDW_DEVICE v4f load4_any(const float* p) { return *reinterpret_cast<const v4f_unaligned*>(p); }
SHDW_DEVICE void store4_stream_any(float* p, v4f v) {
  __builtin_nontemporal_store(v, reinterpret_cast<v4f_unaligned*>(p));
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
SHDW_DEVICE bool aligned16_device(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// Workgroups are handed to the 8 XCDs (accelerator dies, each with its own L2)
// round-robin by blockIdx.x, so workgroups b and b + 1 never share an L2.  A
// kernel whose neighbouring work items touch the same cache lines (halo rows,
// rows that straddle a line) renumbers its workgroups with this map: XCD x then
// owns one contiguous range of work items and the shared lines are fetched from
// HBM once.  A bijection of [0, grid) for every grid size.
constexpr uint32_t kXcds = 8;
__host__ SHDW_DEVICE uint32_t xcd_contiguous(uint32_t block, uint32_t grid) {
  const uint32_t x = block % kXcds, slot = block / kXcds;
  const uint32_t q = grid / kXcds, r = grid % kXcds;
  return x * q + (x < r ? x : r) + slot;
}

// Between the two: XCD x gets runs of 2^log2_run consecutive work items (its
// workgroups b, b + 8, ... of one run), the runs of the eight XCDs interleaved.
// For kernels that stream and also write a few bytes per workgroup (a row's mean,
// a row's maximum): the workgroups whose small results share a cache line then
// complete that line in one L2, while the stream stays spread over all XCDs.  A
// bijection of [0, grid); the incomplete last span keeps its numbering.
__host__ SHDW_DEVICE uint32_t xcd_runs(uint32_t block, uint32_t grid, uint32_t log2_run) {
  const uint32_t span = kXcds << log2_run;
  if (block >= grid - grid % span) return block;
  const uint32_t turn = block / kXcds, xcd = block % kXcds;
  return (turn >> log2_run) * span + (xcd << log2_run) + (turn & ((1u << log2_run) - 1u));
}

// ---------------------------------------------------------------------------
// Division of a 31-bit unsigned value by a divisor fixed at launch time:
//   q = (mulhi(n, m) + n) >> s
// with s = ceil(log2 d), m = floor(2^32 (2^s - d) / d) + 1.  Exact for every
// n < 2^31 (the sum cannot wrap because mulhi(n, m) < 2^31).
// ---------------------------------------------------------------------------
struct FastDiv {
  uint32_t d = 1, m = 0, s = 0;
};

inline FastDiv make_fastdiv(uint32_t d) {
  FastDiv f;
  f.d = d;
  uint32_t s = 0;
  while ((1ull << s) < d) ++s;
  f.s = s;
  f.m = static_cast<uint32_t>(((1ull << 32) * ((1ull << s) - d)) / d + 1);
  return f;
}

SHDW_DEVICE uint32_t fd_div(uint32_t n, const FastDiv& f) {
  return (__umulhi(n, f.m) + n) >> f.s;
}
SHDW_DEVICE void fd_divmod(uint32_t n, const FastDiv& f, uint32_t& q, uint32_t& r) {
  q = fd_div(n, f);
  r = n - q * f.d;
}

// ---------------------------------------------------------------------------
// Division by a divisor that many dividends share.  t / d, correctly rounded, is the
// fp64 product t * r rounded to fp32, with r within 2^-52 of 1 / d: the product is then
// within 2^-51 of the quotient, and a quotient of two fp32 numbers that is a normal fp32
// number lies on no midpoint between two of them and no nearer to one than 2^-49 of its
// size (|A 2^k - M B| >= 1 for a dividend A, a divisor B of 24 bits and a midpoint M of 25).
// Subnormal quotients can lie on a midpoint: a wave that holds one divides.  Zeros in
// the dividends need no division; a wave looks twice before it divides for them.
// Four instructions an element where a division takes eleven, one of them at half rate.
// ---------------------------------------------------------------------------
// 1 / d in fp64: the hardware's estimate (2^-22 or better) and two Newton steps; as the
// estimate where those are undefined (0, infinite, NaN), so that t * r is t / d there too.
SHDW_DEVICE double reciprocal(float d) {
  const double dd = static_cast<double>(d), r0 = __builtin_amdgcn_rcp(dd);
  double r = __builtin_fma(__builtin_fma(-dd, r0, 1.0), r0, r0);
  r = __builtin_fma(__builtin_fma(-dd, r, 1.0), r, r);
  return r == r ? r : r0;
}

// t[j] / d[j] for N dividends of a lane, r[j] = reciprocal(d[j]); every lane of the wave
// that runs this must hold some dividend.
template <int N, class D, class R>
SHDW_DEVICE void quotients(float (&t)[N], D&& d, R&& r) {
  constexpr float kLeast = 0x1p-126f;
  float q[N];
#pragma unroll
  for (int j = 0; j < N; ++j) q[j] = static_cast<float>(static_cast<double>(t[j]) * r(j));
  float lo = __builtin_fabsf(q[0]);
#pragma unroll
  for (int j = 1; j < N; ++j) lo = __builtin_fminf(lo, __builtin_fabsf(q[j]));
  if (__builtin_amdgcn_ballot_w64(!(lo >= kLeast)) != 0) {
    bool whole = true;
#pragma unroll
    for (int j = 0; j < N; ++j) whole = whole && (t[j] == 0.f || __builtin_fabsf(q[j]) >= kLeast);
    if (__builtin_amdgcn_ballot_w64(!whole) != 0) {
      asm volatile("");  // keeps the compiler from evaluating both sides
#pragma unroll
      for (int j = 0; j < N; ++j) q[j] = t[j] / d(j);
    }
  }
#pragma unroll
  for (int j = 0; j < N; ++j) t[j] = q[j];
}
SHDW_DEVICE v4f quotients4(v4f t, float d, double r) {
  float q[4] = {t[0], t[1], t[2], t[3]};
  quotients(q, [d](int) { return d; }, [r](int) { return r; });
  return v4f{q[0], q[1], q[2], q[3]};
}

// ---------------------------------------------------------------------------
// wave64 exchange.  Steps 1..8 stay inside a row of 16 lanes and use DPP
// (no LDS traffic); 16 and 32 cross rows and go through ds_bpermute.
// ---------------------------------------------------------------------------
template <int CTRL>
SHDW_DEVICE int dpp_i32(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
SHDW_DEVICE float dpp_f32(float v) {
  return __int_as_float(dpp_i32<CTRL>(__float_as_int(v)));
}
template <int CTRL>
SHDW_DEVICE double dpp_f64(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = dpp_i32<CTRL>(static_cast<int>(b));
  const int hi = dpp_i32<CTRL>(static_cast<int>(b >> 32));
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}
// The lane in front's, 0 in lane 0: with a constant there the shift is an operand of the addition that
// follows, where dpp_f32 takes an instruction of its own, which the chain of a sum waits for (whole-plane
// averages of 512 x 12544 with signs 39.3 -> 29.4 us).
SHDW_DEVICE float lane_in_front(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
template <int CTRL>
SHDW_DEVICE uint32_t dpp_u32(uint32_t v) {
  return static_cast<uint32_t>(dpp_i32<CTRL>(static_cast<int>(v)));
}

constexpr int kDppXor1 = 0xB1;        // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;        // quad_perm [2,3,0,1]
constexpr int kDppWaveShr1 = 0x138;    // lane i takes lane i - 1
constexpr int kDppRor4 = 0x124;        // lane i takes lane i - 4 (modulo 16) inside 16
constexpr int kDppRor8 = 0x128;        // lane i <-> i + 8 (modulo 16) inside 16
constexpr int kDppHalfMirror = 0x141;  // lane i <-> 7-i inside 8
constexpr int kDppMirror = 0x140;      // lane i <-> 15-i inside 16

}  // namespace shdw

#endif  // SHADOW_AMD_CSRC_DEVICE_COMMON_H_
