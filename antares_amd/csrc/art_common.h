// Shared helpers of libantares_amd.so: error reporting and launch checks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <string>

#include "../../include/antares_amd.h"

namespace art {

std::string& last_error();
int fail(const char* fmt, ...) __attribute__((format(printf, 1, 2)));

struct Workspace {
  void* base = nullptr;      // device memory
  size_t bytes = 0;
};
// Workspace of (current device, stream).  Launches on one stream are ordered, so they can share partial-result
// memory; launches on different streams are not, so every stream gets a workspace of its own, allocated and zeroed
// the first time the stream is seen (up to kMaxStreamsPerDevice streams per device; that first use must not happen
// while the stream is being captured into a graph, because it allocates).  Returns nullptr with the error set.
Workspace* workspace(hipStream_t stream);
int release_stream(hipStream_t stream);
constexpr int kMaxStreamsPerDevice = 40;      // torch hands out 32 pooled streams per device besides the default one

// Looks up, for the current device, the address of the scratch array built into the code object (used by
// art_gemv_w4a16_noalloc).  Called once per device by art_init.
int gemv_noalloc_setup(int device);

// Compute units of the current device (queried once per device).
int compute_units();

// Blocks per head the split decode attention may use, shared by its producer (art_llm.hip) and the projection that
// merges the per-part records (art_gemv_w4.hip).
constexpr int kMaxAttnParts = 8;

// True when the byte ranges [a, a + an) and [b, b + bn) overlap.
inline bool overlaps(const void* a, size_t an, const void* b, size_t bn) {
  const uintptr_t a0 = (uintptr_t)a, b0 = (uintptr_t)b;
  return a0 < b0 + bn && b0 < a0 + an;
}

// Workspace layout.  The exchange words and the accumulators keep their meaning between launches,
// so they never share bytes with scratch data.
constexpr size_t kExchangeOffset = 0;                    // launch tag + one word per block of the phase-chain probe (tagged, never zeroed again)
constexpr size_t kExchangeBytes = 64 * 1024;
constexpr size_t kSlotOffset = 64 * 1024;                // 64-bit split-K accumulators (zero between launches)
constexpr size_t kScratchOffset = 4 * 1024 * 1024;       // partial sums, tile counts (any content)

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
constexpr unsigned int kBufferFlags = 0x00020000u;       // word 3 of a buffer descriptor: 32-bit data

// 64 lanes x 16 bytes from base + lane offset straight into LDS at lds_dst + 16 * lane.  The instruction takes
// the LDS address from m0, which nothing else here uses (the compiler warns that it does not preserve a reserved register
// that is named as clobbered; nothing has to be preserved).  The waits are written by hand: the compiler does not see
// these loads.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_lds_x4(const void* base, unsigned int off, unsigned int lds_dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_dst) : "m0");
}
// The same, 16 or 4 bytes a lane, from base + scalar offset + lane offset, the base in a buffer descriptor (buffer_of); LDS address: a scalar plus a constant.
// Nothing but the scalar offset has to move on from one load to the next.
template <unsigned LDS> __device__ __forceinline__ void buffer_lds_x4(u32x4_t buffer, unsigned int off, unsigned int scalar_off, unsigned int lds) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %4 offen lds" ::"v"(off), "s"(buffer), "s"(lds), "n"(LDS), "s"(scalar_off) : "m0", "scc");
}
template <unsigned LDS> __device__ __forceinline__ void buffer_lds_x1(u32x4_t buffer, unsigned int off, unsigned int scalar_off, unsigned int lds) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dword %0, %1, %4 offen lds" ::"v"(off), "s"(buffer), "s"(lds), "n"(LDS), "s"(scalar_off) : "m0", "scc");
}
#pragma clang diagnostic pop

// Descriptor of a plain buffer that starts at an address uniform over the wavefront: no stride, no limit but 4 GiB.
__device__ __forceinline__ u32x4_t buffer_of(const void* p) {
  const unsigned long long v = (unsigned long long)p;
  return u32x4_t{(unsigned int)__builtin_amdgcn_readfirstlane((int)v), (unsigned int)__builtin_amdgcn_readfirstlane((int)(v >> 32)) & 0xffffu, 0xffffffffu,
                 kBufferFlags};
}

// The unit of block b when runs of 2^shift units go round the eight XCDs (block b runs on XCD b % 8), for a multiple of 8 << shift units;
// shift 0: unit b.
__device__ __forceinline__ int unit_of_runs(int b, int shift) {
  const int i = b >> 3;
  return (i >> shift << (shift + 3)) + ((b & 7) << shift) + (i & ((1 << shift) - 1));
}

// A base address that is the same for every lane, in scalar registers whatever surrounds the load.
__device__ __forceinline__ const void* uniform(const void* p) {
  const unsigned long long v = (unsigned long long)p;
  return (const void*)((unsigned long long)(unsigned int)__builtin_amdgcn_readfirstlane((int)v) |
                       (unsigned long long)(unsigned int)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32);
}

// x / d for x below 2^30: x * mul >> shift with mul = ceil(2^shift / d), shift = 30 + ceil(log2 d).
struct Div {
  unsigned int mul, shift, by;
};
inline Div make_div(unsigned int d) {
  const unsigned int s = d > 1 ? 32 - __builtin_clz(d - 1) : 0;
  return Div{(unsigned int)(((1ull << (30 + s)) + d - 1) / d), 30 + s, d};
}
__device__ __forceinline__ unsigned int over(unsigned int x, const Div& d) { return (unsigned int)((unsigned long long)x * d.mul >> d.shift); }

// g / (1 + e^-g) of a value that fp16 holds.  t, g times log2(e) cut to 13 bits, is exact; e^-g = 2^n 2^(t - n + the rest).
// The quotient is corrected once; numerator and denominator are divided by 16, so that its reciprocal stays a normal
// number.  Zeros, infinities and NaN come out as of the division itself (-infinity: NaN).
__device__ __forceinline__ float silu(float g) {
  const float at = __builtin_amdgcn_fmed3f(g, -96.0f, 96.0f), t = at * -1.442626953125f, n = rintf(t);
  const float e = ldexpf(__builtin_amdgcn_exp2f(fmaf(at, -6.8087776e-5f, t - n)), (int)n);
  const float num = g * 0.0625f, den = fmaf(e, 0.0625f, 0.0625f), r = __builtin_amdgcn_rcpf(den), q = num * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(0.0f - den, q, num), r, q), den, num);
}

}  // namespace art

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every outstanding
// global load of the wave (vmcnt(0)), which drains register prefetches at each barrier; this one
// leaves them in flight.  Use it only where the data exchanged through the barrier lives in LDS.
__device__ __forceinline__ void art_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

#define ART_HIP(expr)                                                                   \
  do {                                                                                  \
    hipError_t _e = (expr);                                                             \
    if (_e != hipSuccess)                                                               \
      return art::fail("%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), __FILE__, __LINE__); \
  } while (0)

#define ART_REQUIRE(cond, ...)            \
  do {                                    \
    if (!(cond)) return art::fail(__VA_ARGS__); \
  } while (0)

#define ART_LAUNCH_CHECK()                                                                \
  do {                                                                                    \
    hipError_t _e = hipGetLastError();                                                    \
    if (_e != hipSuccess)                                                                 \
      return art::fail("kernel launch failed: %s (%s:%d)", hipGetErrorString(_e), __FILE__, __LINE__); \
  } while (0)
