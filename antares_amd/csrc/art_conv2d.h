// What the convolution kernels share: element types, sizes, and the place of an output point in the padded image.
#pragma once
#include "art_common.h"

namespace art {
namespace conv {

constexpr int kThreads = 256;
constexpr int kTaps = 9;                        // 3 x 3
constexpr int kChunkBytes = 64;                 // channels of a point that are staged at a time

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <typename T> struct Elem;
template <> struct Elem<_Float16> {
  typedef _Float16 vec __attribute__((ext_vector_type(8)));
  typedef unsigned short raw;
  static __device__ __forceinline__ f32x16 multiply(vec a, vec b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
template <> struct Elem<float> {
  typedef float vec __attribute__((ext_vector_type(4)));
  typedef float raw;
  // instruction m multiplies k = m (lanes 0-31) and k = 4 + m (lanes 32-63) of 8
  static __device__ __forceinline__ f32x16 multiply(vec a, vec b, f32x16 c, int first = 0, int last = 4) {
#pragma unroll
    for (int m = first; m < last; ++m) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[m], b[m], c, 0, 0, 0);
    return c;
  }
};

struct Geometry {
  int N, C, H, W, F, HO, WO, ph, pw;
  int columns;          // output points: N * HO * WO
  int chunks;           // runs of 64 bytes of channels
  int row_tiles;        // 32-feature tiles of the packed filter
  int row_blocks;       // blocks along the features
  int span;             // points the LDS buffers hold
};

// Output point -> its place in the padded image (where tap (0, 0) reads).
__device__ __forceinline__ int place_of(int column, const Geometry& g) {
  const unsigned hw = (unsigned)(g.HO * g.WO), n = (unsigned)column / hw, r = (unsigned)column % hw;
  const unsigned ho = r / (unsigned)g.WO, wo = r % (unsigned)g.WO;
  return (int)((n * (unsigned)(g.HO + 2) + ho) * (unsigned)(g.WO + 2) + wo);
}

// Forms 4 to 7 (art_conv2d_staged.hip): blocks of 64 features x 64 points, 64 x 128, 128 x 128, and 64 x 64 with short sums (float32
// only), over a copy of the image that is laid out for them.  `packed` takes the filter, behind it the image, and behind that the results of the slices of channels.
size_t staged_bytes(const Geometry& g, int slices);
size_t staged_lds(const Geometry& g);
int run_staged(const void* x, const void* w, void* packed, void* y, const Geometry& g, int f16, int form, int slices, int blocks, hipStream_t stream);

}  // namespace conv

// y[i] = sum over slices of partial[slice * count + i], in order and in float64 (art_gemm_tile.hip).
int sum_slices(const float* partial, float* y, long long count, int slices, hipStream_t stream);

}  // namespace art
