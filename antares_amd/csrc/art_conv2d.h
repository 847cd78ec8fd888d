// What the convolution kernels share: element types, sizes, and the place of an output point in the padded image.
#pragma once
#include "art_common.h"

namespace art {
namespace conv {

using ::art::Div;
using ::art::make_div;
using ::art::over;

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
  Div results, width;   // output points of an image, of a row
  Div image, wide;      // padded points of an image, of a row
  Div blocks_across;    // row_blocks
};

// Output point -> its place in the padded image (where tap (0, 0) reads).
__device__ __forceinline__ int place_of(int column, const Geometry& g) {
  const unsigned n = over((unsigned)column, g.results), r = (unsigned)column - n * g.results.by, ho = over(r, g.width), wo = r - ho * g.width.by;
  return (int)((n * (unsigned)(g.HO + 2) + ho) * g.wide.by + wo);
}

// A wavefront's tiles to memory: accumulator element e is feature f0 + (e / 4) * 8 + (lane / 32) * 4 + e % 4 of the tile, point
// lane % 32 at to[j].  One addition per store: worked out anew each time, the addresses were a quarter of the kernels' code.
template <int MT, int NT>
__device__ __forceinline__ void store_results(const f32x16 (&total)[MT][NT], float* y, const size_t (&to)[NT], int column, int last, int f_first, const Geometry& g) {
  const int hl = (threadIdx.x & 63) >> 5;
  const size_t plane = g.results.by;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    if (column + j * 32 > last) continue;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int f0 = f_first + i * 32;
      float* p = y + to[j] + (size_t)(f0 + hl * 4) * plane;
      if (f0 + 32 <= g.F) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          __builtin_nontemporal_store(total[i][j][e], p);
          p += (e & 3) == 3 ? 5 * plane : plane;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          if (f0 + (e >> 2) * 8 + hl * 4 + (e & 3) < g.F) __builtin_nontemporal_store(total[i][j][e], p);
          p += (e & 3) == 3 ? 5 * plane : plane;
        }
      }
    }
  }
}

// Forms 4 to 7 (art_conv2d_staged.hip): blocks of 64 features x 64 points, 64 x 128, 128 x 128, and 64 x 64 with short sums (float32
// only), over a copy of the image that is laid out for them.  `packed` takes the filter, behind it the image, and behind that the results of the slices of channels.
// The copy holds the images of a pass, kMostCopy bytes of them (or one image).
constexpr size_t kMostCopy = 128 << 20;
int images_of_pass(const Geometry& g);
size_t staged_bytes(const Geometry& g, int slices);
size_t staged_lds(const Geometry& g);
int run_staged(const void* x, const void* w, void* packed, void* y, const Geometry& g, int f16, int form, int slices, hipStream_t stream);

// Forms 8 to 10 (art_conv2d_direct.hip): blocks of 16 features x 16, 32 or 64 points over all channels, in one launch, without copies.
bool direct_fits(const Geometry& g, int f16, int form);
double direct_time(const Geometry& g, int f16, int form);
int run_direct(const void* x, const void* w, void* y, const Geometry& g, int f16, int form, hipStream_t stream);

}  // namespace conv

// y[i] = sum over slices of partial[slice * count + i], in order and in float64 (art_gemm_tile.hip).
int sum_slices(const float* partial, float* y, long long count, int slices, hipStream_t stream);

}  // namespace art
