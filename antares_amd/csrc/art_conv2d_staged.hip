// 3 x 3 convolutions over a staged image (see art_conv2d.hip for the operation and the other kernel): a first launch packs the
// filter and copies the image with the channels of a point side by side, the second one multiplies.
//
// Why: the kernel that gathers the image as it lies in memory spends most of its time before its first product - its code is
// 12 to 20 KiB, run once, and every staged point takes divisions, comparisons and 2- or 4-byte loads.
// With nothing but the products left in its loop it still took 16.2 of 21.8 us at float16 32 x 128 x 28 x 28 -> 128.  Here
//   * the copy holds the image padded to HO + 2 rows of WO + 2 points, [64 bytes of channels][point][64 bytes], zeros where the
//     image or its channels end.  It is made by the launch that packs the filter anyway;
//   * a block's run of points is then contiguous per chunk of channels and goes straight into LDS (global_load_lds, 16 bytes per
//     lane, no registers, no arithmetic), into a ring of three chunks, two chunks ahead of its use.  The 16-byte pieces of
//     point p are swapped by (p / 4) % 4, on the way in by the lane's global address, so that 16 neighbouring points are read
//     from all banks;
//   * a tap is a constant number of points added to a lane's point; the filter comes from L2 straight into registers, several
//     taps ahead;
//   * stores run over the features with one addition each;
//   * few blocks: the chunks of channels are cut into slices, whose results a third launch adds;
//   * the copy takes 128 MiB at the most: larger batches go in passes of as many images as fit.
// Measured, all launches, against what ran before (the gathering kernel or the generic lowering), us: float16 1 x 40 x 42 x 42 -> 152
// 10.1 -> 9.0, 2 x 40 x 12 x 12 -> 64 9.6 -> 7.9, 9 x 240 x 13 x 13 -> 104 19.4 -> 13.8, 3 x 184 x 51 x 51 -> 184 23.6 -> 19,
// 32 x 128 x 28 x 28 -> 128 22.7 -> 21.7 (6 to 7 of them the copy of 7 MB, 13 the products: four chunks of 1.3 us, code, first
// loads and stores); float32 9 x 216 x 17 x 17 -> 64 23 -> 20, 5 x 72 x 21 x 21 -> 48 20 -> 13.5, 2 x 232 x 52 x 52 -> 24 375 -> 37.
// Geometric mean over 116 and 214 sizes 1.4 times as fast.  Bound by latency below some 15 us: the first launch 3 us, 1 us (float16) or
// 2.7 us (float32, the matrix instructions) per chunk.
#include "art_conv2d.h"

namespace {

using namespace art::conv;
using art::load_lds_x4;
using art::uniform;

struct Staged {
  Geometry g;
  int places;                // padded points in all
  int filter_blocks, place_blocks;
  const char* image_copy;
  Div blocks;                // blocks of a slice of the chunks
  int slices, slice_chunks, longer;      // chunks of a slice; the first `longer` slices have one more
  long long results_all;     // N * F * HO * WO
  int half_last;             // of the last chunk only the lower half of the channels exists
};

// Blocks in front: filter [F][C][taps] -> [chunk][tap][32 features][half][lane][16 bytes], zeros past F and C.  The others: 64 points of
// a chunk of channels, a wavefront per 16 bytes of them.  Bound by latency for small images, by memory for large ones.
template <typename T>
__global__ __launch_bounds__(kThreads) void conv2d_stage_kernel(const T* __restrict__ x, const T* __restrict__ w, T* __restrict__ packed, T* __restrict__ copy, Staged s) {
  constexpr int V = 16 / sizeof(T);
  typedef typename Elem<T>::vec vec;
  const Geometry& g = s.g;
  if ((int)blockIdx.x < s.filter_blocks) {
    const int id = blockIdx.x * kThreads + threadIdx.x;
    if (id >= g.chunks * kTaps * g.row_tiles * 128) return;
    const int lane = id & 63, half = (id >> 6) & 1;
    const unsigned rest = (unsigned)(id >> 7);
    const int r = (int)(rest % (unsigned)g.row_tiles);
    const unsigned qt = rest / (unsigned)g.row_tiles;
    const int t = (int)(qt % (unsigned)kTaps), q = (int)(qt / (unsigned)kTaps);
    const int f = r * 32 + (lane & 31), c0 = (q * 4 + half * 2 + (lane >> 5)) * V;
    vec v;
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = (f < g.F && c0 + j < g.C) ? w[((size_t)f * g.C + c0 + j) * kTaps + t] : (T)0;
    reinterpret_cast<vec*>(packed)[id] = v;
    return;
  }
  __shared__ __align__(16) vec turned[64 * 4];          // the points' pieces meet here, so that the stores are whole lines
  const int b = blockIdx.x - s.filter_blocks, q = b / s.place_blocks, piece = threadIdx.x >> 6, local = threadIdx.x & 63;
  const unsigned place = (unsigned)(b - q * s.place_blocks) * 64 + local;
  const unsigned n = over(place, g.image), r = place - n * g.image.by, ph = over(r, g.wide);
  const int h = (int)ph - g.ph, wc = (int)(r - ph * g.wide.by) - g.pw, c0 = (q * 4 + piece) * V;
  const bool in = place < (unsigned)s.places && h >= 0 && h < g.H && wc >= 0 && wc < g.W;
  const size_t plane = (size_t)g.H * g.W;
  const T* from = x + (in ? ((size_t)n * g.C * g.H + h) * g.W + wc : 0);
  T held[V];
#pragma unroll
  for (int j = 0; j < V; ++j) held[j] = from[(c0 + j < g.C ? c0 + j : g.C - 1) * plane];       // the same channel in all lanes
  vec v;
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] = in && c0 + j < g.C ? held[j] : (T)0;
  turned[local * 4 + (piece ^ (local >> 2 & 3))] = v;
  __syncthreads();
  const int point = threadIdx.x >> 2;
  const unsigned to = place - local + point;
  if (to < (unsigned)s.places) reinterpret_cast<vec*>(copy)[((size_t)q * s.places + to) * 4 + (threadIdx.x & 3)] = turned[point * 4 + ((threadIdx.x & 3) ^ (point >> 2 & 3))];
}

// MT, NT: 32 x 32 tiles of a wavefront along features and points, 2 x 2 wavefronts.  FINE (float32, one tile): four products by
// themselves, these sums in pairs to a tap's half, a tap and a row of taps, and the rows in float64.
template <typename T, int MT, int NT, bool FINE>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, MT == 2 ? 2 : 4))) void conv2d_staged_kernel(const T* __restrict__ packed, float* __restrict__ y, Staged s) {
  typedef typename Elem<T>::vec vec;
  constexpr int TN = 64 * NT;
  constexpr int kSets = MT == 1 ? kTaps : 3, kAhead = kSets - 1;    // taps of the filter in registers
  constexpr int kFilterLoads = kTaps * MT * 2;                      // of a wavefront and chunk
  constexpr int kLook = MT == 2 ? 2 : 4;                            // taps whose points are in registers
  constexpr int kSum = MT == 1 && NT == 1 ? 3 : kTaps;            // taps summed by themselves
  extern __shared__ __align__(16) char lds[];
  const Geometry& g = s.g;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, hl = lane >> 5;
  // workgroups go to the eight XCDs round robin: an XCD gets a contiguous run of blocks
  const int per = gridDim.x >> 3, left = gridDim.x & 7, xcd = blockIdx.x & 7;
  const int block = xcd * per + (xcd < left ? xcd : left) + (blockIdx.x >> 3);
  const int slice = (int)over((unsigned)block, s.blocks), in_slice = block - slice * (int)s.blocks.by, run = (int)over((unsigned)in_slice, g.blocks_across);
  const int chunk0 = slice * s.slice_chunks + (slice < s.longer ? slice : s.longer), chunks = s.slice_chunks + (slice < s.longer ? 1 : 0);
  const int rb = in_slice - run * (int)g.blocks_across.by, column0 = run * TN;
  const int last = (column0 + TN < g.columns ? column0 + TN : g.columns) - 1;
  const int wide = (int)g.wide.by, place0 = place_of(column0, g);
  const int units = (place_of(last, g) - place0 + 2 * wide + 3 + 15) >> 4;          // 16 points = 1 KiB of a chunk
  const unsigned buffer = (unsigned)((g.span + 15) >> 4) << 10;                   // bytes of a chunk's points
  const size_t chunk_bytes = (size_t)s.places * kChunkBytes;
  const char* image = s.image_copy + (size_t)place0 * kChunkBytes + (size_t)chunk0 * chunk_bytes;
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds;
  // lane l brings 16 bytes of point l / 4 of a unit: piece (l % 4) ^ (l / 16) goes to where piece l % 4 would be
  const unsigned piece = (unsigned)((lane >> 2) * kChunkBytes + ((lane & 3) ^ (lane >> 4)) * 16);
  auto bring = [&](int q, unsigned slot, int first, int step) {      // this wavefront's units of a chunk; past the last chunk that one again
    const char* from = image + (size_t)(q < chunks ? q : chunks - 1) * chunk_bytes;
    for (int u = first; u < units; u += step) load_lds_x4(uniform(from), piece + (unsigned)u * 1024, lds0 + slot + (unsigned)u * 1024);
  };

  // the filter: 64 x 16 bytes per 32 features, half and tap
  const int filter_taps = chunks * kTaps;
  const size_t filter_step = (size_t)g.row_tiles * 128 * 16;
  const char* filter = reinterpret_cast<const char*>(packed) + ((size_t)rb * 2 + wm) * MT * 128 * 16 + lane * 16 + (size_t)chunk0 * kTaps * filter_step;
  vec a[kSets][MT][2];
  auto fetch_filter = [&](int set, int tap) {
    const char* p = filter + (size_t)(tap < filter_taps ? tap : filter_taps - 1) * filter_step;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) a[set][i][h] = *reinterpret_cast<const vec*>(p + (i * 2 + h) * 1024);
  };

  bring(0, 0, wave, 4);
  asm volatile("" ::: "memory");
#pragma unroll
  for (int t = 0; t < kAhead; ++t) fetch_filter(t, t);
  asm volatile("" ::: "memory");
  bring(1, buffer, wave, 4);

  // this lane's output points: their place in the block's run, and where the result goes
  unsigned at[NT];
  size_t to[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    int column = column0 + wn * 32 * NT + j * 32 + (lane & 31);
    if (column > last) column = last;
    at[j] = (unsigned)(place_of(column, g) - place0);
    const unsigned n = over((unsigned)column, g.results);
    to[j] = (size_t)n * g.F * g.results.by + ((unsigned)column - n * g.results.by);
  }

  double fine[FINE ? 16 : 1] = {};
  f32x16 total[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) total[i][j] = f32x16(0);

  // everything but the filter's first taps and chunk 1 has arrived once only as many loads are left as were issued behind it
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAhead * MT * 2) : "memory");
  art_lds_barrier();
  unsigned cur = 0, next = buffer, fill = 2 * buffer;
#pragma unroll 1
  for (int q = 0; q < chunks; ++q) {
    const bool full = MT == 2 || !s.half_last || chunk0 + q + 1 < g.chunks;
    // a chunk (one tile per wavefront: a row of taps before that) is summed by itself and then joins the total
    f32x16 acc[MT][NT], row[MT][NT];
    vec b[kLook][2][NT];
    auto look = [&](int t) {                          // both halves of the points of a tap
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const unsigned p = at[j] + (unsigned)((t / 3) * wide + t % 3);
        const unsigned o = cur + p * kChunkBytes + (((unsigned)hl * 16) ^ (p * 4 & 48));
        b[t % kLook][0][j] = *reinterpret_cast<const vec*>(lds + o);
        b[t % kLook][1][j] = *reinterpret_cast<const vec*>(lds + (o ^ 32));
      }
    };
#pragma unroll
    for (int t = 0; t < kLook - 1; ++t) look(t);
#pragma unroll
    for (int t = 0; t < kTaps; ++t) {
      if (t < 8) bring(q + 2, fill, wave + 4 * t, t == 7 ? 4 : 1 << 20);           // a unit at a time; what is left with the last
      fetch_filter((t + kAhead) % kSets, q * kTaps + t + kAhead);
      if (t + kLook - 1 < kTaps) look(t + kLook - 1);
      __builtin_amdgcn_sched_barrier(0);              // left to the scheduler, the loads sink to their use
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h == 1 && !full) break;
        if constexpr (FINE) {
          const vec x = a[t % kSets][0][h], p = b[t % kLook][h][0];
          const f32x16 step = Elem<T>::multiply(x, p, f32x16(0), 0, 2) + Elem<T>::multiply(x, p, f32x16(0), 2, 4);
          acc[0][0] = h == 0 ? step : acc[0][0] + step;
          continue;
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            row[i][j] = Elem<T>::multiply(a[t % kSets][i][h], b[t % kLook][h][j], h == 0 && t % kSum == 0 ? f32x16(0) : row[i][j]);
      }
      if constexpr (FINE) row[0][0] = t % kSum == 0 ? acc[0][0] : row[0][0] + acc[0][0];
      if (t % kSum != kSum - 1) continue;
      if constexpr (FINE) {
#pragma unroll
        for (int e = 0; e < 16; ++e) fine[e] += (double)row[0][0][e];
        continue;
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = t < kSum ? row[i][j] : acc[i][j] + row[i][j];
    }
#pragma unroll
    for (int i = 0; i < MT && !FINE; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) total[i][j] += acc[i][j];
    // chunk q + 1 was asked for before any load of this chunk, and more than the filter's loads were issued in it
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFilterLoads) : "memory");
    art_lds_barrier();
    const unsigned freed = cur;
    cur = next;
    next = fill;
    fill = freed;
  }
  if constexpr (FINE)
#pragma unroll
    for (int e = 0; e < 16; ++e) total[0][0][e] = (float)fine[e];
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // nothing of the ring is on its way when its space is given back

  store_results<MT, NT>(total, y + slice * s.results_all, to, column0 + wn * 32 * NT + (lane & 31), last, ((rb * 2 + wm) * MT) * 32, g);
}

size_t filter_bytes(const Geometry& g) { return ((size_t)g.chunks * kTaps * ((g.F + 127) / 128) * 4 * 2048 + 255) & ~(size_t)255; }
size_t places_of(const Geometry& g, int images) { return (size_t)images * (g.HO + 2) * (g.WO + 2); }
// the last unit of 16 points may reach 15 points past the copy
size_t copy_bytes(const Geometry& g, int images) { return ((size_t)g.chunks * places_of(g, images) * kChunkBytes + 1024 + 255) & ~(size_t)255; }

template <typename T, int MT, int NT, bool FINE = false>
int launch(const void* packed, void* y, const Staged& s, hipStream_t st) {
  const size_t bytes = art::conv::staged_lds(s.g);
  static size_t configured = 0;
  if (bytes > configured) {
    ART_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(conv2d_staged_kernel<T, MT, NT, FINE>), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    configured = 160 * 1024;
  }
  conv2d_staged_kernel<T, MT, NT, FINE><<<dim3((unsigned)s.blocks.by * s.slices), dim3(kThreads), bytes, st>>>((const T*)packed, (float*)y, s);
  ART_LAUNCH_CHECK();
  return 0;
}

// One pass over s.g.N images, the first ones of x and y; `images`: the most of a pass, which the copy has room for.
template <typename T>
int run(const void* x, const void* w, void* packed, void* y, Staged& s, int form, int images, hipStream_t st) {
  const Geometry& g = s.g;
  T* copy = reinterpret_cast<T*>((char*)packed + filter_bytes(g));
  s.image_copy = (const char*)copy;
  conv2d_stage_kernel<T><<<dim3((unsigned)(s.filter_blocks + s.place_blocks * g.chunks)), dim3(kThreads), 0, st>>>((const T*)x, (const T*)w, (T*)packed, copy, s);
  ART_LAUNCH_CHECK();
  float* partial = reinterpret_cast<float*>((char*)packed + filter_bytes(g) + copy_bytes(g, images));
  void* to = s.slices > 1 ? partial : y;
  if (form == 4 ? launch<T, 1, 1>(packed, to, s, st) : form == 5 ? launch<T, 1, 2>(packed, to, s, st)
      : form == 6 ? launch<T, 2, 2>(packed, to, s, st) : launch<T, 1, 1, sizeof(T) == 4>(packed, to, s, st))
    return 1;
  return s.slices > 1 ? art::sum_slices(partial, (float*)y, s.results_all, s.slices, st) : 0;
}

}  // namespace

int art::conv::images_of_pass(const Geometry& g) {
  const size_t images = kMostCopy / ((size_t)g.chunks * places_of(g, 1) * kChunkBytes);
  return images < 1 ? 1 : images < (size_t)g.N ? (int)images : g.N;
}
size_t art::conv::staged_bytes(const Geometry& g, int slices) {
  const int images = images_of_pass(g);
  return filter_bytes(g) + copy_bytes(g, images) + (slices > 1 ? (size_t)slices * images * g.results.by * g.F * sizeof(float) : 0);
}
size_t art::conv::staged_lds(const Geometry& g) { return (size_t)((g.span + 15) / 16) * 3 * 1024; }

int art::conv::run_staged(const void* x, const void* w, void* packed, void* y, const Geometry& g, int f16, int form, int slices, hipStream_t stream) {
  Staged s{};
  s.g = g;
  s.filter_blocks = (g.chunks * kTaps * g.row_tiles * 128 + kThreads - 1) / kThreads;
  s.slices = slices;
  s.slice_chunks = g.chunks / slices;
  s.longer = g.chunks % slices;
  const int per_chunk = f16 ? 32 : 16, points = form == 4 || form == 7 ? 64 : 128, images = images_of_pass(g);
  s.half_last = g.C - (g.chunks - 1) * per_chunk <= per_chunk / 2;
  // Passes follow each other on the stream: each overwrites the copy (and the slices' results) of the one before it.
  for (int n = 0; n < g.N; n += images) {
    s.g.N = g.N - n < images ? g.N - n : images;
    s.g.columns = s.g.N * (int)g.results.by;
    s.places = (int)places_of(g, s.g.N);
    s.place_blocks = (s.places + 63) / 64;
    s.blocks = make_div((unsigned)((s.g.columns + points - 1) / points * g.row_blocks));
    s.results_all = (long long)s.g.columns * g.F;
    const void* from = (const char*)x + (size_t)n * g.C * g.H * g.W * (f16 ? 2 : 4);
    void* to = (float*)y + (size_t)n * g.results.by * g.F;
    if (f16 ? run<_Float16>(from, w, packed, to, s, form, images, stream) : run<float>(from, w, packed, to, s, form, images, stream)) return 1;
    s.filter_blocks = 0;                              // it stays where the first pass packed it
  }
  return 0;
}
