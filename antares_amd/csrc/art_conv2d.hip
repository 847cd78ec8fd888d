// 3 x 3 convolution, stride 1, NCHW image and FCHW filter, float32 sums, on the gfx950 matrix cores:
//
//   y[n, f, ho, wo] = sum over c, kh, kw of x[n, c, ho + kh - ph, wo + kw - pw] * w[f, c, kh, kw]        (0 outside x)
//
// Replaces, for these programs (AntaresIR.md:166), what the reference's tiled schedule generates
// (backends/c-rocm/schedule/standard/algo_tiling.py:35-98).
//
// Design for MI355X.  As a matrix product (features x output points, k = channels x taps) the operation is bound by the
// matrix cores, but a kernel that gathers the image once per tap is bound by the gathering: it fetches every image value
// nine times in pieces of one element, with an address and two comparisons each.  Here:
//   * the output points of a block (64 or 128 in a row of n, ho, wo) need one CONTIGUOUS run of points of the image
//     padded to HO + 2 rows of WO + 2: the run is staged in LDS once per 64 bytes of channels (32 float16 or
//     16 float32), as [point][channel], and a tap is a constant number of points added to a lane's LDS address.  Global
//     reads run along the points, two of them per lane (a wavefront reads 128 from one channel; rows of the padded image are of an even
//     number, so that both are in one row): what bounds a chunk beside its products is the number of these loads and of the lines
//     that each touches.  16-byte LDS writes put a lane's 8 or 4 channels side by side; 80 bytes from point to point keep reads
//     and writes on distinct banks.  Against a point per load, padding read from the first point of the image, and all loads
//     with the first three taps (one card, us; in float16 with the scalar bases below): float16 32 x 128 x 28 x 28 -> 128 18.3 -> 16.0, 32 x 256 x 14 x 14 -> 256
//     28.0 -> 22.6, 16 x 256 x 28 x 28 -> 256 31.1 -> 26.7, 26 x 120 x 37 x 37 -> 32 18.7 -> 17.9; float32 32 x 128 x 28 x 28 -> 128 79.8 -> 78.2;
//   * the offset of each pair of points, and which of them are inside, is worked out once per block;
//   * the filter is packed first, by a launch of its own, in the order in which wavefronts feed it to the matrix
//     instructions: [64 bytes of channels][tap][32 features][half][lane] with 16 bytes per lane, so that a wavefront's
//     operand is one contiguous kilobyte that comes from L2 straight into registers, a tap ahead of its use;
//   * the next 64 bytes of channels travel to registers while these are multiplied, a few loads with every tap, two LDS buffers, one LDS-only barrier
//     per 64 bytes of channels (18 to 72 matrix instructions per wavefront and barrier for a 3 x 3 filter, not 2 to 8);
//   * a last chunk of which only the lower half exists is multiplied without the upper half (64-feature blocks): float32
//     20 x 24 -> 64, 20 x 20 12.0 -> 10.5 us (generic 11.4), float16 19 x 19 of 16 channels 8.8 -> 7.3 (7.7 to 8.4);
//   * 2 x 2 wavefronts of MT x NT tiles of 32 features x 32 points; blocks of one run of points are neighbours on one XCD.
// Measured, padding 1, both launches, against the generic lowering (a padded copy, then a gathering product): float16
// 32 x 128 x 28 x 28 -> 128 40.2 -> 16.0 us, 24 x 200 x 33 x 33 -> 48 89 -> 23 us, 2 x 160 x 18 x 18 -> 64 57 -> 14 us;
// float32 32 x 128 x 28 x 28 -> 128 113 -> 78 us (the matrix instructions alone take 47), 23 x 128 x 30 x 30 -> 176 119 -> 86.
// The first of these, before its loads had scalar bases (17 us; clocks of a block, 27500 in all at 2.1 GHz; its products alone are 9200): 1150 for the places, 3700 until the first
// image is in LDS, three chunks of 5150 and the last of 3400 (2600 without the filter's loads, which half fill the load path), 2900 for
// the stores of 12.8 MB; packing the filter takes 2.3 us.  Without effect: the filter nine taps ahead, and blocks of four wavefronts
// along the features, which load the filter once and read each point four times from LDS.
// Today it is taken for large images with little to multiply (`choose`); art_conv2d_staged.hip stages the image first.
#include <type_traits>

#include "art_conv2d.h"

namespace {

using namespace art::conv;

constexpr int kPitchBytes = kChunkBytes + 16;   // from one point to the next in LDS
#define ART_GLOBAL __attribute__((address_space(1)))
constexpr unsigned kFirst = 1u, kSecond = 0x80000000u;         // flags beside an offset into x: below 2^31 and even
constexpr size_t kMaxLds = 64 * 1024, kWideLds = 160 * 1024;     // with more than the first a compute unit holds one block

// Filter [F][C][taps] -> [chunk][tap][32 features][half][lane][16 bytes], zeros past F and C.  A thread gathers the 16
// bytes of one lane; bound by latency (about 2 us).
template <typename T>
__global__ __launch_bounds__(kThreads) void conv2d_pack_kernel(const T* __restrict__ w, T* __restrict__ packed, Geometry g) {
  constexpr int V = 16 / sizeof(T);
  const long long id = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (id >= (long long)g.chunks * kTaps * g.row_tiles * 128) return;
  const int lane = (int)(id & 63), half = (int)(id >> 6) & 1;
  const unsigned rest = (unsigned)(id >> 7);
  const int r = (int)(rest % (unsigned)g.row_tiles);
  const unsigned qt = rest / (unsigned)g.row_tiles;
  const int t = (int)(qt % (unsigned)kTaps), q = (int)(qt / (unsigned)kTaps);
  const int f = r * 32 + (lane & 31), c0 = (q * 4 + half * 2 + (lane >> 5)) * V;
  typename Elem<T>::vec v;
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] = (f < g.F && c0 + j < g.C) ? w[((size_t)f * g.C + c0 + j) * kTaps + t] : (T)0;
  reinterpret_cast<typename Elem<T>::vec*>(packed)[id] = v;
}

// PAIRS: a lane brings two neighbouring points at a time (rows of an even number of padded points, so that both are in one row; W >= 2).
template <typename T, int MT, int NT, bool PAIRS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 4))) void conv2d_kernel(const T* __restrict__ x, const T* __restrict__ packed, float* __restrict__ y, Geometry g) {
  typedef typename Elem<T>::vec vec;
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  typedef u32x2 two_words __attribute__((aligned(4)));
  typedef unsigned one_word __attribute__((aligned(2)));
  constexpr bool F16 = sizeof(T) == 2;
  constexpr int P = PAIRS ? 2 : 1;                    // points of an item
  constexpr int kHeld = PAIRS ? (NT == 1 ? 2 : 3) : (NT == 1 ? 3 : 5);        // items per lane that travel while the channels before them are multiplied (more: fetched behind them)
  constexpr int V = 16 / sizeof(T), TN = 64 * NT, kPitch = kPitchBytes / sizeof(T);
  extern __shared__ __align__(16) char lds[];
  T* image = reinterpret_cast<T*>(lds);                                                 // [2][span][pitch]
  unsigned* where = reinterpret_cast<unsigned*>(lds + 2 * (size_t)g.span * kPitchBytes);   // of an item: byte offset into x without the channel, and which of its points are inside
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int wide = (int)g.wide.by;
  // workgroups go to the eight XCDs round robin: an XCD gets a contiguous run of blocks
  const int per = gridDim.x >> 3, left = gridDim.x & 7, xcd = blockIdx.x & 7;
  const int block = xcd * per + (xcd < left ? xcd : left) + (blockIdx.x >> 3);
  const int run = (int)over((unsigned)block, g.blocks_across), rb = block - run * g.row_blocks, column0 = run * TN;
  const int last = (column0 + TN < g.columns ? column0 + TN : g.columns) - 1;
  const int place0 = place_of(column0, g) & ~(P - 1);
  const int count = (place_of(last, g) - place0 + 2 * wide + 3 + P - 1) / P;            // items; P times that <= span

  // A lane that has no use for a point reads the nearest one inside: the first point of x cost every load a line of its own
  // (float16 32 x 256 x 14 x 14 -> 256 33.2 -> 29.8 us).
  for (int i = tid; i < count; i += kThreads) {
    const unsigned p = (unsigned)(place0 + P * i), n = over(p, g.image), r = p - n * g.image.by, row = over(r, g.wide);
    const int h = (int)row - g.ph, w = (int)(r - row * g.wide.by) - g.pw;
    const int hc = h < 0 ? 0 : h < g.H ? h : g.H - 1, wc = w < 0 ? 0 : w <= g.W - P ? w : g.W - P;
    const unsigned inside = hc != h ? 0u : ((unsigned)w < (unsigned)g.W ? kFirst : 0u) | (PAIRS && (unsigned)(w + 1) < (unsigned)g.W ? kSecond : 0u);
    where[i] = ((n * (unsigned)g.C * (unsigned)g.H + (unsigned)hc) * (unsigned)g.W + (unsigned)wc) * (unsigned)sizeof(T) | inside;
  }

  // this lane's output points: LDS place of tap (0, 0), and where the result goes
  int at[NT];
  size_t to[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    int column = column0 + wn * 32 * NT + j * 32 + (lane & 31);
    if (column > last) column = last;
    at[j] = (place_of(column, g) - place0) * kPitch + (lane >> 5) * V;
    const unsigned hw = g.results.by, n = over((unsigned)column, g.results);
    to[j] = (size_t)n * g.F * hw + ((unsigned)column - n * hw);
  }
  // Item i of a lane: points P (lane + 64 i) .. + P - 1, channels wave * V .. + V - 1 of the chunk.  Loads go out without a branch between
  // them (points and channels past the end re-read the last one) and stay as they came until they are put into LDS: a
  // branch or a conversion behind each load is a wait for it.
  const size_t plane = (size_t)g.H * g.W * sizeof(T);
  const int items = (count + 63) >> 6;
  typedef typename std::conditional<F16, unsigned, typename std::conditional<PAIRS, u32x2, unsigned>::type>::type Word;      // of one channel
  struct Item { Word v[V]; };
  auto place = [&](int i) { return where[lane + 64 * i < count ? lane + 64 * i : count - 1]; };
  auto fetch = [&](int q, unsigned from, int j, Item& r) {
    const int c0 = (q * 4 + wave) * V, c = c0 + j < g.C ? c0 + j : g.C - 1;               // the same in all lanes
    const char* base = reinterpret_cast<const char*>(x) + c * plane;
    unsigned off = from & ~(kFirst | kSecond);
    if constexpr (F16) {
      // Scalar base, 32-bit offset: the compiler would add in 64 bits in every lane for every load (34 sizes 1.019 times as fast as so, 32 x 128 x 28 x 28 -> 128
      // 17.0 -> 16.3 us, 26 x 64 x 31 x 31 -> 112 13.3 -> 12.7; in float32 the products hide it, 0.98 to 1.03).
      ART_GLOBAL const char* from_base = (ART_GLOBAL const char*)base;
      asm("" : "+s"(from_base), "+v"(off));
      if constexpr (PAIRS) r.v[j] = *(ART_GLOBAL const one_word*)(from_base + (size_t)off);
      else r.v[j] = *(ART_GLOBAL const unsigned short*)(from_base + (size_t)off);
    } else if constexpr (PAIRS) {
      r.v[j] = *reinterpret_cast<const two_words*>(base + (size_t)off);
    } else {
      r.v[j] = *reinterpret_cast<const unsigned*>(base + (size_t)off);
    }
  };
  auto put = [&](int q, int i, unsigned from, const Item& r) {
    const int point = P * (lane + 64 * i), c0 = (q * 4 + wave) * V;
    vec v[P];
#pragma unroll
    for (int k = 0; k < P; ++k) {
      // both inside: first and second; one of a pair inside: it is the one further in of the two that were read
      const bool in = (from & (k ? kSecond : kFirst)) != 0, second = PAIRS && ((from & kSecond) ? k == 1 && (from & kFirst) : k == 0);
      if constexpr (F16) {
        const unsigned halves = !in ? 0x0c0c0c0cu : second ? 0x07060302u : 0x05040100u;
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        u32x4 packed_halves;
#pragma unroll
        for (int j = 0; j < 4; ++j) packed_halves[j] = __builtin_amdgcn_perm(r.v[2 * j + 1], r.v[2 * j], halves);
        v[k] = __builtin_bit_cast(vec, packed_halves);
      } else {
#pragma unroll
        for (int j = 0; j < V; ++j) {
          unsigned word;
          if constexpr (PAIRS) word = second ? r.v[j][1] : r.v[j][0];
          else word = r.v[j];
          v[k][j] = __builtin_bit_cast(T, in ? word : 0u);
        }
      }
      if (c0 + V > g.C) {
#pragma unroll
        for (int j = 0; j < V; ++j) if (c0 + j >= g.C) v[k][j] = (T)0;
      }
    }
    if (point >= P * count) return;
#pragma unroll
    for (int k = 0; k < P; ++k) *reinterpret_cast<vec*>(image + ((size_t)(q & 1) * g.span + point + k) * kPitch + wave * V) = v[k];
  };
  auto fetch_and_put = [&](int q, int i) {
    Item r;
    const unsigned from = place(i);
#pragma unroll
    for (int j = 0; j < V; ++j) fetch(q, from, j, r);
    put(q, i, from, r);
  };

  // The filter: a wavefront's MT x 2 operands of a tap, 64 x 16 bytes each, asked for kAhead taps before their use (a
  // tap is 64 to 256 cycles of matrix instructions, L2 answers after several hundred).
  constexpr int kSets = MT == 1 ? kTaps : 3, kAhead = kSets - 1;
  const vec* filter = reinterpret_cast<const vec*>(packed) + ((size_t)rb * 2 + wm) * MT * 128 + lane;
  const size_t filter_step = (size_t)g.row_tiles * 128;
  constexpr int kSum = MT == 1 && NT == 1 ? 3 : kTaps;            // taps summed by themselves
  constexpr int kRows = sizeof(T) == 2 && kSum == 3 ? 2 : 1;      // float16: and the halves of the channels
  constexpr int kPerTap = (kHeld * V + kTaps - 2) / (kTaps - 1);      // loads of the next chunk's image that go out with a tap
  vec a[kSets][MT][2];
  auto fetch_filter = [&](int set, int tap) {
    const vec* p = filter + (size_t)tap * filter_step;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) a[set][i][h] = p[(i * 2 + h) * 64];
  };

  art_lds_barrier();                                  // `where` is written
  Item held[kHeld];
  unsigned from[kHeld];
#pragma unroll
  for (int i = 0; i < kHeld; ++i) from[i] = place(i);
#pragma unroll
  for (int i = 0; i < kHeld; ++i)
#pragma unroll
    for (int j = 0; j < V; ++j) fetch(0, from[i], j, held[i]);
#pragma unroll
  for (int t = 0; t < kAhead; ++t) fetch_filter(t, t);      // asked for last: loads come back in order
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kHeld; ++i) put(0, i, from[i], held[i]);
  for (int i = kHeld; i < items; ++i) fetch_and_put(0, i);
  art_lds_barrier();
  f32x16 total[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) total[i][j][e] = 0.f;
  // `half`: only the lower half of the (last) chunk's channels exist, the upper half's products are left out
  auto chunk = [&](int q, auto last_chunk, auto half) {
    constexpr bool kMore = !decltype(last_chunk)::value;
    constexpr int kHalves = decltype(half)::value ? 1 : 2;
    const T* tile = image + (size_t)(q & 1) * g.span * kPitch;
    // a chunk is summed by itself and then added to the total (where registers allow, a row of taps by itself before that, in
    // float16 for each half of the channels: 1 % of the time, 10 % of the error): the error of a sum grows with the length of its chain
    f32x16 acc[MT][NT], row[kRows][MT][NT];
    vec b[2][NT];
    auto look = [&](int step) {                       // the points of half `step % kHalves` of a tap
      const int t = step / kHalves, h = step % kHalves;
      const T* from = tile + ((t / 3) * wide + t % 3) * kPitch;
#pragma unroll
      for (int j = 0; j < NT; ++j) b[step & 1][j] = *reinterpret_cast<const vec*>(from + at[j] + h * 2 * V);
    };
    look(0);
#pragma unroll
    for (int t = 0; t < kTaps; ++t) {
      if (kMore) {
#pragma unroll
        for (int k = t * kPerTap; k < (t + 1) * kPerTap && k < kHeld * V; ++k) fetch(q + 1, from[k / V], k % V, held[k / V]);
      }
      if (kMore || t + kAhead < kTaps) fetch_filter((t + kAhead) % kSets, q * kTaps + t + kAhead);
      __builtin_amdgcn_sched_barrier(0);              // left to the scheduler, the loads sink to their use
#pragma unroll
      for (int h = 0; h < kHalves; ++h) {
        const int step = t * kHalves + h;
        if (step + 1 < kTaps * kHalves) look(step + 1);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            row[h % kRows][i][j] = Elem<T>::multiply(a[t % kSets][i][h], b[step & 1][j], h < kRows && t % kSum == 0 ? f32x16(0) : row[h % kRows][i][j]);
      }
      if (t % kSum != kSum - 1) continue;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const f32x16 sum = kRows == 2 && kHalves == 2 ? row[0][i][j] + row[kRows - 1][i][j] : row[0][i][j];
          acc[i][j] = t < kSum ? sum : acc[i][j] + sum;
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) total[i][j] += acc[i][j];
    if (kMore) {
#pragma unroll
      for (int i = 0; i < kHeld; ++i) put(q + 1, i, from[i], held[i]);
      for (int i = kHeld; i < items; ++i) fetch_and_put(q + 1, i);
      art_lds_barrier();      // the other buffer is written, this one is free
    }
  };
  for (int q = 0; q + 1 < g.chunks; ++q) chunk(q, std::false_type{}, std::false_type{});
  if (MT == 1 && g.C - (g.chunks - 1) * 4 * V <= 2 * V) chunk(g.chunks - 1, std::true_type{}, std::true_type{});   // MT = 2 has no registers left for it
  else chunk(g.chunks - 1, std::true_type{}, std::false_type{});

  store_results<MT, NT>(total, y, to, column0 + wn * 32 * NT + (lane & 31), last, ((rb * 2 + wm) * MT) * 32, g);
}

// The most points a block of `columns` output points can need: every step to the next row skips two points, every
// step to the next image two rows.
int span_of(const Geometry& g, int columns, bool pairs = false) {
  if (columns > g.columns) columns = g.columns;
  const long long wide = g.WO + 2 + (pairs && g.WO % 2), hw = (long long)g.HO * g.WO;
  const long long rows = (columns - 1 + g.WO - 1) / g.WO, images = (columns - 1 + hw - 1) / hw;
  const long long span = columns - 1 + rows * (wide - g.WO) + images * 2 * wide + 2 * wide + 3 + (pairs ? 2 : 0);
  return span > (1 << 20) ? 1 << 20 : (int)span;
}

size_t lds_of(int span) { return (size_t)span * (2 * kPitchBytes + 4); }

// Forms: 1 = 64 features x 64 points per block, 2 = 64 x 128, 3 = 128 x 128; 4, 5, 6 the same over the staged image, 7 = 64 x 64
// there with short sums (float32), plus 256 x slices of the channels (0: one); 8, 9, 10 = 16 features x 16, 32, 64 points (art_conv2d_direct.hip).
bool direct(int form) { return form >= 8 && form <= 10; }
int shape_of(int form) { return (form & 255) % 3; }
int features_of(int form) { return direct(form) ? 16 : shape_of(form) == 0 ? 128 : 64; }
int points_of(int form) { return direct(form) ? 16 << (form - 8) : shape_of(form) == 1 ? 64 : 128; }
int slices_of(int form) { return form >> 8 ? form >> 8 : 1; }

bool geometry(Geometry& g, int f16, int N, int C, int H, int W, int F, int HO, int WO, int ph, int pw) {
  g = Geometry{N, C, H, W, F, HO, WO, ph, pw};
  if (N < 1 || C < 1 || H < 1 || W < 1 || F < 1 || HO < 1 || WO < 1) return false;
  // byte offsets into x and places in the padded image are 32-bit
  if ((long long)HO > (1 << 20) || (long long)WO > (1 << 20)) return false;
  const long long image = (long long)(HO + 2) * (WO + 2);
  if (image > (1LL << 30) / N || (long long)H * W > (1LL << 30) / ((long long)N * C)) return false;
  if ((long long)N * C * H * W * (f16 ? 2 : 4) > (1LL << 31)) return false;
  g.columns = N * HO * WO;
  g.results = make_div((unsigned)(HO * WO));
  g.width = make_div((unsigned)WO);
  g.image = make_div((unsigned)((HO + 2) * (WO + 2)));
  g.wide = make_div((unsigned)(WO + 2));
  g.chunks = (C + (f16 ? 31 : 15)) / (f16 ? 32 : 16);
  return (long long)g.chunks * kTaps * ((F + 127) / 128) * 4 < (1 << 22);      // packed filter below 4 GiB
}

bool fits(Geometry g, int f16, int form) {
  const int kind = form & 255;
  if (form < 1 || kind < 1 || (kind > (f16 ? 6 : 7) && !direct(form))) return false;
  g.span = span_of(g, points_of(form));
  if (direct(form)) return art::conv::direct_fits(g, f16, form);
  if (kind <= 3) return form == kind && lds_of(g.span) <= (f16 && form == 1 ? kWideLds : kMaxLds);
  return slices_of(form) <= 64 && slices_of(form) <= g.chunks && staged_lds(g) <= 160 * 1024;
}

long long blocks_of(const Geometry& g, int form) {
  return (long long)((g.columns + points_of(form) - 1) / points_of(form)) * ((g.F + features_of(form) - 1) / features_of(form));
}

// What a form takes, in microseconds, both launches: a fixed part, per chunk of a block a time that grows with the blocks that
// share a compute unit and with how unevenly they do, a ramp per further round, and the stores.  Fitted to 330 sizes a form in float16 and
// 310 in float32, two thirds of them of 16 to 256 channels and features, images of 7 to 56 squared and batches of 1 to 32: 5 and 1 to 3 % off.
// (float16 64 x 64: its fixed part, 5.95, is 0.45 above that fit, which would have it taken at 7 % of 20000 sizes where now another form, mostly the staged
// 64 x 64, is.  At 200 of these the one taken now is 1.064 times as fast in the mean, at 127 by more than 5 %, at six slower by more than 5 %, up to 8.)
constexpr int kUnits = 256;                      // compute units of an MI355X
double launch_time(const Geometry& g, int f16, int form) {
  struct Cost { double fixed, alone, shared, uneven, again, store; };
  static const Cost cost[2][3] = {{{5.364, 2.772, 2.427, 2.502, 0.862, 0.193}, {5.916, 4.966, 4.242, 4.677, 1.743, 0.148}, {6.714, 8.862, 8.215, 9.696, 1.217, 0.148}},
                                  {{5.950, 1.524, 1.065, 0.756, 0.404, 0.241}, {6.181, 1.748, 0.815, 0.889, 1.157, 0.234}, {6.879, 2.374, 1.306, 1.421, 1.398, 0.193}}};
  const Cost& c = cost[f16 != 0][form - 1];
  const int per_chunk = f16 ? 32 : 16;
  const double chunks = g.chunks - (form < 3 && g.C - (g.chunks - 1) * per_chunk <= per_chunk / 2 ? 0.5 : 0.0);
  const double rounds = (double)blocks_of(g, form) / kUnits, full = rounds > 1 ? rounds : 1, uneven = ceil(rounds) > full ? ceil(rounds) - full : 0;
  // an image so wide that a compute unit holds two blocks or one (float16 64 x 64): 2.0 and 3.8 a chunk and round over ten sizes, 10 % off
  const size_t lds = lds_of(span_of(g, points_of(form)));
  const double shared = lds <= kMaxLds ? c.shared : lds <= kWideLds / 2 ? 2.0 : 3.8;
  return c.fixed + chunks * (c.alone + shared * (full - 1) + (lds <= kMaxLds ? c.uneven : shared) * uneven) + c.again * (full - 1) + c.store * 4e-6 * g.columns * g.F;
}

// The same for the staged forms (the launch that stages the image included): a fixed part, per chunk of a block's slice a time
// that grows with the blocks that share a compute unit and with how unevenly they do, the copy, the stores, and for slices the
// third launch.  Fitted to 116 sizes in float16 and, float32, to the 2058 times of 320 sizes that are within 1.5 times the fastest: 3.1 and 3 % off.  What
// is picked of all forms in float32 is 0.48 % slower than the fastest in the mean, 2.2 % of the sizes by more than 5 % (0.63 and 4.1 % with the
// constants before the gathering forms loaded two points at a time: these came out 2 % below, the staged ones 3 % above what they take).
double staged_time(const Geometry& g, int f16, int form, int slices) {
  struct Cost { double fixed, alone, shared, uneven; };
  struct Rest { double sum, sum_bytes, copy, store; };
  static const Cost cost[2][4] = {{{5.82, 2.736, 2.642, 2.469}, {6.48, 4.700, 4.335, 4.628}, {8.11, 8.376, 8.365, 9.814}, {6.25, 4.809, 5.443, 5.217}},
                                  {{6.52, 0.998, 0.861, 0.730}, {7.14, 1.309, 0.900, 0.661}, {8.03, 1.836, 1.636, 1.386}, {}}};
  static const Rest rest[2] = {{2.55, 0.348, 0.440, 0.246}, {2.62, 0.342, 0.510, 0.242}};
  const Cost& c = cost[f16 != 0][form - 4];
  const Rest& r = rest[f16 != 0];
  const int per_chunk = f16 ? 32 : 16;
  const double half = form != 6 && g.C - (g.chunks - 1) * per_chunk <= per_chunk / 2 ? 0.5 : 0.0;
  const double rounds = (double)blocks_of(g, form) * slices / kUnits, full = rounds > 1 ? rounds : 1, megabytes = 4e-6 * g.columns * g.F;
  const double chunks = slices > 1 ? (g.chunks + slices - 1) / slices : g.chunks - half;
  const double t = c.fixed + chunks * (c.alone + c.shared * (full - 1) + c.uneven * (ceil(rounds) > full ? ceil(rounds) - full : 0)) +
                   r.copy * 64e-6 * g.chunks * g.N * (g.HO + 2) * (g.WO + 2);
  const double passes = (g.N + images_of_pass(g) - 1) / images_of_pass(g);
  return c.fixed * (passes - 1) + (slices == 1 ? t + r.store * megabytes : t + r.sum + r.sum_bytes * (slices + 1) * megabytes);
}

// Where the generic lowering has no matrix instructions for the convolution: it sums on the vector units.
bool on_vector_units(const Geometry& g) { return g.F < 32 || g.columns < 32 || 9 * g.C < 32 || blocks_of(g, 1) < 16; }

// Whether a form's sums are no longer than those of the generic kernels that it takes the place of.  On the vector units 64 terms and
// more are spread over a wavefront: float32 form 7 only, float16 the blocks of 64 x 64, whose rows of taps are summed by themselves - the
// gathering one by halves of the channels, too: 0.64 to 0.99 times the generic kernels' error; the staged one (0.6 to 1.02) is 1.00 to 1.07
// times from 17 to 47 channels that are not 24, 32 or 40 and is left out there.
// Fewer terms are a chain there: 0.42 to 0.93 times its error in these blocks, 0.46 to 1.0 in the larger ones.
// Elsewhere float16 with fewer than 32 channels that are not 8 or 16 and so on: the larger blocks sum 18 instructions in a row where
// the generic kernels need 9 C / 16 (5 to 31 channels 1.02 to 1.22 times their error, the blocks of 64 x 64 0.66 to 1.01
// times; with four channels both are above it).
bool exact_enough(const Geometry& g, int f16, int form) {
  if (direct(form)) return true;
  if (!on_vector_units(g)) return !f16 || (g.C > 4 && shape_of(form) == 1) || g.C >= 32 || g.C % 8 == 0;
  if (9 * g.C < 64) return true;
  if (!f16) return (form & 255) == 7;
  return form == 1 || ((form & 255) == 4 && (g.C <= 16 || g.C % 8 == 0 || g.C >= 48));
}

// What comes on top of these times outside of the sizes they were fitted to: a filter of more than 256 x 256 is packed for longer, and
// each further round of blocks over the staged image has a ramp of its own.  With it they are 6 (float32) and 10 % (float16) off over 530
// such sizes (10 and 21 without); the forms picked are 0.2 to 1.5 % slower than the fastest either way, so it is no part of the picking.
double outside_time(const Geometry& g, int f16, int form) {
  const double filter = 1e-6 * art_conv2d_packed_bytes(f16, g.C, g.F), most = f16 ? 1.2 : 2.4, rounds = (double)blocks_of(g, form) * slices_of(form) / kUnits;
  return (filter > most ? (f16 ? 2.547 : 1.749) * (filter - most) : 0.0) + ((form & 255) > 3 && rounds > 1 ? (f16 ? 1.584 : 0.811) * (rounds - 1) : 0.0);
}

// What the generic kernels take, in microseconds, 6 to 16 % off where the two are close.  On the vector units a thread or a wavefront per
// result, or, for many results, a thread per 4 x 4 or 4 x 2 of them.  On the matrix instructions a padded copy of the image and blocks of
// 128 x 128 or 64 x 64 as it chooses them (plans.py), from 1024 terms on in slices where they are few.  us, generic / here:
//   float32 2 x 232 -> 24, 52 x 52 375 / 37; 1 x 24 -> 32, 15 x 15 7.6 / 13.7; 58 x 12 -> 4, 158 x 158 82 / 621; 205 x 40 -> 24, 33 x 33
//   6457 / 213; 7 x 34 -> 4058, 6 x 6 17 / 25; 6 x 9 -> 294, 76 x 76 39 / 50; 9 x 216 -> 64, 17 x 17 23 / 20;
//   float16 28 x 40 -> 16, 42 x 42 319 / 19; 1 x 16 -> 40, 7 x 7 5.6 / 7.0; 63 x 20 -> 4, 90 x 90 59 / 107; 2 x 65 -> 2887, 8 x 8 13.5 / 17.7;
//   9 x 240 -> 104, 13 x 13 19 / 13.8.
double generic_time(const Geometry& g, int f16) {
  const double results = 1e-6 * g.columns * g.F, products = results * 9 * g.C, image = 1e-6 * g.N * g.C * g.H * g.W;
  if (on_vector_units(g)) {
    const bool patches = g.F % 4 == 0 && g.WO % 2 == 0 && (double)g.columns * g.F >= 131072.0 * (g.WO % 4 == 0 ? 16 : 8);
    return patches ? (f16 ? 11.36 + 0.094 * products + 1.507 * image : 11.63 + 0.064 * products + 1.611 * image)
                   : (f16 ? 5.3 + 1.3 * products : 5.5 + 1.1 * products);
  }
  struct Cost { double fixed, alone, shared, uneven, store, copy, sum; };
  static const Cost cost[2][2] = {{{6.211, 1.813, 1.628, 1.308, 1.193, 2.021, 4.178}, {7.35, 5.891, 6.289, 1.18, 1.539, 2.211, 3.0}},
                                  {{6.297, 0.851, 0.99, 0.347, 0.727, 0.0, 3.926}, {7.821, 1.47, 2.894, 1.055, 1.447, 1.719, 3.0}}};
  const long long big = blocks_of(g, 3), small = blocks_of(g, 1);
  const int side = big < 16 || small < (f16 ? 700 : 900) * ((big + (f16 ? 511 : 255)) / (f16 ? 512 : 256)) ? 0 : 1;
  const Cost& c = cost[f16 != 0][side];
  long long slices = 1;
  if (small < 512 && 9 * g.C >= 1024) {
    slices = 9 * g.C / 256 < (1024 + small - 1) / small ? 9 * g.C / 256 : (1024 + small - 1) / small;
    slices = slices > 8 ? 8 : slices;
  }
  const double rounds = (double)(side ? big : small) * slices / kUnits, full = rounds > 1 ? rounds : 1, per = 9 * g.C / 64.0 / slices;
  return c.fixed + per * (c.alone + c.shared * (full - 1) + c.uneven * (ceil(rounds) > full ? ceil(rounds) - full : 0)) + c.store * results * slices +
         c.copy * image + (slices > 1 ? c.sum : 0.0);
}

// The form for these sizes, or 0: the generic kernels are faster or sum more exactly there.
//  * One of the forms that are exact enough, by the estimates: the channels sliced where there are few blocks (float32 9 x 216 -> 64, 17 x 17
//    20 us, 46 without slices), the image staged unless it is large and there is little to multiply (float16 18 x 64 -> 48, 51 x 51 15.3
//    gathered, 16.8 staged, 1 x 40 -> 152, 42 x 42 10.0 and 9.0).
//  * It is taken where one of them is estimated below the generic kernels (on the matrix instructions, 5 % above): over 1100 sizes a type outside of
//    16 to 256 channels and features and 7 to 56 squared (770 to fit it and 335 new ones), 0.7 to 1.3 (float32) and 1.5 to 1.7 %
//    (float16) off the faster one in the mean; within them 0.1 to 0.9 %.  One of them, whichever it is: for many rounds the staged pick may be
//    estimated above the generic kernels where a gathered form is not (float16 197 x 19 -> 80, 24 x 24 51 us, 36 staged, 32 gathered).
//  * Fewer than 8 channels: a chunk is mostly zeros.  Over 200 sizes the generic kernels were 1.14 (float32) and 1.10 times as fast in the
//    mean, up to 5.6 and 7.5 (float16 10 x 3 -> 2, 151 x 151 7.6 / 58).  Faster here at all 19 sizes: two or three channels with 32 features and
//    half a million results on in float16 (9 x 3 -> 105, 26 x 26 10.1 / 8.1, 40 x 3 -> 50, 87 x 87 159 / 74), 64 and a million in float32
//    (14 x 2 -> 109, 38 x 38 15.6 / 14.1, 8 x 3 -> 105, 42 x 42 14.9 / 10.7).
//  * Images too wide for 64 KiB of LDS are staged, or gathered by blocks with 160 KiB where only these sum exactly enough (float16, 17 to 47
//    channels on the vector units' ground): 18 x 44 -> 29, 120 x 120 102 us, 3 x 33 -> 21, 147 x 147 32 (staged 79 and 25, generic 8347 and 558).
//  * A copy of more than 128 MiB for one image is not made: the image is gathered.  Beside the packed filter a call takes 192 MiB at the
//    most, 128 for the copy and 64 for slices (4 kUnits blocks of 128 x 128).
// `gathered`: the best of the forms that need no more than the packed filter, for callers that have no more.
int choose(const Geometry& g, int f16, bool gathered, double* time = nullptr) {
  const bool image_like = (g.C == 2 || g.C == 3) && g.F >= (f16 ? 32 : 64) && (long long)g.columns * g.F >= (f16 ? 1 << 19 : 1 << 20);
  if (g.C < 8 && !image_like && !gathered) return 0;
  const bool staged = !gathered && (size_t)g.chunks * (g.HO + 2) * (g.WO + 2) * kChunkBytes <= kMostCopy;
  const bool vector_units = on_vector_units(g);
  int best = 0;
  double t_best = 1e30, t_outside = 1e30;
  auto consider = [&](int form, double t) {
    if (!fits(g, f16, form)) return;
    if (t < t_best) { best = form; t_best = t; }
    if (t + outside_time(g, f16, form) < t_outside) t_outside = t + outside_time(g, f16, form);
  };
  for (int form = 1; form <= 7; ++form) {
    if (!exact_enough(g, f16, form) || (form == 7 && (f16 || !vector_units))) continue;
    if (form <= 3 && (lds_of(span_of(g, points_of(form))) <= kMaxLds || (vector_units && !exact_enough(g, f16, 4)))) consider(form, launch_time(g, f16, form));
    for (int slices : {1, 2, 3, 4, 5, 6, 8, 12})
      if (form > 3 && staged && slices <= g.chunks && (slices == 1 || slices * blocks_of(g, form) <= 4 * kUnits)) consider(form + (slices > 1 ? 256 * slices : 0), staged_time(g, f16, form, slices));
  }
  if (!best || !(gathered || image_like || t_outside < (vector_units ? 1.0 : 1.05) * generic_time(g, f16))) return 0;
  if (time) *time = t_best + outside_time(g, f16, best);
  return best;
}

template <typename T, int MT, int NT, bool PAIRS>
int launch(const void* x, const void* packed, void* y, const Geometry& g, unsigned blocks, hipStream_t st) {
  static bool configured = false;
  if (lds_of(g.span) > kMaxLds && !configured) {
    ART_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(conv2d_kernel<T, MT, NT, PAIRS>), hipFuncAttributeMaxDynamicSharedMemorySize, kWideLds));
    configured = true;
  }
  conv2d_kernel<T, MT, NT, PAIRS><<<dim3(blocks), dim3(kThreads), lds_of(g.span), st>>>((const T*)x, (const T*)packed, (float*)y, g);
  ART_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int run(const void* x, const void* w, void* packed, void* y, const Geometry& g, int form, hipStream_t st) {
  const long long lanes = (long long)g.chunks * kTaps * g.row_tiles * 128;
  conv2d_pack_kernel<T><<<dim3((unsigned)((lanes + kThreads - 1) / kThreads)), dim3(kThreads), 0, st>>>((const T*)w, (T*)packed, g);
  ART_LAUNCH_CHECK();
  const unsigned blocks = (unsigned)blocks_of(g, form);
  // Two points at a time, in rows of an even number, unless a row has one or the odd column does not fit into LDS any more.
  const int span = span_of(g, points_of(form), true);
  if (g.W >= 2 && (long long)(g.HO + 2) * (g.WO + 2 + g.WO % 2) <= (1 << 30) / g.N &&
      lds_of(span) <= (lds_of(g.span) > kMaxLds ? kWideLds : kMaxLds)) {
    Geometry even = g;
    even.span = span;
    even.wide = make_div((unsigned)(g.WO + 2 + g.WO % 2));
    even.image = make_div((unsigned)(g.HO + 2) * even.wide.by);
    return form == 1 ? launch<T, 1, 1, true>(x, packed, y, even, blocks, st) : form == 2 ? launch<T, 1, 2, true>(x, packed, y, even, blocks, st)
                                                                                       : launch<T, 2, 2, true>(x, packed, y, even, blocks, st);
  }
  return form == 1 ? launch<T, 1, 1, false>(x, packed, y, g, blocks, st) : form == 2 ? launch<T, 1, 2, false>(x, packed, y, g, blocks, st)
                                                                                    : launch<T, 2, 2, false>(x, packed, y, g, blocks, st);
}

}  // namespace

extern "C" int art_conv2d_form(int f16, int N, int C, int H, int W, int F, int HO, int WO, int ph, int pw, int form) {
  Geometry g;
  if (!geometry(g, f16, N, C, H, W, F, HO, WO, ph, pw)) return 0;
  return form ? (fits(g, f16, form) ? form : 0) : choose(g, f16, true);
}

extern "C" int art_conv2d_exact_enough(int f16, int N, int C, int H, int W, int F, int HO, int WO, int ph, int pw, int form) {
  Geometry g;
  return geometry(g, f16, N, C, H, W, F, HO, WO, ph, pw) && fits(g, f16, form) && exact_enough(g, f16, form);
}

extern "C" int art_conv2d_choose(int f16, int N, int C, int H, int W, int F, int HO, int WO, int ph, int pw) {
  Geometry g;
  return geometry(g, f16, N, C, H, W, F, HO, WO, ph, pw) ? choose(g, f16, false) : 0;
}

// The form of art_conv2d_direct.hip for these sizes, or 0 where its time is estimated above that of what `choose` takes, or of the generic
// kernels where that takes none.
//  * Over 900 sizes (a third of them outside of 16 to 256 channels and features and 7 to 56 squared) what is taken then is 1.42 to 1.49 (float32) and 1.18 times
//    as fast as before in the mean, on 6 of them more than 5 % slower (up to 1.28 times).
//  * Not where the generic kernels have few terms or most taps are outside of the image (their estimate is twice their time there): fewer than 8
//    channels (3 x 4 x 6 x 6 -> 108 2.9 us, 4.2 here), images of fewer than four points (13 x 8 x 1 x 1 -> 78 2.4 and 4.4).
//  * Not for more than 100 million products on the matrix instructions' ground: the other forms' larger blocks catch up there, and half
//    of all wrong picks were beyond it (9 x 48 x 34 x 34 -> 80 22.3 us, 27.6 here), for 1.5 % of the gain.
extern "C" int art_conv2d_direct(int f16, int N, int C, int H, int W, int F, int HO, int WO, int ph, int pw) {
  Geometry g;
  if (!geometry(g, f16, N, C, H, W, F, HO, WO, ph, pw) || C < 8 || (long long)HO * WO < 4) return 0;
  if (9.0 * g.columns * F * C > 1e8 && !on_vector_units(g)) return 0;
  double least = 1e30;
  int best = 0;
  for (int form = 8; form <= 10; ++form) {
    if (!fits(g, f16, form)) continue;
    const double t = art::conv::direct_time(g, f16, form);
    if (t < least) { least = t; best = form; }
  }
  if (!best) return 0;
  double other = 0.0;
  if (!choose(g, f16, false, &other)) other = generic_time(g, f16);
  return least < other ? best : 0;
}

extern "C" size_t art_conv2d_packed_bytes(int f16, int C, int F) {
  const size_t chunks = ((size_t)C + (f16 ? 31 : 15)) / (f16 ? 32 : 16);
  return chunks * kTaps * (((size_t)F + 127) / 128) * 4 * 2048;
}

extern "C" size_t art_conv2d_scratch_bytes(int f16, int N, int C, int H, int W, int F, int HO, int WO, int ph, int pw, int form) {
  Geometry g;
  if (!geometry(g, f16, N, C, H, W, F, HO, WO, ph, pw) || !fits(g, f16, form)) return 0;
  return direct(form) ? 0 : (form & 255) <= 3 ? art_conv2d_packed_bytes(f16, C, F) : staged_bytes(g, slices_of(form));
}

extern "C" int art_conv2d(const void* x_dev, const void* w_dev, void* packed_dev, void* y_dev, int f16, int N, int C, int H, int W, int F, int HO,
                          int WO, int ph, int pw, int form, void* stream) {
  Geometry g;
  ART_REQUIRE(geometry(g, f16, N, C, H, W, F, HO, WO, ph, pw) && fits(g, f16, form), "art_conv2d: sizes the kernel does not take (form %d)", form);
  ART_REQUIRE(x_dev && w_dev && (packed_dev || direct(form)) && y_dev, "art_conv2d: null pointer");
  const uintptr_t size = f16 ? 2 : 4;
  ART_REQUIRE((uintptr_t)x_dev % size == 0 && (uintptr_t)w_dev % size == 0 && (direct(form) || (uintptr_t)packed_dev % 16 == 0) && (uintptr_t)y_dev % 4 == 0,
              "art_conv2d: misaligned tensor");
  ART_REQUIRE(!art::overlaps(y_dev, (size_t)N * F * HO * WO * 4, x_dev, (size_t)N * C * H * W * size) &&
                  !art::overlaps(y_dev, (size_t)N * F * HO * WO * 4, w_dev, (size_t)F * C * 9 * size),
              "art_conv2d: the result must not overlap an operand");
  g.row_blocks = (F + features_of(form) - 1) / features_of(form);
  g.row_tiles = g.row_blocks * (features_of(form) / 32);
  g.blocks_across = make_div((unsigned)g.row_blocks);
  g.span = span_of(g, points_of(form));
  if (direct(form)) return art::conv::run_direct(x_dev, w_dev, y_dev, g, f16, form, (hipStream_t)stream);
  if ((form & 255) > 3)
    return run_staged(x_dev, w_dev, packed_dev, y_dev, g, f16, form & 255, slices_of(form), (hipStream_t)stream);
  return f16 ? run<_Float16>(x_dev, w_dev, packed_dev, y_dev, g, form, (hipStream_t)stream)
             : run<float>(x_dev, w_dev, packed_dev, y_dev, g, form, (hipStream_t)stream);
}
