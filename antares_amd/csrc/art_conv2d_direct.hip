// 3 x 3 convolutions of few products in ONE launch (see art_conv2d.hip for the operation and the other kernels).
//
// Why: below some 20 us the other forms are bound by their launches - the filter (and the image) packed by one, the products,
// for few blocks the slices' sums by a third - each with its own ramp and its own trip to memory behind the one before.
// Here nothing is packed and nothing meets in memory:
//   * a block owns 16 features x 16 NT output points over all channels; its wavefronts take the channels in turn, 8 (float32) or 16 at a
//     time, and meet once in LDS, in float64;
//   * a wavefront brings what its channels need by itself, without barriers: the block's run of points of the padded image
//     (a lane has up to four of them, their places are worked out once) and the channels * 9 values of each feature, which are
//     contiguous as they lie in memory, in 16-byte pieces.  The next channels travel to registers while these are multiplied;
//   * image [channel][point] (float16: two channels to a word), filter [feature][channels * 9] in 304 bytes: the 64 lanes of an
//     operand read touch 64 banks;
//   * v_mfma_f32_16x16x4_f32 and 16x16x16_f16: the small tiles give the most blocks, and what bounds a block is the chain of its
//     wavefronts' instructions (a unit of channels, 16 points: 0.8 us; its products alone 0.25);
//   * sums: float32 four products by themselves, two of these per tap, a row of taps, all rows in float64; float16 the 48 products of a
//     row of taps, all rows in float64.  Over 400 sizes where this is the faster kernel its error against 64 bits is the smaller one
//     at every size: float32 0.65e-7 (form 7, the shortest sums before, 0.65 to 0.75e-7, the others and the generic kernels 1.3e-7), float16
//     0.54e-7 (0.6 to 0.85e-7).
// Measured, against what ran before, us: float32 4 x 40 x 8 x 8 -> 104 12.9 -> 4.6, 16 x 48 x 20 x 20 -> 16 18.2 -> 6.2, 18 x 136 x 8 x 8 -> 32
// 14.4 -> 6.7, 2 x 232 x 52 x 52 -> 24 35.8 -> 20.9; float16 1 x 104 x 9 x 9 -> 176 9.4 -> 5.4, 1 x 72 x 23 x 23 -> 40 8.4 -> 5.8, 30 x 16 x 9 x 9 -> 64
// 6.6 -> 5.0.  Over 320 sizes of the range float32 1.51 times as fast in the mean (1.7 where it is taken), float16 1.2 (1.34).  Tiles of 32 features, and
// products of a row of taps ahead of their sums, were no faster; 16 wavefronts that spill registers lose 1 us.
#include "art_conv2d.h"

namespace {

using namespace art::conv;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

constexpr int kMostPoints = 4;                      // of the run, per lane
constexpr int kFilterPitch = 304;                   // bytes of a feature in LDS: CH * 9 values are 288
constexpr int kPieces = 18;                         // 16 bytes each of them
template <typename T> constexpr int kChannels = 32 / (int)sizeof(T);      // that a wavefront takes at a time: 8 float32, 16 float16
// Wavefronts of a block: as many as the registers of a lane allow without spilling.
constexpr int most_waves(int size, int NT, int KP) { return NT == 4 ? 8 : KP * NT * (6 - size) <= 8 ? 16 : 12; }
constexpr size_t kLds = 160 * 1024;

struct Direct {
  int units;                // runs of kChannels
  int segment;              // columns that blocks do not reach across: an image's, or all
  Div tiles;                // blocks along a segment
  int pitch;                // points of a channel in LDS, a multiple of 4
  int wave_bytes;           // LDS of a wavefront
  int whole;                // the filter is 16-byte aligned
};

template <typename T, int NT, int KP>
__global__ __launch_bounds__(64 * most_waves(sizeof(T), NT, KP)) void conv2d_direct_kernel(const T* __restrict__ x, const T* __restrict__ w, float* __restrict__ y, Geometry g, Direct d) {
  constexpr bool F16 = sizeof(T) == 2;
  constexpr int V = 16 / sizeof(T), CH = kChannels<T>;
  constexpr int kLoads = (kPieces * 16 + 63) / 64;
  typedef typename Elem<T>::vec vec;
  typedef typename Elem<T>::raw raw;
  extern __shared__ __align__(16) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int l16 = lane & 15, quarter = lane >> 4;
  // workgroups go to the eight XCDs round robin: an XCD gets a contiguous run of blocks
  const int per = gridDim.x >> 3, left = gridDim.x & 7, xcd = blockIdx.x & 7;
  const int block = xcd * per + (xcd < left ? xcd : left) + (blockIdx.x >> 3);
  const int run = (int)over((unsigned)block, g.blocks_across), f_first = (block - run * g.row_blocks) * 16, seg = (int)over((unsigned)run, d.tiles);
  const int end = (seg + 1) * d.segment, column0 = seg * d.segment + (run - seg * (int)d.tiles.by) * 16 * NT;
  const int last = (column0 + 16 * NT < end ? column0 + 16 * NT : end) - 1;
  const int wide = (int)g.wide.by, place0 = place_of(column0, g);
  const int points = place_of(last, g) - place0 + 2 * wide + 3, items = (points + 63) >> 6;      // <= g.span, 1 to KP

  // this lane's points of the run: where they are in x, without the channel
  unsigned from[KP];
  bool in[KP];
#pragma unroll
  for (int i = 0; i < KP; ++i) {
    const unsigned p = (unsigned)(place0 + (lane + 64 * i < points ? lane + 64 * i : points - 1)), n = over(p, g.image), r = p - n * g.image.by, row = over(r, g.wide);
    const int h = (int)row - g.ph, c = (int)(r - row * g.wide.by) - g.pw, near_h = h < 0 ? 0 : h < g.H ? h : g.H - 1, near_c = c < 0 ? 0 : c < g.W ? c : g.W - 1;
    in[i] = lane + 64 * i < points && h == near_h && c == near_c;
    from[i] = ((n * (unsigned)g.C * (unsigned)g.H + (unsigned)near_h) * (unsigned)g.W + (unsigned)near_c) * (unsigned)sizeof(T);      // outside: the nearest point inside
  }
  // this lane's output points: their place in the run
  int at[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int column = column0 + j * 16 + l16;
    at[j] = place_of(column < last ? column : last, g) - place0;
  }
  // this lane's pieces of the filter: feature, piece of its CH * 9 values
  unsigned piece[kLoads];
  int piece_to[kLoads], piece_at[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int id = lane + 64 * i < kPieces * 16 ? lane + 64 * i : kPieces * 16 - 1, f = id / kPieces, r = id - f * kPieces;
    piece[i] = (unsigned)(f_first + f < g.F ? f_first + f : g.F - 1) * (unsigned)(g.C * kTaps * (int)sizeof(T));
    piece_at[i] = r * 16;
    piece_to[i] = f * kFilterPitch + r * 16;
  }
  const int plane = g.H * g.W * (int)sizeof(T);
  // x is at most 2 GiB: a channel is a scalar offset.  With a pointer for each every load costs a 64-bit sum in each lane, of the chain that bounds a
  // block: 130 sizes 1.022 times as fast as so, us: float32 1 x 152 x 8 x 8 -> 48 7.7 -> 7.0, 9 x 224 x 12 x 12 -> 24 9.6 -> 8.8, float16 21 x 184 x 35 x 35 -> 16 21.2 -> 19.6.
  const auto image_in = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(x), 0, -1, art::kBufferFlags);
  const int row_bytes = g.C * kTaps * (int)sizeof(T);      // C % V == 0: whole pieces
  typedef raw pair __attribute__((ext_vector_type(2)));
  pair held[KP][CH / 2];
  vec filter[kLoads];
  // What a lane has no use for it reads again from a place that is valid (nothing branches around a load), and puts zeros.
  auto fetch = [&](int unit) {
    const int c0 = unit * CH;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int o = c0 * (kTaps * (int)sizeof(T)) + piece_at[i];
      const char* p = reinterpret_cast<const char*>(w) + (size_t)(piece[i] + (unsigned)(o < row_bytes ? o : 0));
      if (d.whole) {                                // the same in all lanes
        filter[i] = *reinterpret_cast<const vec*>(p);
      } else {
#pragma unroll
        for (int k = 0; k < V; ++k) filter[i][k] = reinterpret_cast<const T*>(p)[k];
      }
    }
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      if (i > 0 && i >= items) break;               // the same in all lanes
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int at = (c0 + j < g.C ? c0 + j : g.C - 1) * plane;
        if constexpr (F16) held[i][j >> 1][j & 1] = __builtin_amdgcn_raw_buffer_load_b16(image_in, (int)from[i], at, 0);
        else held[i][j >> 1][j & 1] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(image_in, (int)from[i], at, 0));
      }
    }
  };
  char* const image = lds + wave * d.wave_bytes;
  char* const taps = image + CH * d.pitch * (int)sizeof(T);
  auto put = [&](int unit) {
    const int c0 = unit * CH;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int o = c0 * (kTaps * (int)sizeof(T)) + piece_at[i];
      if (64 * i + 63 < kPieces * 16 || lane + 64 * i < kPieces * 16) *reinterpret_cast<vec*>(taps + piece_to[i]) = o < row_bytes ? filter[i] : vec(0);
    }
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      if (i > 0 && i >= items) break;
      if (lane + 64 * i >= d.pitch) continue;
      if constexpr (F16) {
#pragma unroll
        for (int j = 0; j < CH; j += 2) {           // C is even: both channels exist or neither
          reinterpret_cast<pair*>(image)[(j >> 1) * d.pitch + lane + 64 * i] = in[i] && c0 + j < g.C ? held[i][j >> 1] : pair(0);
        }
      } else {
#pragma unroll
        for (int j = 0; j < CH; ++j) reinterpret_cast<float*>(image)[j * d.pitch + lane + 64 * i] = in[i] && c0 + j < g.C ? held[i][j >> 1][j & 1] : 0.f;
      }
    }
  };
  // the lanes of a wavefront read what others of it have put
  auto meet = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  double fine[NT][4] = {};
  if (wave < d.units) fetch(wave);
  for (int unit = wave; unit < d.units; unit += waves) {
    put(unit);
    meet();
    if (unit + waves < d.units) fetch(unit + waves);
#pragma unroll
    for (int kh = 0; kh < 3; ++kh) {
      f32x4 row[NT];
#pragma unroll
      for (int kw = 0; kw < 3; ++kw) {
        const int t = kh * 3 + kw, shift = kh * wide + kw;
        if constexpr (F16) {
          h4 a;
#pragma unroll
          for (int k = 0; k < 4; ++k) a[k] = *reinterpret_cast<const _Float16*>(taps + l16 * kFilterPitch + ((quarter * 4 + k) * kTaps + t) * 2);
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const unsigned* p = reinterpret_cast<const unsigned*>(image) + quarter * 2 * d.pitch + at[j] + shift;
            row[j] = __builtin_amdgcn_mfma_f32_16x16x16f16(a, __builtin_bit_cast(h4, u32x2{p[0], p[d.pitch]}), kw == 0 ? f32x4(0) : row[j], 0, 0, 0);
          }
        } else {
          float a[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) a[k] = *reinterpret_cast<const float*>(taps + l16 * kFilterPitch + ((k * 4 + quarter) * kTaps + t) * 4);
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            f32x4 four[2];
#pragma unroll
            for (int k = 0; k < 2; ++k)
              four[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[k], reinterpret_cast<const float*>(image)[(k * 4 + quarter) * d.pitch + at[j] + shift], f32x4(0), 0, 0, 0);
            row[j] = kw == 0 ? four[0] + four[1] : row[j] + (four[0] + four[1]);
          }
        }
      }
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) fine[j][e] += (double)row[j][e];
    }
    meet();
  }

  // the wavefronts' sums meet: [wavefront][feature][point], element e of a tile is feature 4 (lane / 16) + e, point lane % 16
  constexpr int kResults = 16 * 16 * NT;
  double* const sums = reinterpret_cast<double*>(lds);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) sums[wave * kResults + (quarter * 4 + e) * (16 * NT) + j * 16 + l16] = fine[j][e];
  __syncthreads();
  for (int i = tid; i < kResults; i += blockDim.x) {
    const int f = f_first + i / (16 * NT), column = column0 + i % (16 * NT);
    double s = 0.0;
    for (int k = 0; k < waves; ++k) s += sums[k * kResults + i];
    if (f >= g.F || column > last) continue;
    const unsigned n = over((unsigned)column, g.results);
    y[((size_t)n * g.F + f) * g.results.by + ((unsigned)column - n * g.results.by)] = (float)s;
  }
}

// As many wavefronts as have something to do, and no more than it takes rounds for anyway.
int waves_of(int units, int most) {
  const int rounds = (units + most - 1) / most;
  return (units + rounds - 1) / rounds;
}

// Blocks that stay inside an image need fewer points of it (no step of two rows to the next one), and leave some of their own unused.
bool by_image(const Geometry& g, int points) { return g.N > 1 && g.HO * g.WO >= 8 * points; }
int run_of(const Geometry& g, int points) {
  const int most = by_image(g, points) ? g.HO * g.WO : g.columns, n = points < most ? points : most, wide = g.WO + 2;
  const long long hw = (long long)g.HO * g.WO, images = g.N == 1 || by_image(g, points) ? 0 : (n - 1 + hw - 1) / hw;
  const long long run = n - 1 + (n - 1 + g.WO - 1) / g.WO * 2 + images * 2 * wide + 2LL * wide + 3;
  return run > (1 << 20) ? 1 << 20 : (int)run;
}

struct Layout {
  int segment, units, waves, pitch, wave_bytes, points;
  long long blocks;
  bool far;                 // four points per lane, not two
};
Layout layout_of(const Geometry& g, int f16, int NT) {
  Layout l;
  const int run = run_of(g, 16 * NT), channels = f16 ? 16 : 8;
  l.far = run > 128;
  l.segment = by_image(g, 16 * NT) ? g.HO * g.WO : g.columns;
  l.units = (g.C + channels - 1) / channels;
  l.points = run;
  l.pitch = (run + 3) & ~3;
  l.wave_bytes = 32 * l.pitch + kFilterPitch * 16;
  const int room = (int)(kLds / (size_t)l.wave_bytes), most = most_waves(f16 ? 2 : 4, NT, l.far ? 4 : 2);
  l.waves = waves_of(l.units, room < most ? room : most);
  l.blocks = (long long)(g.columns / l.segment) * ((l.segment + 16 * NT - 1) / (16 * NT)) * ((g.F + 15) / 16);
  return l;
}

size_t lds_of(const Layout& l, int NT) {
  const size_t sums = (size_t)l.waves * 16 * 16 * NT * 8, own = (size_t)l.waves * l.wave_bytes;
  return own > sums ? own : sums;
}

template <typename T, int NT, int KP>
int launch(const void* x, const void* w, void* y, const Geometry& g, const Layout& l, hipStream_t st) {
  static bool configured = false;
  if (!configured) {
    ART_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(conv2d_direct_kernel<T, NT, KP>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds));
    configured = true;
  }
  const Direct d{l.units, l.segment, make_div((unsigned)((l.segment + 16 * NT - 1) / (16 * NT))), l.pitch, l.wave_bytes, (uintptr_t)w % 16 == 0};
  conv2d_direct_kernel<T, NT, KP><<<dim3((unsigned)l.blocks), dim3(64 * l.waves), lds_of(l, NT), st>>>((const T*)x, (const T*)w, (float*)y, g, d);
  ART_LAUNCH_CHECK();
  return 0;
}

template <typename T, int NT>
int run(const void* x, const void* w, void* y, const Geometry& g, hipStream_t st) {
  const Layout l = layout_of(g, sizeof(T) == 2, NT);
  return l.far ? launch<T, NT, 4>(x, w, y, g, l, st) : launch<T, NT, 2>(x, w, y, g, l, st);
}

}  // namespace

bool art::conv::direct_fits(const Geometry& g, int f16, int form) {
  return form >= 8 && form <= 10 && g.C % (f16 ? 8 : 4) == 0 && run_of(g, 16 << (form - 8)) <= 64 * kMostPoints &&
         (long long)g.F * g.C * kTaps * (f16 ? 2 : 4) < 1LL << 31 && layout_of(g, f16, 1 << (form - 8)).blocks < 1LL << 30;
}

// What a form takes, in microseconds: a fixed part, for each round of a block's wavefronts over the channels a time that grows with
// their number and with the points that a lane brings, and for blocks that share a compute unit, or do so unevenly, a time per unit of
// channels.  Fitted to 1465 times of 580 sizes, a third of them outside of 16 to 256 channels and features and 7 to 56 squared: 6 to 8 % off.
// Float16 blocks of which LDS holds two to a compute unit, five to seven wavefronts that take all channels in one turn over rows of some 40 to 128 points, take 1.3
// times that beyond one round (up to 2.0): 47 x 80 x 16 x 104 -> 11 34.6 us in another form, 59.9 here.  What is taken instead is 1.30 times as fast
// in the mean of 32 sizes of 60000 (up to 256 images, 1024 channels, 512 features, 128 x 128).  Not in float32 or for several turns: where it chose
// between the forms here, 0.90 and 0.75 to 0.95 times.
double art::conv::direct_time(const Geometry& g, int f16, int form) {
  struct Cost { double fixed, round, image, wave, shared, image_shared, uneven, image_uneven; };
  static const Cost cost[2][3] = {{{3.538, 0.0, 0.183, 0.183, 0.223, 0.058, 0.309, 0.026}, {4.356, 0.0, 0.178, 0.270, 0.362, 0.046, 0.0, 0.182}, {4.910, 1.472, 0.231, 0.290, 0.884, 0.010, 1.080, 0.0}},
                                  {{3.477, 0.0, 0.287, 0.244, 0.306, 0.034, 0.167, 0.150}, {3.966, 0.258, 0.303, 0.281, 0.521, 0.0, 0.496, 0.010}, {4.561, 1.144, 0.202, 0.285, 0.803, 0.0, 0.658, 0.0}}};
  const Cost& c = cost[f16 != 0][form - 8];
  const Layout l = layout_of(g, f16, 1 << (form - 8));
  const int items = (l.points + 63) / 64, turns = (l.units + l.waves - 1) / l.waves;
  const double rounds = (double)l.blocks / 256, full = rounds > 1 ? rounds : 1, uneven = ceil(rounds) > full ? ceil(rounds) - full : 0;
  const bool pairs = f16 && items == kMostPoints && turns == 1 && rounds > 1 && kLds / lds_of(l, 1 << (form - 8)) == 2;
  return c.fixed + (pairs ? 1.3 : 1.0) * (turns * (c.round + c.image * items + c.wave * l.waves) +
                                          l.units * ((c.shared + c.image_shared * items) * (full - 1) + (c.uneven + c.image_uneven * items) * uneven));
}

int art::conv::run_direct(const void* x, const void* w, void* y, const Geometry& g, int f16, int form, hipStream_t st) {
  static const decltype(&run<float, 1>) by_form[2][3] = {{run<float, 1>, run<float, 2>, run<float, 4>}, {run<_Float16, 1>, run<_Float16, 2>, run<_Float16, 4>}};
  return by_form[f16 != 0][form - 8](x, w, y, g, st);
}
