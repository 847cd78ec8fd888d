// Matrix products of small and odd sizes on the gfx950 matrix cores:
//
//   C[M, N] = A[M, K] @ B[K, N]      float16 (float32 sums, one rounding) or float32
//   C[M, N] = A[M, K] @ B[N, K]^T    int8 with int32 sums
//
// all row-major, any M, any N and K of at least one 16-byte vector.  Replaces, for these programs (AntaresIR.md:115), what
// the reference's tiled schedule generates (backends/c-rocm/schedule/standard/algo_tiling.py:35-98).
//
// Design for MI355X.  The kernels for large products (art_gemm_f16.hip, art_gemm_f32.hip) own 256 x 256 or 128 x 128 of C
// and need aligned rows; a product of a few hundred rows and columns gives them a handful of blocks for 256 compute
// units.  Here
//   * a block of 2 x 2 wavefronts owns 64 x 64, 64 x 128 or 128 x 128 of C and a slice of K; slices leave float32 (int32)
//     tiles that a second launch adds in order.  Block and slices come from an estimate of the launch time (`choose`);
//   * k goes in chunks of 128 bytes: global -> two register stages -> two LDS buffers, one LDS-only barrier per chunk,
//     loads two to three chunks ahead of their use and two to four blocks of a compute unit beside each other;
//   * every load is 16 bytes from any address: rows need no alignment.  A vector that would reach past the end of a row is
//     read where the row ends and shifted down on its way into LDS, zeros behind it; only the last chunk of K and the last
//     tile of columns do that.  Nothing outside the operands is read;
//   * rows of A (and of B in the transposed form) are 144 bytes apart in LDS, so that 16 lanes read 16-byte vectors from
//     all banks; B as it lies in memory, [k][n], is read with ds_read_b64_tr_b16 (float16) or 4 bytes at a time (float32);
//   * float32: a chunk of 32 values of k is summed by itself and then added to the total; where the generic lowering would
//     sum on the vector units in short slices (FINE, see `fine`), four values of k by themselves, these sums in pairs, and
//     the chunks and slices in float64.  One chain over k has 1.4e-7 (64 terms) to 1.1e-6 (4090) against 64 bits, the
//     generic kernels 1.4e-7 to 1e-6 and, in short slices, 0.7e-7 to 1.6e-7; this 1.1e-7 to 2.3e-7 and, FINE, 0.64e-7 to 0.73e-7;
//   * a chunk goes to LDS behind the products of the one before, float16 with a block per compute unit in front of them (see the loop);
//   * blocks on one XCD are a contiguous run of (slice, tile), its L2 holds what they share.
// Bound by latency below some 10 us - a launch, a chain of chunks whose loads L2 answers after several hundred
// nanoseconds, a second launch for slices -, then by the matrix instructions (float32) or the loads (64 x 64 blocks of float16
// fetch a byte per 32 operations).  Measured against what ran before (the generic lowering's tiles, padded copies and sliced
// sums, or the kernels for large products), us: float16 145 x 223 x 869 87 -> 8, 169 x 1158 x 2507 54 -> 12, 1792 x 128 x 3584
// 72 -> 12, 1024 x 2048 x 1024 27 -> 13, 136 x 448 x 104 4.5 -> 4.5; float32 320 x 192 x 512 94 -> 10, 391 x 239 x 503 19 -> 10,
// 1109 x 238 x 829 28 -> 16; int8 984 x 1904 x 1520 82 -> 11, 448 x 128 x 576 24 -> 5.  Geometric mean over 1260 sizes of 64 to 4096: 2.1,
// 1.5 and 1.6 times as fast; over 4200 with M, N or K below 64 or odd large ones: 2.0, 1.34 and 1.64.
#include <type_traits>

#include "art_conv2d.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_any __attribute__((ext_vector_type(4), aligned(1)));       // 16 bytes from any address
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr int kThreads = 256;
constexpr int kUnits = 256;                  // compute units of an MI355X
constexpr int kChunk = 128;                  // bytes of k of a row that are staged at a time
constexpr int kRow = kChunk + 16;            // bytes from row to row in LDS where k is contiguous

template <typename T> struct Elem;
template <> struct Elem<_Float16> {
  typedef h8 vec;
  typedef f32x16 acc;
  typedef float sum;
  typedef _Float16 out;
  static __device__ __forceinline__ acc multiply(vec a, vec b, acc c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
template <> struct Elem<float> {
  typedef f32x4 vec;
  typedef f32x16 acc;
  typedef float sum;
  typedef float out;
  // instruction m multiplies k = m (lanes 0-31) and k = 4 + m (lanes 32-63) of 8
  static __device__ __forceinline__ acc multiply(vec a, vec b, acc c, int first = 0, int last = 4) {
#pragma unroll
    for (int m = first; m < last; ++m) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[m], b[m], c, 0, 0, 0);
    return c;
  }
};
template <> struct Elem<signed char> {
  typedef i32x4 vec;
  typedef i32x16 acc;
  typedef int sum;
  typedef int out;
  static __device__ __forceinline__ acc multiply(vec a, vec b, acc c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
};

// The 16 bytes moved down by `bytes` (0 .. 16), zeros from above.
__device__ __forceinline__ u32x4 shifted_down(u32x4 v, unsigned int bytes) {
  unsigned long long lo = v[0] | (unsigned long long)v[1] << 32, hi = v[2] | (unsigned long long)v[3] << 32;
  if (bytes >= 8) { lo = hi; hi = 0; bytes -= 8; }
  if (bytes == 8) { lo = hi; bytes = 0; }
  const unsigned int r = 8 * bytes;
  lo = lo >> r | (hi << 1) << (63 - r);
  hi >>= r;
  return u32x4{(unsigned int)lo, (unsigned int)(lo >> 32), (unsigned int)hi, (unsigned int)(hi >> 32)};
}

__device__ __forceinline__ int xcd_unit(int b, int nb) {
  const int q = nb >> 3, r = nb & 7, xcd = b & 7, idx = b >> 3;
  return xcd < r ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
}

struct Sizes {
  int M, N, K;
  int row_tiles, col_tiles;
  int chunks, splits;          // chunks of K, cut into `splits` slices
  int slice, longer;           // chunks of a slice; the first `longer` slices have one more
  int blocks;
  int by_tile;                 // blocks are numbered by tile, then slice, not the other way round
  art::Div inner, shorter;     // splits or tiles, the smaller of row_tiles and col_tiles
};

// BT: B is [N, K].  TM, TN: 32 x 32 tiles of a wavefront along rows and columns.
template <typename T, bool BT, int TM, int TN, bool FINE>
__global__ __launch_bounds__(kThreads, TM * TN == 4 || (sizeof(T) == 4 && (TN == 2 || FINE)) ? 2 : 3) void gemm_tile_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                                                   typename Elem<T>::out* __restrict__ C,
                                                                                   typename Elem<T>::sum* __restrict__ partial, Sizes z) {
  typedef Elem<T> E;
  typedef typename E::vec vec;
  constexpr int S = sizeof(T), V = 16 / S, KC = kChunk / S;            // elements of a vector, of a chunk of k
  constexpr int BM = 64 * TM, BN = 64 * TN;
  constexpr int NA = BM / 32, NB = BN / 32;                            // vectors a thread stages per chunk
  constexpr int kBRow = BT ? kRow : S == 2 ? BN * 2 + 64 : BN * 4 + 32;        // bytes from row to row of B in LDS: neighbouring rows of k on other banks
  constexpr int kABytes = BM * kRow, kBuffer = kABytes + (BT ? BN : KC) * kBRow;
  extern __shared__ __align__(16) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, h = lane >> 5;
  // All arguments that the loads need in one trip, and no division: fetched and divided where they are used, they were five
  // trips and five divisions in front of the first load (float32 240 x 552 x 3200 19.8 -> 19.4 us, 336 x 320 x 1080 10.6 -> 9.8,
  // float16 159 x 776 x 2472 9.0 -> 8.6, 200 x 600 x 760 7.0 -> 6.6; int8 as before).
  asm volatile("" ::"s"(A), "s"(B), "s"(z.M), "s"(z.N), "s"(z.K), "s"(z.row_tiles), "s"(z.col_tiles), "s"(z.slice), "s"(z.longer), "s"(z.blocks),
               "s"(z.inner.mul), "s"(z.inner.shift), "s"(z.inner.by), "s"(z.by_tile), "s"(z.shorter.mul), "s"(z.shorter.shift), "s"(z.shorter.by));
  const int unit = xcd_unit(blockIdx.x, z.blocks), outer = (int)art::over((unsigned)unit, z.inner), rest = unit - outer * (int)z.inner.by;
  const int split = z.by_tile ? rest : outer, tile = z.by_tile ? outer : rest;
  // neighbours along the shorter side of the grid of tiles
  const int along = (int)art::over((unsigned)tile, z.shorter), across = tile - along * (int)z.shorter.by;
  const int tm = z.row_tiles < z.col_tiles ? across : along, tn = z.row_tiles < z.col_tiles ? along : across;
  const int m0 = tm * BM, n0 = tn * BN;
  const int first = split * z.slice + (split < z.longer ? split : z.longer), count = z.slice + (split < z.longer ? 1 : 0);

  // ---- what this thread stages.  Byte offsets; rows past M (N) repeat the last one: their products are not stored.
  unsigned int a_row[NA], a_k, b_row[NB], b_at[NB], b_shift[NB];
  a_k = (unsigned)(first * KC + (tid & 7) * V);                        // k of this thread's vectors of A (and of B^T)
  const unsigned k_last = (unsigned)(z.K - V);                         // where the last vector of a row starts
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int m = m0 + (tid >> 3) + 32 * i;
    a_row[i] = (unsigned)(m < z.M ? m : z.M - 1) * (unsigned)z.K * S;
  }
  constexpr int PB = BN * S / 16;                                      // vectors of a row of B
  unsigned int b_k = (unsigned)(first * KC + tid / PB);                // row of this thread's first vector of B; the others are 256 / PB rows apart
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if constexpr (BT) {
      const int n = n0 + (tid >> 3) + 32 * i;
      b_row[i] = (unsigned)(n < z.N ? n : z.N - 1) * (unsigned)z.K * S;
      b_at[i] = b_shift[i] = 0;
    } else {
      const int n = n0 + (tid % PB) * V, last = z.N - V;
      b_at[i] = (unsigned)(n < last ? n : last) * S;
      b_shift[i] = n <= last ? 0u : (unsigned)(n - last < V ? n - last : V) * S;
      b_row[i] = 0;
    }
  }
  const unsigned b_pitch = (unsigned)z.N * S, b_rows = (unsigned)z.K - 1;
  const bool ragged_n = !BT && n0 + BN > z.N && z.N % V != 0;         // vectors of B that would reach past a row's end
  const char* Ab = reinterpret_cast<const char*>(A);
  const char* Bb = reinterpret_cast<const char*>(B);

  u32x4 ga[2][NA], gb[2][NB];
  // The next chunk in order; past the last one of K the last vectors are read again, into a stage that nobody stores.
  auto fetch = [&](auto stage) {
    constexpr int R = decltype(stage)::value;
    const unsigned k = (a_k < k_last ? a_k : k_last) * S;
#pragma unroll
    for (int i = 0; i < NA; ++i) ga[R][i] = *reinterpret_cast<const u32x4_any*>(Ab + a_row[i] + k);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if constexpr (BT) {
        gb[R][i] = *reinterpret_cast<const u32x4_any*>(Bb + b_row[i] + k);
      } else {
        const unsigned r = b_k + i * (kThreads / PB);
        gb[R][i] = *reinterpret_cast<const u32x4_any*>(Bb + ((r < b_rows ? r : b_rows) * b_pitch + b_at[i]));
      }
    }
    a_k += KC;
    b_k += KC;
  };
  auto put = [&](int chunk, auto stage) {             // chunk: number in all of K
    constexpr int R = decltype(stage)::value;
    char* as = lds + (chunk - first & 1) * kBuffer;
    char* bs = as + kABytes;
    if (ragged_n || (chunk == z.chunks - 1 && z.K % KC != 0)) {
      const unsigned k = (unsigned)(chunk * KC + (tid & 7) * V), over = k <= k_last ? 0u : (k - k_last < V ? k - k_last : V) * S;
#pragma unroll
      for (int i = 0; i < NA; ++i) ga[R][i] = shifted_down(ga[R][i], over);
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const unsigned r = (unsigned)(chunk * KC + tid / PB + i * (kThreads / PB));
        gb[R][i] = shifted_down(gb[R][i], BT ? over : r <= b_rows ? b_shift[i] : 16u);
      }
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) *reinterpret_cast<u32x4*>(as + ((tid >> 3) + 32 * i) * kRow + (tid & 7) * 16) = ga[R][i];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if constexpr (BT) *reinterpret_cast<u32x4*>(bs + ((tid >> 3) + 32 * i) * kRow + (tid & 7) * 16) = gb[R][i];
      else *reinterpret_cast<u32x4*>(bs + (tid / PB + i * (kThreads / PB)) * kBRow + (tid % PB) * 16) = gb[R][i];
    }
  };

  typename E::acc acc[TM][TN];
  double fine[FINE ? 16 : 1];                         // FINE (one tile per wavefront): the total
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;
  if constexpr (FINE)
#pragma unroll
    for (int e = 0; e < 16; ++e) fine[e] = 0.0;

  // operands of 32 bytes of k: rows wm * 32 TM + 32 i + lane % 32 of A, columns wn * 32 TN + 32 j + lane % 32 of B
  const int s16 = lane & 15;
  auto multiply = [&](int buffer, auto steps) {       // steps of 32 bytes of k: all four, or the first two
    typename E::acc part[TM][TN], pair;               // float32: sums of the chunk (FINE: of the step before, of the first two steps)
    const char* as = lds + buffer * kBuffer + (wm * 32 * TM + (lane & 31)) * kRow + h * 16;
    const char* bs = lds + buffer * kBuffer + kABytes;
#pragma unroll
    for (int q = 0; q < decltype(steps)::value; ++q) {
      vec a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const vec*>(as + i * 32 * kRow + q * 32);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = wn * 32 * TN + j * 32;
        if constexpr (BT) {
          b[j] = *reinterpret_cast<const vec*>(bs + (n + (lane & 31)) * kRow + q * 32 + h * 16);
        } else if constexpr (S == 2) {
          // a transposing read takes 4 (k) x 16 (n) per 16 lanes and hands lane L the four k of column L
          const char* p = bs + (q * 16 + h * 8 + (s16 >> 2)) * kBRow + (n + (lane & 16) + (s16 & 3) * 4) * 2;
          const h4 lo = __builtin_bit_cast(h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p)));
          const h4 hi = __builtin_bit_cast(h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * kBRow)));
          b[j] = h8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
          const char* p = bs + (q * 8 + h * 4) * kBRow + (n + (lane & 31)) * 4;
#pragma unroll
          for (int m = 0; m < 4; ++m) b[j][m] = *reinterpret_cast<const float*>(p + m * kBRow);
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (S != 4) {
            acc[i][j] = E::multiply(a[i], b[j], acc[i][j]);
          } else if constexpr (!FINE) {
            part[i][j] = E::multiply(a[i], b[j], q == 0 ? typename E::acc(0) : part[i][j]);
          } else {
            const typename E::acc step = E::multiply(a[i], b[j], typename E::acc(0), 0, 2) + E::multiply(a[i], b[j], typename E::acc(0), 2, 4);
            if (q & 1) pair = q == 1 ? part[i][j] + step : pair + (part[i][j] + step);
            else part[i][j] = step;
          }
        }
    }
    if constexpr (FINE) {
#pragma unroll
      for (int e = 0; e < 16; ++e) fine[e] += (double)pair[e];
    } else if constexpr (S == 4) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += part[i][j];
    }
  };
  // float32, where the matrix instructions take most of the time: the half of a last chunk that is all zeros is left out
  const bool half_last = S == 4 && z.K % KC != 0 && z.K % KC <= KC / 2;
  auto multiply_chunk = [&](int t) {
    if (S == 4 && half_last && first + t == z.chunks - 1) multiply(t & 1, std::integral_constant<int, 2>{});
    else multiply(t & 1, std::integral_constant<int, 4>{});
  };

  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  fetch(S0{});
  fetch(S1{});
  __builtin_amdgcn_sched_barrier(0);
  put(first, S0{});
  fetch(S0{});
  art_lds_barrier();
  // Chunk t is in LDS buffer t % 2, chunk t + 1 in the other register stage, chunk t + 2 on its way.
  if constexpr (FINE) {                               // (its registers do not hold a loop with code behind it)
    for (int t = 0; t < count; t += 2) {
      multiply_chunk(t);
      if (t + 1 == count) break;
      put(first + t + 1, S1{});
      fetch(S1{});
      art_lds_barrier();
      multiply_chunk(t + 1);
      if (t + 2 == count) break;
      put(first + t + 2, S0{});
      fetch(S0{});
      art_lds_barrier();
    }
  } else {
    // No exit in the middle of the loop: one that leaves behind an odd chunk makes the compiler wait for chunk t + 2's loads where
    // chunk t + 1 goes to LDS (2 to 4 % over 300 sizes).  EARLY: the next chunk goes to LDS in front of the products, not behind
    // them; with a block of its own on each compute unit nothing else hides that (float16 192 x 3656 x 2944 19.9 -> 16.9 us, 968 x
    // 1880 x 3928 40.5 -> 34.8), with two to three it is slower (1472 x 1920 x 3136 39.8 -> 44.1); float32 and int8 gain nothing.
    auto loop = [&](auto early) {
      constexpr bool EARLY = decltype(early)::value;
      auto step = [&](int chunk, auto buffer, auto stage) {
        using Four = std::integral_constant<int, 4>;
        if constexpr (!EARLY) multiply(decltype(buffer)::value, Four{});
        put(chunk, stage);
        fetch(stage);
        if constexpr (EARLY) multiply(decltype(buffer)::value, Four{});
        art_lds_barrier();
      };
      int t = 0;
      for (; t + 2 < count; t += 2) {
        step(first + t + 1, S0{}, S1{});
        step(first + t + 2, S1{}, S0{});
      }
      return t;
    };
    const int t = S == 2 && z.blocks <= kUnits ? loop(std::true_type{}) : loop(std::false_type{});
    multiply_chunk(t);
    if (t + 1 < count) {
      put(first + t + 1, S1{});
      art_lds_barrier();
      multiply_chunk(t + 1);
    }
  }

  if constexpr (FINE)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[0][0][e] = (float)fine[e];

  // accumulator element e: row (e / 4) * 8 + 4 h + e % 4 of the tile, column lane % 32
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn * 32 * TN + j * 32 + (lane & 31);
    if (n >= z.N) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm * 32 * TM + i * 32 + (e >> 2) * 8 + h * 4 + (e & 3);
        if (m >= z.M) continue;
        const size_t at = (size_t)m * z.N + n;
        if (z.splits > 1) partial[(size_t)split * z.M * z.N + at] = acc[i][j][e];
        else C[at] = (typename E::out)acc[i][j][e];
      }
  }
}

// C = sum of the slices' tiles, in order.  Block b takes the eighth b % 8 of the columns of `rows` rows of 4 `quads` elements (rows 1: of all
// elements; 0: blocks in order).  Four neighbouring elements per thread, eight slices requested at a time.
template <typename Sum, typename Total, typename Out>
__global__ __launch_bounds__(256) void gemm_tile_sum_kernel(const Sum* __restrict__ partial, Out* __restrict__ C, long long count, int splits, int rows, int quads,
                                                           unsigned mul, unsigned shift, unsigned by) {      // Div of an eighth, as numbers: these are in registers when a kernel starts
  typedef Sum sum4 __attribute__((ext_vector_type(4), aligned(4)));
  typedef Total total4 __attribute__((ext_vector_type(4)));
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (rows > 0) {
    const unsigned at = (blockIdx.x >> 3) * 256 + threadIdx.x, row = rows > 1 ? art::over(at, art::Div{mul, shift, by}) : at < by ? 0 : 1;
    const unsigned quad = (blockIdx.x & 7) * by + at - row * by;
    if ((int)row >= rows || (int)quad >= quads) return;
    i = (long long)row * quads + quad;
  }
  i *= 4;
  if (i >= count) return;
  if (i + 4 <= count) {
    total4 t = __builtin_convertvector(*reinterpret_cast<const sum4*>(partial + i), total4);
    for (int s0 = 1; s0 < splits; s0 += 8) {
      sum4 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const sum4*>(partial + (s0 + j < splits ? s0 + j : 0) * count + i);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (s0 + j < splits) t += __builtin_convertvector(v[j], total4);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) C[i + k] = (Out)t[k];
    return;
  }
  for (long long k = i; k < count; ++k) {
    Total t = (Total)partial[k];
    for (int s = 1; s < splits; ++s) t += (Total)partial[s * count + k];
    C[k] = (Out)t;
  }
}

// Where the slices are added.  Blocks run on the XCDs in runs; numbered by tile, an XCD has all slices of an eighth of the tiles, which is an
// eighth of the rows or, where there are more columns of tiles, of the columns, and the pass adds them on that XCD, from its L2.  Numbered by
// slice, every XCD reads but its part of k of the operands.  By tile
//  * from 16 tiles on: with 8 to 15 of them 0.98 times as fast by tile, with fewer 0.94;
//  * an eighth of the columns only with 800 of them and more, or of whole lines (partial sums, N % 256 == 0): of 640 to 800 others 8 of 21 were 3 to
//    5 % slower by tile, 1.00 times as fast in the mean;
//  * as long as an XCD's L2 (4 MiB) holds the operands that it reads then, an eighth of the longer one and all of the other.  Beyond that
//    0.97 times as fast in float16 (633 x 1136 x 3597 20.9 us by slice, 24.0 by tile), up to it 1.05; float32, more bound by its products, 1.015 between 4 and
//    6 MiB, 0.99 beyond.
// Over 490 products of 16 tiles and more, up to 4096 x 4096 x 4096, 1.03 times as fast as all by slice, at worst 7 % slower.  us, by slice and by tile: float16 448 x 512 x 1344 8.0 -> 7.2, 704 x 472 x 2128 11.9 -> 10.2, float32 128 x 1600 x 640
// 10.1 -> 9.0, int8 3592 x 64 x 3048 8.5 -> 7.3; by slice it stays at 6.2 for int8 128 x 192 x 3328 (7.6 by tile).
bool numbered_by_tile(int type, int M, int N, int K, int row_tiles, int col_tiles) {
  const long long longer = M > N ? M : N, shorter = M > N ? N : M;
  return (long long)row_tiles * col_tiles >= 16 && (row_tiles >= col_tiles || (N % 4 == 0 && N >= 640 && (N >= 800 || N % 256 == 0))) &&
         (longer / 8 + shorter) * K * (type == 0 ? 2 : type == 1 ? 4 : 1) <= (type == 1 ? 6LL << 20 : 4LL << 20);
}

template <typename Sum, typename Total, typename Out>
void launch_sum(const Sum* partial, Out* C, long long count, int splits, int rows, hipStream_t stream) {
  const long long quads = (count / (rows > 0 ? rows : 1) + 3) / 4, eighth = (quads + 7) / 8;
  const unsigned blocks = rows > 0 ? 8u * (unsigned)((rows * eighth + 255) / 256) : (unsigned)((quads + 255) / 256);
  const art::Div of = art::make_div((unsigned)eighth);
  gemm_tile_sum_kernel<Sum, Total, Out><<<dim3(blocks), dim3(256), 0, stream>>>(partial, C, count, splits, rows, (int)quads, of.mul, of.shift, of.by);
}

// Forms: 1 = 64 x 64 per block, 2 = 64 x 128, 3 = 128 x 128 (not float32: no registers left for the chunk's sums), 4 = 64 x 64
// summed FINE (float32 only).
int rows_of(int form) { return form == 3 ? 128 : 64; }
int columns_of(int form) { return form == 1 || form == 4 ? 64 : 128; }
int size_of(int type) { return type == 0 ? 2 : type == 1 ? 4 : 1; }
int chunks_of(int type, int K) { const int kc = kChunk / size_of(type); return (K + kc - 1) / kc; }

bool has(int type, int form) { return form == 1 || form == 2 || form == (type == 1 ? 4 : 3); }

// Sizes the kernel takes: offsets are 32-bit (a chunk and more past the end of B before they are clamped).
bool takes(int type, int M, int N, int K) {
  if (type < 0 || type > 2) return false;
  const long long s = size_of(type), v = 16 / s, most = 1LL << 32;
  if (M < 1 || N < 1 || K < v || (type != 2 && N < v)) return false;
  const long long wide = K + 4 * kChunk;
  return (long long)M * wide * s < most && (long long)N * wide * s < most && (long long)((M + 63) / 64) * ((N + 63) / 64) < 1 << 24;
}

// What a launch takes, in microseconds: a fixed part; per chunk of a block's slice a time that grows with the blocks that
// share a compute unit and with how unevenly they do; the stores; and for slices the second launch and the tiles between.
// Fitted to 7000 launches (387 sizes of 64 to 4096 in M, N, K, odd ones among them), 5 % off.  Over 1270 other sizes of that range the
// form and slices it picks are 1.2 (float16), 0.5 (float32) and 0.4 % (int8) slower than the fastest ones in the mean, over 4260 outside
// of it (M or N down to 1 and up to 16384, K of 4 to 16384) 1.4, 1.0 and 1.6 %.
struct Cost { double fixed, alone, shared, uneven; };
struct Rest { double sum, sum_bytes, store; };
constexpr Cost kCost[3][3] = {{{3.67, 0.321, 0.210, 0.195}, {4.81, 0.494, 0.361, 0.272}, {6.17, 0.753, 0.439, 0.310}},
                              {{3.24, 0.816, 0.514, 0.574}, {4.22, 1.360, 1.031, 1.048}, {3.35, 1.114, 0.736, 0.628}},
                              {{3.55, 0.309, 0.217, 0.294}, {4.57, 0.452, 0.432, 0.370}, {5.83, 0.731, 0.502, 0.501}}};
constexpr Rest kRest[3] = {{2.31, 0.408, 0.425}, {2.73, 0.388, 0.242}, {2.09, 0.403, 0.208}};       // per million floats, per million bytes
double launch_time(int type, int M, int N, int K, int form, int splits) {
  const Cost& c = kCost[type][form > 2 ? 2 : form - 1];
  const Rest& r = kRest[type];
  const double tiles = (double)((M + rows_of(form) - 1) / rows_of(form)) * ((N + columns_of(form) - 1) / columns_of(form));
  const double rounds = tiles * splits / kUnits, full = rounds > 1 ? rounds : 1, million = 1e-6 * M * N, out = type == 0 ? 2 : 4;
  const int per_slice = (chunks_of(type, K) + splits - 1) / splits;
  const double t = c.fixed + per_slice * (c.alone + c.shared * (full - 1) + c.uneven * (ceil(rounds) > full ? ceil(rounds) - full : 0));
  return splits == 1 ? t + r.store * out * million : t + r.sum + r.sum_bytes * (splits + out / 8) * 4 * million;
}
// The same for the kernels for large aligned products: blocks of 256 x 256 (float16) or 128 x 128 (float32), one per
// compute unit and round.  Fitted to 96 and 23 sizes, 4 and 3 % off; the lower of the two estimates is the faster kernel for
// all of them but two of float32, by up to 7 %: 4096 x 4096 x 4096 130 us there and 185 here, 2048 x 2048 x 2048 50 and 34,
// 1024 x 1024 x 1024 24 and 9; float32 2048 x 2048 x 2048 135 and 152, 1024 x 2048 x 1024 67 and 46.
double large_time(int type, int M, int N, int K) {
  const double side = type == 0 ? 256 : 128, rounds = ceil(ceil(M / side) * ceil(N / side) / kUnits), million = 1e-6 * M * N;
  return type == 0 ? 5.26 + rounds * (0.0184 * K + 2.54) + 0.719 * million : 5.15 + rounds * 0.0601 * K + 0.655 * million;
}
// Where the generic lowering has no matrix instructions for the product: it sums on the vector units.
bool on_vector_units(int M, int N, int K) { return M < 32 || N < 32 || K < 32 || (long long)((M + 63) / 64) * ((N + 63) / 64) < 16; }
// Float32 products whose k is spread over a wavefront or a block there: from 64 values of k on, below 65536 results.  Their sums are
// 0.7e-7 to 1.6e-7 from 64 bits over 1100 sizes (M or N down to 1); the chunk sums have 1.05e-7 to 1.9e-7, above it for K of 64 to some 900
// (7104 x 4 x 128 0.74e-7 and 1.14e-7, 1 x 10453 x 637 0.91 and 1.36), FINE 0.64e-7 to 0.73e-7.  A thread for each result is a chain over k:
// the chunk sums have its error up to 32 values of k and less from there on (0.44 times with 65536 and more results).  On the matrix
// instructions they are at or below it at all 1750 sizes.
bool fine(int type, int M, int N, int K, bool large) { return type == 1 && !large && on_vector_units(M, N, K) && K >= 64 && (long long)M * N < 65536; }

// The generic lowering's time, on the vector units and on the matrix instructions, or a time that nothing reaches where it was not
// the faster one.  Fitted to 4100 sizes, M and N of 1 to 16384, K of 4 to 16384, odd ones among them: where the two are within a factor of
// two of each other 6 to 17 % off (25 % for float32 of 65536 and more results).  The kernel picked is 0.4 to 4.5 % slower than the
// faster one in the mean of a kind.
double generic_time(int type, int M, int N, int K) {
  const double million = 1e-6 * M * N, kk = K / 64.0;
  if (on_vector_units(M, N, K)) {
    // a thread per result, or per 4 x 4 of them; a wavefront per result, its k across the lanes; sums in two launches; a thread per
    // result again.  Per launch, 64 values of k, million products, and million results (wavefronts: products, where a row of B is
    // not one line: neighbouring k are then lines of their own).  us, generic / here:
    // float16 24 x 61 x 446 3.9 / 6.2, 1088 x 24 x 192 8.5 / 4.3, 1440 x 56 x 24 3.3 / 4.0, 8 x 3968 x 1024 113 / 6.4; float32
    // 64 x 6 x 832 3.5 / 8.9, 45 x 704 x 192 15.5 / 7.7, 5 x 9920 x 5376 1870 / 68; int8 920 x 1 x 370 3.1 / 4.6, 23 x 963 x 105 6.9 / 4.1.
    struct Units { double fixed, k, products, rest; };
    constexpr Units kShort[3] = {{2.459, 1.542, 0.212, 0.7}, {2.439, 1.6, 0.18, 1.307}, {2.412, 1.098, 0.205, 1.026}};
    constexpr Units kPatch[2] = {{1.064, 9.852, 0.048, 0.728}, {2.099, 7.648, 0.058, 1.219}};
    constexpr Units kWave[3] = {{2.928, 0.042, 0.91, 0.911}, {2.753, 0.053, 0.874, 1.287}, {3.024, 0.0, 0.869, 0.025}};
    constexpr Units kSliced[3] = {{6.354, 0.0, 0.701, 1.325}, {3.698, 0.039, 0.605, 2.055}, {5.306, 0.016, 0.248, 0.0}};
    constexpr Units kThread[2] = {{1.47, 1.61, 0.113, 8.452}, {0.345, 2.65, 0.191, 5.087}};
    const double results = (double)M * N, line = (double)N * size_of(type) / 128, apart = million * K * (line < 1 ? line : 1);
    auto time = [&](const Units& u, double rest) { return u.fixed + u.k * kk + u.products * million * K + u.rest * rest; };
    if (K < 64) return type != 2 && results >= 131072 * 16 && M % 4 == 0 && N % 4 == 0 && K >= 8 ? time(kPatch[type], million) : time(kShort[type], million);
    if (type != 2 && results >= 65536) return time(kThread[type], million);
    if (K < 1024 || results > 8192) return time(kWave[type], apart);
    // a long k and hardly any results: float32 72 x 8 x 16352 23 / 31, int8 31 x 2 x 6301 4.2 / 8.8, in the mean 1.9 and 1.2 times as fast
    // there; float16 here where the estimate, 17 % off, is a fifth below: 8 x 128 x 7904 31 / 7.6, 47 x 9 x 4106 4.3 / 11.7
    if (results > 1024) return time(kSliced[type], apart);
    return type == 0 ? time({4.345, 0.006, 0.619, 1.204}, apart) : 0.0;
  }
  // Operands that the matrix kernels fetch in whole vectors and results that leave in whole lines; elsewhere, and in float32, they are 5 %
  // faster at the most (int8 1472 x 1216 x 41: 10) and up to 2.9 times slower (int8 5369 x 3613 x 80 55 / 19, float16 7212 x 8134 x 615 390 / 175).
  if (type == 1 || K % (16 / size_of(type)) != 0 || N % (type == 0 ? 8 : 16) != 0) return 1e30;
  // Blocks of 128 x 128 or 64 x 64 as it chooses them (plans.py); taken where it is a tenth faster by this estimate, 9 % off.  us,
  // generic / here: float16 4672 x 4992 x 32 20.4 / 24.9, 2216 x 7464 x 216 41.1 / 33.6; int8 4608 x 15168 x 64 56 / 66, 2176 x 2880 x 32
  // 8.3 / 9.4, 3392 x 1664 x 192 9.8 / 10.0, 4096 x 4096 x 4096 106 / 98.  0.5 to 2.3 % off the faster one in the mean, at single sizes up to
  // 16 % slower than it (int8 5952 x 1088 x 320 10.6 / 12.2).
  constexpr Cost kMatrix[2][2] = {{{3.9, 0.588, 0.091, 0.34}, {5.562, 0.895, 0.945, 0.332}}, {{4.236, 0.209, 0.169, 0.264}, {4.462, 0.507, 0.449, 0.15}}};
  constexpr double kStore[2][2] = {{0.443, 0.694}, {0.395, 0.701}};
  const long long big = (long long)((M + 127) / 128) * ((N + 127) / 128), small = (long long)((M + 63) / 64) * ((N + 63) / 64);
  const int side = small < 700 * ((big + 511) / 512) ? 0 : 1;
  const Cost& c = kMatrix[type / 2][side];
  const double rounds = (double)(side ? big : small) / kUnits, full = rounds > 1 ? rounds : 1;
  return 1.1 * (c.fixed + kk * (c.alone + c.shared * (full - 1) + c.uneven * (ceil(rounds) - full)) + kStore[type / 2][side] * million);
}

// What a block's columns past a row's last whole vector cost, per chunk: they are shifted on their way into LDS.  For all columns of a
// thin product, 0.18 us between rows of whole vectors and others in float16, 0.19 in float32.  Not part of the choice of slices.
double ragged_time(int type, int N, int K, int splits) {
  return type == 2 || N % (16 / size_of(type)) == 0 ? 0.0 : 0.12 * ((chunks_of(type, K) + splits - 1) / splits);
}

// 256 * form + slices for these sizes, or 0: another kernel is faster.  `large`: the kernel for large products takes
// them.  `own`: the best of the forms here, whatever the others take.  Slices take 128 MiB at the most: of 6000 float32 products of 1000 to
// 4096 two would take more, and lose 1 % by the estimate (with 64 MiB 6 % of them up to 5 %).
constexpr long long kMostSlices = 1LL << 25;                 // float32 (int32) values
int choose(int type, int M, int N, int K, bool large, bool own) {
  if (!takes(type, M, N, K)) return 0;
  const long long results = (long long)M * N;
  const int chunks = chunks_of(type, K);
  const bool short_sums = fine(type, M, N, K, large);
  double best = 1e30;
  int code = 0;
  for (int form = 1; form <= 4; ++form) {
    if (!has(type, form) || (type == 1 && (form == 4) != short_sums)) continue;
    for (int splits : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 24}) {
      if (splits > chunks || (splits > 1 && splits * results > kMostSlices)) break;
      const double t = launch_time(type, M, N, K, form, splits);
      if (t < best) { best = t; code = 256 * form + splits; }
    }
  }
  if (own) return code;
  if (large) return best < large_time(type, M, N, K) ? code : 0;
  return best + ragged_time(type, N, K, code & 255) < generic_time(type, M, N, K) ? code : 0;
}

template <typename T, bool BT, int TM, int TN, bool FINE = false>
int launch(const void* a, const void* b, void* c, void* partial, const Sizes& z, hipStream_t st) {
  constexpr int S = sizeof(T), BM = 64 * TM, BN = 64 * TN;
  constexpr int bytes = 2 * (BM * kRow + (BT ? BN * kRow : kChunk / S * (S == 2 ? BN * 2 + 64 : BN * 4 + 32)));
  static bool configured = false;
  if (!configured) {
    ART_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_kernel<T, BT, TM, TN, FINE>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    configured = true;
  }
  gemm_tile_kernel<T, BT, TM, TN, FINE><<<dim3((unsigned)z.blocks), dim3(kThreads), bytes, st>>>(
      (const T*)a, (const T*)b, (typename Elem<T>::out*)c, (typename Elem<T>::sum*)partial, z);
  ART_LAUNCH_CHECK();
  return 0;
}

template <typename T, bool BT>
int run(const void* a, const void* b, void* c, void* partial, const Sizes& z, int form, hipStream_t st) {
  int rc;
  if (form == 1) rc = launch<T, BT, 1, 1>(a, b, c, partial, z, st);
  else if (form == 2) rc = launch<T, BT, 1, 2>(a, b, c, partial, z, st);
  else if constexpr (sizeof(T) == 4) rc = launch<T, BT, 1, 1, true>(a, b, c, partial, z, st);
  else rc = launch<T, BT, 2, 2>(a, b, c, partial, z, st);
  if (rc) return rc;
  if (z.splits == 1) return 0;
  const long long count = (long long)z.M * z.N;
  typedef typename std::conditional<sizeof(T) == 4, double, typename Elem<T>::sum>::type total;
  launch_sum<typename Elem<T>::sum, total, typename Elem<T>::out>((const typename Elem<T>::sum*)partial, (typename Elem<T>::out*)c, count, z.splits,
                                                                   z.by_tile ? (z.row_tiles < z.col_tiles ? z.M : 1) : 0, st);
  ART_LAUNCH_CHECK();
  return 0;
}

}  // namespace

int art::sum_slices(const float* partial, float* y, long long count, int slices, hipStream_t stream) {
  launch_sum<float, double, float>(partial, y, count, slices, 0, stream);
  ART_LAUNCH_CHECK();
  return 0;
}

extern "C" int art_gemm_tile_form(int type, int M, int N, int K, int large, int form, int splits) {
  if (form == 0) return choose(type, M, N, K, large != 0, splits != 0);
  return takes(type, M, N, K) && has(type, form) && splits >= 1 && splits <= 64 && splits <= chunks_of(type, K) ? 256 * form + splits : 0;
}

extern "C" int art_gemm_tile(const void* a_dev, const void* b_dev, void* c_dev, void* partial_dev, int type, int M, int N, int K, int form, int splits,
                             void* stream) {
  ART_REQUIRE(takes(type, M, N, K) && has(type, form), "art_gemm_tile: sizes the kernel does not take (type %d, M=%d N=%d K=%d, form %d)", type, M, N, K, form);
  const int chunks = chunks_of(type, K);
  ART_REQUIRE(splits >= 1 && splits <= chunks && splits <= 64, "art_gemm_tile: 1 to 64 slices of at least a chunk (got %d of %d chunks)", splits, chunks);
  ART_REQUIRE(a_dev && b_dev && c_dev && (splits == 1 || partial_dev), "art_gemm_tile: null pointer");
  const uintptr_t s = size_of(type), out = type == 0 ? 2 : 4;
  ART_REQUIRE((uintptr_t)a_dev % s == 0 && (uintptr_t)b_dev % s == 0 && (uintptr_t)c_dev % out == 0 && (uintptr_t)partial_dev % 16 == 0,
              "art_gemm_tile: misaligned tensor");
  ART_REQUIRE(!art::overlaps(c_dev, (size_t)M * N * out, a_dev, (size_t)M * K * s) && !art::overlaps(c_dev, (size_t)M * N * out, b_dev, (size_t)N * K * s),
              "art_gemm_tile: the result must not overlap an operand");
  const int row_tiles = (M + rows_of(form) - 1) / rows_of(form), col_tiles = (N + columns_of(form) - 1) / columns_of(form);
  const int tiles = row_tiles * col_tiles, by_tile = splits > 1 && numbered_by_tile(type, M, N, K, row_tiles, col_tiles);
  const Sizes z{M, N, K, row_tiles, col_tiles, chunks, splits, chunks / splits, chunks % splits, tiles * splits,
                by_tile, art::make_div((unsigned)(by_tile ? splits : tiles)), art::make_div((unsigned)(row_tiles < col_tiles ? row_tiles : col_tiles))};
  hipStream_t st = (hipStream_t)stream;
  return type == 0 ? run<_Float16, false>(a_dev, b_dev, c_dev, partial_dev, z, form, st)
       : type == 1 ? run<float, false>(a_dev, b_dev, c_dev, partial_dev, z, form, st)
                   : run<signed char, true>(a_dev, b_dev, c_dev, partial_dev, z, form, st);
}
