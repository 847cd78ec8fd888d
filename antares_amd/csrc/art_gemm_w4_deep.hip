// Weight-only int4 GEMM for small products (4 to 512 rows): the arithmetic of art_gemm_w4.hip,
//     y[m,n] = sum_k x[m,k] * w[k,n],   w[k,n] = fp16(s[g,n] * fp16(q[k,n] - z[g,n])),   group g = k / 128,
// on the matrix cores with fp32 accumulation, for sizes where that kernel's blocks of 128 columns either leave most of the chip
// without work or need K-splits, whose sums a second launch adds: a chain of groups one after another, or two launches.
//
//   * a block owns 16, 32 or 64 rows, 32 columns (or 64, with up to 32 rows) and all of K (or of a K split); its eight wavefronts
//     take the quantisation groups in turn, so that K is worked on eight-fold in parallel without a second launch, and meet once, at the
//     end, in LDS;
//   * a wavefront works by itself: what its next group needs - 2 or 4 KiB of packed weights, their scales and zero points, 4 to 16 KiB of x -
//     goes from global memory into LDS of its own (no barrier in the loop), into the place that the group before has just been read
//     from.  Fetching weights two or three groups ahead was slower (16 rows over 4096 x 4096 7.5 -> 8.4 and 9.0 us): the loads that are
//     needed first queue behind them;
//   * the blocks of a tile's rows share its weights, neighbouring tiles the lines of the packed weights (32 or 64 of 128 bytes a row): they run
//     on one XCD, at the same time.
//
// What bounds it: the launch and one trip to memory (3.0 us) at the smallest sizes; beyond them the load path of a compute unit, 0.1 to 0.2 us a
// group for all eight wavefronts - every block takes in all of x, and a row's 32 bytes of weights cost it as much as 64.  64 columns halve both,
// with half as many blocks: better from some 150 of them on.  64 rows of x and 64 columns do not fit LDS.
// Measured (MI355X, weights from the last-level cache; the best form of the kernels before -> this one): 16 rows over 1024 x 1024 6.0 -> 3.7 us, 1024 x 5376
// 6.9 -> 4.5, 2048 x 6144 8.4 -> 6.0, 4096 x 4096 8.6 -> 7.5, 4096 x 12288 13.1 -> 10.9; 32 rows over 2048 x 2048 7.2 -> 5.2, 2048 x 10752
// 10.2 -> 7.6; 64 rows over 1024 x 5376 7.1 -> 5.9, 2048 x 6144 10.5 -> 8.1, and not better over 4096 x 12288 (16.2 and 21.8).  Sizes of 512 to
// 11008 x 512 to 14700, geometric mean where the better of both is taken (art_gemm_w4.hip chooses): 1.31 times up to 16 rows, 1.25 up to 32, 1.16 up to
// 128, 1.08 up to 256, 1.05 up to 512.
#include "art_w4_mfma.h"

#include <type_traits>

namespace {

using namespace art::w4;

template <int V> using Int = std::integral_constant<int, V>;

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int GK = 128;
constexpr int Q_BYTES = 512;                        // scales at 0, zero points at 256; the rest takes the idle lanes
constexpr int w_bytes(int CT) { return (GK / 2) * 32 * CT; }
constexpr int wave_bytes(int XR, int CT) { return w_bytes(CT) + Q_BYTES + XR * GK * 2; }
constexpr size_t lds_bytes(int XR, int CT) { return (size_t)kWaves * wave_bytes(XR, CT); }      // 52, 68, 84, 100, 148 KB

// XR: rows of x that are fetched (16, 32, 64); rows past M repeat the last one.  CT: 32-column tiles of a block.
template <int XR, int CT, Tail TAIL>
__global__ __launch_bounds__(kThreads, XR == 16 ? 4 : 2) void gemm_w4a16_deep_kernel(
    const _Float16* __restrict__ x, const unsigned char* __restrict__ qweight, const _Float16* __restrict__ scales,
    const unsigned char* __restrict__ qzeros, int K, int N, int M, int inner, unsigned int inv_inner, int each, int units, int m_blocks, unsigned int inv_blocks, _Float16* y, float* __restrict__ partial,
    int splits, int groups_of_split, int longer, Magic mg, const _Float16* residual, Rope rope) {
  constexpr int MT = XR == 64 ? 2 : 1, BN = 32 * CT, W_BYTES = w_bytes(CT);
  constexpr int XL = XR / 4, WL = W_BYTES / 1024;   // loads of x and of the packed weights per group
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  asm volatile("" ::"s"(units), "s"(m_blocks), "s"(inv_blocks), "s"(splits), "s"(groups_of_split), "s"(longer));      // all of them are asked for before the first branch
  int unit = (blockIdx.x & 7) * each + (blockIdx.x >> 3);            // (tile, K split, block of rows); neighbours on one XCD
  if (unit >= units) return;
  int m0 = 0;
  if (m_blocks > 1) {
    const int block = unit;
    unit = (int)__umulhi(block, inv_blocks);        // block / m_blocks
    m0 = (block - unit * m_blocks) * XR;
  }
  const int across = inner < 0 ? -inner : inner, outer = inv_inner ? (int)__umulhi(unit, inv_inner) : unit, rest = unit - outer * across;      // unit / across
  const int tile = inner < 0 ? rest : outer, split = inner < 0 ? outer : rest;
  const int g_begin = split * groups_of_split + (split < longer ? split : longer), g_count = groups_of_split + (split < longer ? 1 : 0);
  const int mine = (g_count - wave + kWaves - 1) / kWaves;           // groups wave, wave + 8, ... of the split

  // The block's columns, in pieces of 16: two of a tile are neighbours, a gate's and its up projection's (kSwiglu), or 64 columns of a
  // head apart (kRope).  A piece is inside the matrix or outside of it as a whole.
  const int n0 = tile * (TAIL == kPlain ? BN : BN / 2);
  auto piece_at = [&](int piece) {                  // its first column
    const int n = n0 + (piece >> 1) * 16;
    if (TAIL == kPlain) return n0 + piece * 16;
    if (TAIL == kSwiglu) return (piece & 1) * (N / 2) + n;
    return (n >> 6) * 128 + (n & 63) + (piece & 1) * 64;
  };
  auto inside = [&](int piece) { return TAIL == kPlain ? n0 + piece * 16 < N : TAIL == kRope || n0 + (piece >> 1) * 16 < N / 2; };
  auto safe = [&](int pos) { return inside(pos >> 4) ? piece_at(pos >> 4) + (pos & 15) : 0; };

  unsigned char* const own = smem + wave * wave_bytes(XR, CT);
  unsigned char* const own_x = own + W_BYTES + Q_BYTES;
  const unsigned int lds_own = (unsigned int)(size_t)(__attribute__((address_space(3))) unsigned char*)smem + wave * wave_bytes(XR, CT);
  const int s16 = lane & 15, hi16 = (lane >> 4) & 1, h = lane >> 5;

  f16v acc[MT][CT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][ct][r] = 0.f;

  if (mine > 0) {
    const int g0 = g_begin + wave;
    Rows<false> w_rows(qweight + (size_t)g0 * (GK / 2) * N, kWaves * (GK / 2) * N, mine), x_rows(x + (size_t)m0 * K + (size_t)g0 * GK, kWaves * GK * 2, mine),
        s_rows(scales + (size_t)g0 * N, kWaves * 2 * N, mine), z_rows(qzeros + (size_t)g0 * (N / 2), kWaves * (N / 2), mine);
    // Position (row, piece p) of the packed weights holds piece p, with two tiles p ^ (2 in every other four rows): the 32 lanes of a
    // transposing read, 8 rows of two pieces, touch every bank once.
    constexpr int P = 2 * CT;                       // pieces of a row
    auto swizzle = [](int row) { return CT == 1 ? 0 : ((row >> 2) & 1) * 2; };
    unsigned int woff[WL], xoff[XL];
#pragma unroll
    for (int u = 0; u < WL; ++u) {
      const int r = u * (64 / P) + lane / P;
      woff[u] = (unsigned int)r * N + safe(((lane & (P - 1)) ^ swizzle(r)) * 16);
    }
    const unsigned int soff = 2u * safe((2 * lane) & (BN - 1)), zoff = (unsigned int)safe((8 * lane) & (BN - 1)) >> 1;
#pragma unroll
    for (int u = 0; u < XL; ++u) {
      const int r = 4 * u + (lane >> 4);
      xoff[u] = (unsigned int)(m0 + r < M ? r : M - 1 - m0) * (2 * K) + (((lane & 15) ^ (r & 15)) * 16);
    }
    auto fetch_x4 = [&](auto u_tag) {
      constexpr int U = decltype(u_tag)::value;
      const unsigned int to = lds_own + W_BYTES + Q_BYTES;
      buffer_lds_x4<U * 1024>(x_rows.buffer, xoff[U], x_rows.at, to);
      buffer_lds_x4<(U + 1) * 1024>(x_rows.buffer, xoff[U + 1], x_rows.at, to);
      buffer_lds_x4<(U + 2) * 1024>(x_rows.buffer, xoff[U + 2], x_rows.at, to);
      buffer_lds_x4<(U + 3) * 1024>(x_rows.buffer, xoff[U + 3], x_rows.at, to);
    };
    auto fetch = [&]() {                            // everything of the wavefront's next group
      buffer_lds_x4<0>(w_rows.buffer, woff[0], w_rows.at, lds_own);
      buffer_lds_x4<1024>(w_rows.buffer, woff[1], w_rows.at, lds_own);
      if constexpr (CT == 2) {
        buffer_lds_x4<2048>(w_rows.buffer, woff[2], w_rows.at, lds_own);
        buffer_lds_x4<3072>(w_rows.buffer, woff[3], w_rows.at, lds_own);
      }
      buffer_lds_x1<W_BYTES>(s_rows.buffer, soff, s_rows.at, lds_own);
      buffer_lds_x1<W_BYTES + 256>(z_rows.buffer, zoff, z_rows.at, lds_own);
      fetch_x4(Int<0>{});
      if constexpr (XL >= 8) fetch_x4(Int<4>{});
      if constexpr (XL == 16) { fetch_x4(Int<8>{}); fetch_x4(Int<12>{}); }
      w_rows.next();
      s_rows.next();
      z_rows.next();
      x_rows.next();
    };
    // ---- operand roles as in art_gemm_w4.hip: a transposing read hands a lane 16 values of k of its column
    int b_off[CT];                                  // + 8 BN q
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) b_off[ct] = (h * 32 + (s16 >> 1)) * BN + ((2 * ct + hi16) ^ swizzle(s16 >> 1)) * 16 + (s16 & 1) * 8;
    const int a_row = (lane & 31) & (XR == 16 ? 15 : 31);            // (16 rows: the upper lanes repeat them, their sums are dropped)

    fetch();
    for (int left = mine; left > 0; --left) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      i32x2 pk[CT][4];
      _Float16 raw_s[CT];
      unsigned int raw_z[CT];
      h8 fa[MT][8];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
#pragma unroll
        for (int q = 0; q < 4; ++q) pk[ct][q] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*)(own + b_off[ct] + 8 * BN * q));
        const int pos = ct * 32 + hi16 * 16 + s16;
        raw_s[ct] = *reinterpret_cast<const _Float16*>(own + W_BYTES + pos * 2);
        raw_z[ct] = own[W_BYTES + 256 + (pos >> 1)];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int t = 0; t < MT; ++t) fa[t][e] = *reinterpret_cast<const h8*>(own_x + (t * 32 + a_row) * 256 + (((8 * h + e) ^ s16) * 16));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (left > 1) fetch();
      __builtin_amdgcn_sched_barrier(0);
      h2 s2[CT], zz2[CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const unsigned int z = (raw_z[ct] >> ((s16 & 1) * 4)) & 15u;
        s2[ct] = h2{raw_s[ct], raw_s[ct]};
        zz2[ct] = as_h2(z | (z << 20) | mg.bias);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          h2 p[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) p[j] = as_h2(and_or(nibble_pair((unsigned int)pk[ct][e >> 1][e & 1], j), mg.mask, mg.bias)) - zz2[ct];
#pragma unroll
          for (int j = 0; j < 4; ++j) p[j] = p[j] * s2[ct];
          const h8 b = h8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[t][ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[t][e], b, acc[t][ct], 0, 0, 0);
        }
    }
  }

  // ---- the eight wavefronts meet, in their order.  Sums lie as in the registers: element 4 q + i of row tile t in lane l is row
  // 32 t + 8 q + 4 (l / 32) + i; a thread adds V neighbours of them.
  constexpr int QUADS = 4 * MT * CT, V = QUADS / 2;
  typedef float fv __attribute__((ext_vector_type(V)));
  f32x4* const mine_at = reinterpret_cast<f32x4*>(own);
#pragma unroll
  for (int j = 0; j < QUADS; ++j) {
    const f16v& a = acc[(j >> 2) % MT][(j >> 2) / MT];
    mine_at[j * 64 + lane] = f32x4{a[4 * (j & 3)], a[4 * (j & 3) + 1], a[4 * (j & 3) + 2], a[4 * (j & 3) + 3]};
  }
  __syncthreads();
  const int quad = QUADS == 8 ? wave : wave >> 1, part = QUADS == 8 ? 0 : 2 * (wave & 1);      // of this thread; neighbouring threads have neighbouring columns
  fv sum;
  {
    fv of[kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) of[w] = *reinterpret_cast<const fv*>(smem + w * wave_bytes(XR, CT) + (quad * 64 + lane) * 16 + part * 4);
    sum = of[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) sum += of[w];
  }
  const int t = (quad >> 2) % MT, ct = (quad >> 2) / MT, piece = 2 * ct + hi16, row0 = m0 + t * 32 + (quad & 3) * 8 + h * 4 + part;
  if (!inside(piece)) return;                       // both of a pair or neither, but for kPlain
  const int col = piece_at(piece) + s16;
  if (splits > 1) {
    const PartialTile to(partial, split, M, N);
    const unsigned int at = to.at(row0, col);
#pragma unroll
    for (int i = 0; i < V; ++i) to.store(at, i, sum[i]);
    return;
  }
  if constexpr (TAIL == kPlain) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      if (row0 + i >= M) return;
      const size_t out = (size_t)(row0 + i) * N + col;
      _Float16 o = (_Float16)sum[i];
      if (residual) o = (_Float16)((float)o + (float)residual[out]);
      y[out] = o;
    }
  } else {
#pragma unroll
    for (int i = 0; i < V; i += 2) {                // lanes 0-15 and their partners 16-31: the former take row i, the latter row i + 1
      const float here = sum[i], next = sum[i + 1];
      const auto pair = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned int, here), __builtin_bit_cast(unsigned int, next), false, false);
      const float a = (float)(_Float16)__builtin_bit_cast(float, (unsigned int)pair[0]), b = (float)(_Float16)__builtin_bit_cast(float, (unsigned int)pair[1]);
      const int row = row0 + i + hi16;
      if (row >= M) continue;
      const int first_col = piece_at(piece & ~1) + s16;
      if constexpr (TAIL == kSwiglu) {
        y[(size_t)row * (N / 2) + first_col] = (_Float16)(art::silu(a) * b);
      } else {
        const int head = first_col >> 7, j = first_col & 127;
        _Float16* const to = rope.at(head) + (size_t)row * rope.heads * 128 + j;
        _Float16 first = (_Float16)a, second = (_Float16)b;
        if (rope.rotated(head)) {
          const float2 angle = rope.angles[(size_t)row * 64 + j];
          first = (_Float16)(a * angle.y - b * angle.x);
          second = (_Float16)(b * angle.y + a * angle.x);
        }
        to[0] = first;
        to[64] = second;
      }
    }
  }
}

}  // namespace

int art::w4::gemm_deep(const _Float16* x, const unsigned char* qweight, const _Float16* scales, const unsigned char* qzeros, _Float16* y,
                       float* partial, int M, int K, int N, int splits, int row_tiles, int col_tiles, const _Float16* residual, Tail tail, const Rope& rope, hipStream_t stream) {
#define ART_DEEP(XR, CT) {gemm_w4a16_deep_kernel<XR, CT, kPlain>, gemm_w4a16_deep_kernel<XR, CT, kSwiglu>, gemm_w4a16_deep_kernel<XR, CT, kRope>}
  static const decltype(&gemm_w4a16_deep_kernel<16, 1, kPlain>) kernels[5][3] = {ART_DEEP(16, 1), ART_DEEP(32, 1), ART_DEEP(64, 1), ART_DEEP(16, 2), ART_DEEP(32, 2)};
#undef ART_DEEP
  static const size_t lds[5] = {lds_bytes(16, 1), lds_bytes(32, 1), lds_bytes(64, 1), lds_bytes(16, 2), lds_bytes(32, 2)};
  static bool configured = false;
  if (!configured) {
    for (int i = 0; i < 5; ++i)
      for (int j = 0; j < 3; ++j)
        ART_HIP(hipFuncSetAttribute((const void*)kernels[i][j], hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds[i]));
    configured = true;
  }
  const int rows = M <= 16 ? 16 : 32 * row_tiles, m_blocks = (M + rows - 1) / rows, form = (rows == 16 ? 0 : rows == 32 ? 1 : 2) + (col_tiles == 2 ? 3 : 0);
  const int tiles = deep_tiles(N, tail, col_tiles), units = tiles * splits * m_blocks, each = (units + 7) / 8, G = K / GK;
  const bool by_tile = by_eighths(N, tail);
  const int across = by_tile ? splits : tiles;      // units next to each other: splits of a tile, or tiles of a split
  kernels[form][tail]<<<dim3(8 * each), kThreads, lds[form], stream>>>(
      x, qweight, scales, qzeros, K, N, M, by_tile ? across : -across, (unsigned int)((0x100000000ull + across - 1) / across), each, units, m_blocks,
      (unsigned int)((0x100000000ull + m_blocks - 1) / m_blocks), y, partial, splits, G / splits,
      G % splits, kMagic, residual, rope);
  ART_LAUNCH_CHECK();
  return 0;
}
