// Weight-only int4 GEMM for large batches (whole prompts): the arithmetic of art_gemm_w4.hip,
//     y[m,n] = sum_k x[m,k] * w[k,n],   w[k,n] = fp16(s[g,n] * fp16(q[k,n] - z[g,n])),   group g = k / 128,
// on the matrix cores with fp32 accumulation.  Blocks of 64 rows spend more time unpacking weights than multiplying
// them (166 vector instructions per 16 MFMAs and wavefront); here a block owns 128 or 256 rows, so that an unpacked
// weight is multiplied by four or eight row tiles.
//
//   * four wavefronts, each 32 MT rows x 64 columns (MT = 4: 128 accumulator registers and two blocks per compute
//     unit, MT = 8: 256 and one wavefront per SIMD).  No two wavefronts unpack the same weight.  What bounds the loop is
//     the issue of vector instructions beside the MFMAs: one wavefront alone gets four of them into the shadow of an
//     MFMA (32 cycles) and pays 7 cycles for every further one, two wavefronts get six each.  Hence pairs of k in
//     natural order (half a v_perm and half a shift more per pair of weights) instead of a permutation of every x
//     operand: the loop has 2.1 vector instructions per MFMA at MT = 8 and 4.3 at MT = 4;
//   * per 64 values of k a block needs 8 KiB of packed weights, 4 MT KiB of x and the group's scales and zero points;
//     they go from global memory straight into LDS (buffer loads, no registers in flight), a ring of three slots.
//     The weights run a stage ahead of x, so that the first operands of a stage can be unpacked in the stage before;
//   * the chunk positions are swizzled so that every 16 lanes of a 16-byte read of x (rows 128 bytes apart), and of a
//     transposing byte read of the weights, touch every bank once (SQ_LDS_BANK_CONFLICT 0.5 M cycles in a launch of 33 M
//     wavefront cycles, 1003 rows over 4096 x 12288);
//   * loads come from buffer descriptors, one scalar offset moves on from stage to stage; with four row tiles the ring slots are
//     constants (the loop is three groups long; with eight the compiler spills in such a loop).  A group is 647 instructions with eight
//     row tiles, 470 with four; with 64-bit addresses that stop at the last stage, and differences directly in front of their products (a
//     wait state each), it was 711 and 549, and a K-split's sums left by ten instructions a store instead of two: 200 rows over
//     11008 x 4096 38.7 -> 34.9 us, 1003 rows over 4096 x 12288 101.2 -> 99.1, 8192 x 2048 50.8 -> 47.7;
//   * one round = 16 values of k per lane half = 2 MT MFMAs.  The operands of round e + 1 are read and unpacked between
//     the MFMAs of round e, in four chunks fenced against the scheduler; each chunk also issues at most one load.  Left
//     together the loads of a stage blocked every wavefront of the compute unit at once, about 700 cycles per stage.
// Measured (MI355X, 1003 rows, weights from memory): 4096 x 12288 93 us = 1.08 PFLOP/s (matrix cores busy 0.77 of the time),
// 4096 x 22016 166 us; the 64-row blocks of art_gemm_w4.hip take 131 and 233 us, its 128-row blocks 112 and 211, and the
// kernel there was before this one (64 rows x 256 columns) took 157 and 246.  4096 columns are too few for blocks of 256:
// 4096 x 4096 takes 45 us here and 37.5 with 128 x 128 blocks, 11008 x 4096 97 and 92.
#include "art_w4_mfma.h"

#include <type_traits>

namespace {

using namespace art::w4;

template <int V> using Int = std::integral_constant<int, V>;

constexpr int kThreads = 256;
constexpr int BN = 256, SK = 64;                    // columns of a block, k of a stage
constexpr int NS = 3;                               // stages of the LDS ring
constexpr int W_BYTES = (SK / 2) * BN;              // 32 byte-rows x 256 columns
constexpr int Q_BYTES = 1024;                       // scales (512 B), zero points (128 B), idle lanes
constexpr int C_LD = BN + 8;                        // halves per row of the staged output
constexpr int stage_bytes(int MT) { return W_BYTES + Q_BYTES + MT * 32 * SK * 2; }
constexpr size_t lds_bytes(int MT) { return (size_t)NS * stage_bytes(MT); }
static_assert(128 * C_LD * 2 <= NS * stage_bytes(4), "128 staged output rows fit the ring");

// kSwiglu: the matrix is gate | up (N / 2 columns each); a block owns 128 gate columns and the matching 128 up columns and
// stores y[m, n] = fp16(silu(fp16(gate)) * fp16(up)), N / 2 columns.
template <int MT, Tail TAIL, bool FAR>
__global__ __launch_bounds__(kThreads, MT == 8 ? 1 : 2) void gemm_w4a16_wide_kernel(
    const _Float16* __restrict__ x, const unsigned char* __restrict__ qweight, const _Float16* __restrict__ scales,
    const unsigned char* __restrict__ qzeros, _Float16* y, float* __restrict__ partial, int M, int K, int N, int splits,
    Deal deal, Div by_splits, int groups, int longer, Magic mg, const _Float16* residual, Rope rope) {       // residual may be y itself
  constexpr bool SWIGLU = TAIL == kSwiglu;
  constexpr int STAGE = stage_bytes(MT), BM = 32 * MT;
  constexpr int L = 2 + MT + 1;                     // loads per wavefront and stage
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int unit, m_block;                                // (column tile, K split) pair, block of rows
  if (!deal.take(unit, m_block)) return;
  const int tile = (int)over((unsigned)unit, by_splits), split = unit - tile * splits;
  const TileColumns<TAIL, BN> cols{tile * (SWIGLU ? BN / 2 : BN), N};
  const int m0 = m_block * BM;
  const int g_begin = split * groups + (split < longer ? split : longer), g_count = groups + (split < longer ? 1 : 0);
  const int steps = 2 * g_count;          // splits <= G: at least two
  const unsigned int lds0 = (unsigned int)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;

  // ---- what this lane fetches per stage.  Columns past N and rows past M re-read valid memory; nothing of them is stored.
  unsigned int woff[2], xoff[MT], qoff;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = 4 * (wave + 4 * u) + (lane >> 4);
    woff[u] = (unsigned int)r * N + cols.safe(((lane & 15) ^ (r & 7)) * 16);
  }
#pragma unroll
  for (int u = 0; u < MT; ++u) {
    const int r = 8 * (wave + 4 * u) + (lane >> 3), row = m0 + r < M ? m0 + r : M - 1;
    xoff[u] = (unsigned int)(row - m0) * (2 * K) + (((lane & 7) ^ ((r >> 1) & 7)) * 16);
  }
  // scales and zero points share one load: wavefronts 0 and 1 fetch the scales of columns 2 d, 2 d + 1, half of
  // wavefront 2 the zero points of columns 8 (d - 128) .. + 7, the others repeat the first scales
  const bool is_zero = tid >= 128 && tid < 160;
  qoff = is_zero ? (unsigned int)cols.safe(8 * (tid - 128)) >> 1 : (tid < 128 ? 2u * cols.safe(2 * tid) : 0u);
  const unsigned int qstep = wave == 2 ? N / 2 : 2 * N;
  Rows<FAR> w_rows(qweight + (size_t)g_begin * 64 * N, 32u * N, steps), x_rows(x + (size_t)m0 * K + (size_t)g_begin * 128, SK * 2, steps),
      q_rows(wave == 2 ? (const void*)(qzeros + (size_t)g_begin * qstep) : (const void*)(scales + (size_t)g_begin * N), qstep, g_count);
  const unsigned int lds_w = lds0 + wave * 1024, lds_q = lds0 + wave * 256;

  // Load j of ring slot `slot` (its offset): 0, 1 packed weights, 2 scales and zero points, 3 .. MT + 2 x.  The weights run one
  // stage ahead of x: slot of stage i holds x of stage i and the weights of stage i + 1.
  auto issue = [&](unsigned int slot, auto j_tag) {
    constexpr int J = decltype(j_tag)::value;
    if constexpr (J < 2) buffer_lds_x4<4 * J * 1024>(w_rows.buffer, woff[J], w_rows.at, lds_w + slot);
    else if constexpr (J == 2) buffer_lds_x1<W_BYTES>(q_rows.buffer, qoff, q_rows.at, lds_q + slot);
    else buffer_lds_x4<W_BYTES + Q_BYTES + 4 * (J - 3) * 1024>(x_rows.buffer, xoff[J - 3], x_rows.at, lds_w + slot);
  };
  auto issue_weights = [&](unsigned int slot) { issue(slot, Int<0>{}); issue(slot, Int<1>{}); issue(slot, Int<2>{}); };
  auto issue_x = [&](unsigned int slot) {
    issue(slot, Int<3>{}); issue(slot, Int<4>{}); issue(slot, Int<5>{}); issue(slot, Int<6>{});
    if constexpr (MT == 8) { issue(slot, Int<7>{}); issue(slot, Int<8>{}); issue(slot, Int<9>{}); issue(slot, Int<10>{}); }
  };
  auto next_weights = [&](auto odd_tag) {           // of the stage whose weights were just fetched; a group is two stages
    w_rows.next();
    if constexpr (decltype(odd_tag)::value == 1) q_rows.next();
    if (w_rows.far()) { w_rows.rebase(); q_rows.rebase(); }
  };

  // ---- operand roles.  A transposing read takes 8 byte-rows x 16 columns per 16 lanes: lane s16 supplies the 8-byte
  // piece (row s16 / 2, half s16 % 2) and receives the 8 bytes (16 values of k) of column s16.  Lanes 16-31 take the
  // chunk 8 further on, so that the 32 lanes of a pass touch 16 different chunk positions.
  const int s16 = lane & 15, hi16 = (lane >> 4) & 1, h = lane >> 5;
  int b_off[2], colpos[2];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int chunk = wave * 2 + ct + 8 * hi16;
    b_off[ct] = (h * 16 + (s16 >> 1)) * 256 + ((chunk ^ (s16 >> 1)) * 16) + (s16 & 1) * 8;      // + q * 2048
    colpos[ct] = chunk * 16 + s16;
  }
  int a_off[4];                                     // x chunk 4 h + e of row lane % 32; + 4096 per row tile
#pragma unroll
  for (int e = 0; e < 4; ++e) a_off[e] = W_BYTES + Q_BYTES + (lane & 31) * 128 + (((4 * h + e) ^ ((lane >> 1) & 7)) * 16);

  f16v acc[MT][2];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][c][r] = 0.f;

  i32x2 pk[2][2][2];                                // packed weights: [stage parity][q][column tile]
  _Float16 raw_s[2];
  unsigned int raw_z[2];
  h2 s2[2], zz2[2];                                 // scale, 1024 and 64 + zero point of this lane's two columns
  h8 fa[2][MT];                                     // operands of a round, double buffered: x
  h2 fb[2][2][4];                                   // ... weights, in pairs of k
  auto read_weights = [&](unsigned int slot, int par, int part) {
    const unsigned char* st = smem + slot;
    if (part < 4) pk[par][part >> 1][part & 1] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*)(st + b_off[part & 1] + (part >> 1) * 2048));
  };
  auto read_scales = [&](unsigned int slot, int ct) {
    const unsigned char* st = smem + slot + W_BYTES;
    raw_s[ct] = *reinterpret_cast<const _Float16*>(st + colpos[ct] * 2);
    raw_z[ct] = st[512 + (colpos[ct] >> 1)];
  };
  auto decode_scales = [&](int ct) {
    const unsigned int z = (raw_z[ct] >> ((colpos[ct] & 1) * 4)) & 15u;
    const _Float16 s = cols.inside(colpos[ct]) ? raw_s[ct] : (_Float16)0.f;
    s2[ct] = h2{s, s};
    zz2[ct] = as_h2(z | (z << 20) | mg.bias);
  };
  auto read_x = [&](unsigned int slot, int e, int t) {
    fa[e & 1][t] = *reinterpret_cast<const h8*>(smem + slot + a_off[e] + t * 4096);
  };
  // pairs j and j + 1 (j even) of column tile ct for round e.  Byte j of the word holds k = 2 j (low nibble) and 2 j + 1 (high
  // nibble).  Step by step for both: a difference directly in front of its product costs a wait state.
  auto unpack_two = [&](int par, int e, int ct, int j) {
    const unsigned int w = (unsigned int)pk[par][e >> 1][ct][e & 1];
    const h2 a = as_h2(and_or(nibble_pair(w, j), mg.mask, mg.bias)), b = as_h2(and_or(nibble_pair(w, j + 1), mg.mask, mg.bias));
    const h2 da = a - zz2[ct], db = b - zz2[ct];
    fb[e & 1][ct][j] = da * s2[ct];
    fb[e & 1][ct][j + 1] = db * s2[ct];
  };
  auto multiply = [&](int slot, int t) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      const h2* p = fb[slot][ct];
      const h8 b = h8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
      acc[t][ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[slot][t], b, acc[t][ct], 0, 0, 0);
    }
  };

  // ---- prologue: weights of stage 0 into slot 2, then slots 0 and 1
  issue_weights(2 * STAGE);
  next_weights(Int<0>{});
  issue_weights(0);
  issue_x(0);
  next_weights(Int<1>{});
  x_rows.next();
  issue_weights(STAGE);
  issue_x(STAGE);
  next_weights(Int<0>{});
  x_rows.next();
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");       // loads return in order
  art_lds_barrier();
#pragma unroll
  for (int part = 0; part < 4; ++part) read_weights(2 * STAGE, 0, part);
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) { read_scales(2 * STAGE, ct); decode_scales(ct); }
#pragma unroll
  for (int t = 0; t < MT; ++t) read_x(0, 0, t);
#pragma unroll
  for (int ct = 0; ct < 2; ++ct)
#pragma unroll
    for (int j = 0; j < 4; j += 2) unpack_two(0, 0, ct, j);
  art_lds_barrier();                                // slot 2 is free again

  // A round multiplies 16 values of k per lane half and prepares the operands of the round behind it, in four chunks:
  // MT / 2 MFMAs, MT / 4 reads of x, two unpacked pairs and one load for the stage two ahead.  PAR: which half of its group the
  // stage is.
  constexpr int CT_ = MT / 4;                       // row tiles per chunk
  auto chunk_of = [&](unsigned int s_cur, unsigned int s_next, unsigned int s_fill, auto par_tag, auto e_tag, auto c_tag) {
    constexpr int PAR = decltype(par_tag)::value, E = decltype(e_tag)::value, c = decltype(c_tag)::value;
    __builtin_amdgcn_sched_barrier(0);
    constexpr int kFirst[4] = {3, 7, 11, 0};        // loads of rounds 0, 1, 2; round 3 starts the next stage's
    constexpr int j = kFirst[E] + c;
    if constexpr (E == 3 ? c < 3 : j < L) issue(E == 3 ? s_cur : s_fill, Int<j>{});
    if (E == 2) read_weights(s_cur, PAR ^ 1, c);    // the weights of stage i + 1 came with x of stage i
    if (E == 2 && PAR == 1 && c < 2) read_scales(s_cur, c);
    if (E == 3 && PAR == 1 && c == 0) { decode_scales(0); decode_scales(1); }
#pragma unroll
    for (int t = c * CT_; t < (c + 1) * CT_; ++t) E == 3 ? read_x(s_next, 0, t) : read_x(s_cur, (E + 1) & 3, t);
    unpack_two(E == 3 ? PAR ^ 1 : PAR, (E + 1) & 3, c >> 1, 2 * (c & 1));
#pragma unroll
    for (int t = c * CT_; t < (c + 1) * CT_; ++t) multiply(E & 1, t);
#pragma unroll
    for (int m = 0; m < 2 * CT_; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, MT == 8 ? 3 : 5, 0);
    }
  };
  auto round = [&](unsigned int s_cur, unsigned int s_next, unsigned int s_fill, auto par_tag, auto e_tag) {
    chunk_of(s_cur, s_next, s_fill, par_tag, e_tag, Int<0>{});
    chunk_of(s_cur, s_next, s_fill, par_tag, e_tag, Int<1>{});
    chunk_of(s_cur, s_next, s_fill, par_tag, e_tag, Int<2>{});
    chunk_of(s_cur, s_next, s_fill, par_tag, e_tag, Int<3>{});
    __builtin_amdgcn_sched_barrier(0);
  };
  auto stage = [&](unsigned int s_cur, unsigned int s_next, unsigned int s_fill, auto par_tag) {
    round(s_cur, s_next, s_fill, par_tag, Int<0>{});
    round(s_cur, s_next, s_fill, par_tag, Int<1>{});
    round(s_cur, s_next, s_fill, par_tag, Int<2>{});
    x_rows.next();
    // The next slot is complete once only the x loads of stage i + 2 are outstanding ... and everybody has read all of
    // this one, which then takes stage i + 3.  Behind the last stage the reads return old bytes; nothing uses them.
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");
    art_lds_barrier();
    round(s_cur, s_next, s_fill, par_tag, Int<3>{});
    next_weights(par_tag);                          // of stage i + 4, the same half of its group
  };
  // the weights of slot 2 (stage 3) open the pattern: from here on every round 3 fetches the weights of the next slot
  issue_weights(2 * STAGE);
  next_weights(Int<1>{});
  if constexpr (MT == 8) {                          // (with constants as below the compiler spills in the loop)
    unsigned int s_cur = 0, s_next = STAGE, s_fill = 2 * STAGE;
#pragma unroll 1
    for (int left = g_count; left > 0; --left) {
      stage(s_cur, s_next, s_fill, Int<0>{});
      stage(s_next, s_fill, s_cur, Int<1>{});
      const unsigned int first = s_cur;
      s_cur = s_fill;
      s_fill = s_next;
      s_next = first;
    }
  } else {
    for (int left = g_count;;) {                    // the slots are constants
      stage(0, STAGE, 2 * STAGE, Int<0>{});
      stage(STAGE, 2 * STAGE, 0, Int<1>{});
      if (--left == 0) break;
      stage(2 * STAGE, 0, STAGE, Int<0>{});
      stage(0, STAGE, 2 * STAGE, Int<1>{});
      if (--left == 0) break;
      stage(STAGE, 2 * STAGE, 0, Int<0>{});
      stage(2 * STAGE, 0, STAGE, Int<1>{});
      if (--left == 0) break;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing of the ring is on its way when its space is reused or given back

  // Accumulator element r of row tile t is row t * 32 + (r / 4) * 8 + 4 h + r % 4.
  if (splits > 1) {
    const PartialTile to(partial, split, M, N);
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      if (!cols.inside(colpos[ct])) continue;
      const unsigned int at = to.at(m0 + 4 * h, cols.at(colpos[ct]));
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) to.store(at, t * 32 + (r >> 2) * 8 + (r & 3), acc[t][ct][r]);
    }
    return;
  }
  _Float16* cs = reinterpret_cast<_Float16*>(smem);
  // kRope: a block is two heads, whose angles are the same; a thread has columns 8 (tid % 8) .. + 7 and their partners of both in every
  // 32nd row.  The angles of its next row are on their way while it rotates one.
  const int head = cols.n0 >> 7;
  const bool rotated[2] = {TAIL == kRope && rope.rotated(head), TAIL == kRope && rope.rotated(head + 1)};
  _Float16* const to[2] = {TAIL == kRope ? rope.at(head) : nullptr, TAIL == kRope ? rope.at(head + 1) : nullptr};
  Angles<8> angles;
  auto fetch_angles = [&](int row) { angles = load_angles<8>(rope.angles + (size_t)(row < M ? row : M - 1) * 64 + (tid & 7) * 8); };
  if (rotated[0]) fetch_angles(m0 + (tid >> 3));
#pragma unroll
  for (int p = 0; p < MT / 4; ++p) {                // 128 rows at a time through LDS, out as 16-byte stores
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          cs[(t * 32 + (r >> 2) * 8 + h * 4 + (r & 3)) * C_LD + colpos[ct]] = (_Float16)acc[4 * p + t][ct][r];
    __syncthreads();
    if constexpr (TAIL == kRope) {
#pragma unroll 1
      for (int row = tid >> 3; row < 128; row += kThreads / 8) {
        const int grow = m0 + p * 128 + row, col = (tid & 7) * 8;
        const Angles<8> now = angles;
        if (rotated[0]) fetch_angles(grow + kThreads / 8);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          h8 a = *reinterpret_cast<const h8*>(cs + row * C_LD + k * 128 + col), b = *reinterpret_cast<const h8*>(cs + row * C_LD + k * 128 + col + 64);
          if (rotated[k]) rotate(a, b, now);
          _Float16* const out = to[k] + (size_t)grow * (rope.heads * 128) + col;
          if (grow < M && (k == 0 || cols.inside(128))) {
            *reinterpret_cast<h8*>(out) = a;
            *reinterpret_cast<h8*>(out + 64) = b;
          }
        }
      }
      continue;
    }
    if constexpr (SWIGLU) {
#pragma unroll 1
      for (int c = tid; c < 128 * (BN / 16); c += kThreads) {
        const int row = c >> 4, col = (c & 15) * 8, grow = m0 + p * 128 + row;
        if (grow >= M || !cols.inside(col)) continue;
        const h8 g = *reinterpret_cast<const h8*>(cs + row * C_LD + col), u = *reinterpret_cast<const h8*>(cs + row * C_LD + 128 + col);
        const h4 lo = swiglu4(h4{g[0], g[1], g[2], g[3]}, h4{u[0], u[1], u[2], u[3]}), hi = swiglu4(h4{g[4], g[5], g[6], g[7]}, h4{u[4], u[5], u[6], u[7]});
        *reinterpret_cast<h8_by_8*>(y + (size_t)grow * (N / 2) + cols.at(col)) = h8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
      continue;
    }
#pragma unroll 4
    for (int c = tid; c < 128 * (BN / 8); c += kThreads) {
      const int row = c >> 5, col = (c & 31) * 8, grow = m0 + p * 128 + row;
      if (grow >= M || !cols.inside(col)) continue;
      const size_t at = (size_t)grow * N + cols.at(col);
      h8 o = *reinterpret_cast<const h8*>(cs + row * C_LD + col);
      if (residual) {                               // y = fp16(fp16(product) + residual)
        const h8 res = *reinterpret_cast<const h8_by_8*>(residual + at);
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = (_Float16)((float)o[k] + (float)res[k]);
      }
      *reinterpret_cast<h8_by_8*>(y + at) = o;
    }
  }
}

template <int MT, Tail TAIL, bool FAR = false>
int launch(const _Float16* x, const unsigned char* qweight, const _Float16* scales, const unsigned char* qzeros, _Float16* y,
           float* partial, int M, int K, int N, int splits, const _Float16* residual, const Rope& rope, hipStream_t stream) {
  static bool configured = false;
  if (!configured) {
    ART_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_w4a16_wide_kernel<MT, TAIL, FAR>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds_bytes(MT)));
    configured = true;
  }
  const int col_tiles = tile_count(N, TAIL == kSwiglu, BN), m_blocks = (M + 32 * MT - 1) / (32 * MT);
  dim3 grid;
  const Deal dealt = deal(col_tiles * splits, m_blocks, grid);
  gemm_w4a16_wide_kernel<MT, TAIL, FAR><<<grid, kThreads, lds_bytes(MT), stream>>>(
      x, qweight, scales, qzeros, y, partial, M, K, N, splits, dealt, make_div((unsigned)splits), K / 128 / splits, K / 128 % splits,
      kMagic, residual, rope);
  ART_LAUNCH_CHECK();
  return 0;
}

}  // namespace

int art::w4::gemm_wide(const _Float16* x, const unsigned char* qweight, const _Float16* scales, const unsigned char* qzeros, _Float16* y,
                       float* partial, int M, int K, int N, int splits, int row_tiles, bool far, const _Float16* residual, Tail tail, const Rope& rope,
                       hipStream_t stream) {
  static const decltype(&launch<4, kPlain>) by_rows[3][3] = {{launch<4, kPlain>, launch<4, kSwiglu>, launch<4, kRope>},
                                                             {launch<8, kPlain>, launch<8, kSwiglu>, launch<8, kRope>},
                                                             {launch<4, kPlain, true>, launch<4, kSwiglu, true>, launch<4, kRope, true>}};
  return by_rows[far ? 2 : row_tiles == 8][tail](x, qweight, scales, qzeros, y, partial, M, K, N, splits, residual, rope, stream);
}
