// Weight-only int4 GEMM for a batch of rows (four rows and more): the same arithmetic as the GEMV of art_gemv_w4.hip,
//     y[m,n] = sum_k x[m,k] * w[k,n],   w[k,n] = fp16(s[g,n] * fp16(q[k,n] - z[g,n])),   group g = k / 128,
// on the matrix cores with fp32 accumulation; w is rounded exactly as the reference's dequant + matmul program
// does (samples/05_llama2_7b_int4.py:135-144 exported with a batch axis).  This file holds the entry points, the kernel
// for batches that do not fill blocks of 256 columns x 128 or 256 rows (art_gemm_w4_wide.hip takes those), the pass that
// adds K-splits, and the rule that chooses among it, art_gemm_w4_wide.hip and art_gemm_w4_deep.hip.
//
// Design for MI355X:
//   * a block of eight wavefronts owns 128 columns, 32 MT rows (MT = 1, 2, 4) and a contiguous range of quantisation
//     groups.  Wavefront (c, h) multiplies 32 columns by the k half h of every group, so every weight is unpacked once per
//     block; the two k halves meet in LDS after the loop.  What bounds the loop is the issue of instructions, not the
//     matrix cores (with the MFMAs taken out a group takes as long): a wavefront by itself issues a vector instruction every 8
//     cycles, two of a SIMD one every 4 (the differences and products of halves and byte permutations; shifts and
//     v_bitop3 2), and a group is some 95 / 120 / 157 instructions at MT = 1 / 2 / 4, 56 of them vector instructions that
//     unpack.  Hence ring slots that are constants (the loop is three groups long) and loads from buffer descriptors, where one
//     scalar offset moves on.  With slots and addresses in registers a group was 138 / 149 / 193 instructions, and each store of a
//     K-split's sums ten (a comparison, a branch, 64-bit addresses) instead of two: 16 rows over 1024 x 3072 6.6 -> 6.2 us, over
//     11008 x 4096 12.6 -> 12.0; 50 rows over 4096 x 12288 19.9 -> 18.3; 128 rows over 4096 x 4096 16.0 -> 14.9, 4096 x 22016 32.9 -> 31.4.
//     Sixteen wavefronts with half the work each were slower (the LDS meeting doubles), and so were four column quarters
//     replaced by two (same loop, longer meeting), blocks that start at groups of their own, and branches around the
//     loads of the last groups;
//   * everything a group needs - 8 KiB of packed weights, 8 MT KiB of x, 256 B of scales, 64 B of zero points - goes from
//     global memory straight into LDS (buffer loads: no registers hold data in flight), into a ring of three slots.
//     The weights run a group ahead of x, so that the first operands of a group are unpacked in the one before;
//   * LDS position (row r, chunk p) holds chunk p ^ ((r / 2) & 7) of the weights (rows of 128 bytes) and p ^ (r & 15) of x
//     (rows of 256 bytes): every 16 lanes of a read touch every bank once;
//   * the packed bytes stay packed in LDS.  ds_read_b64_tr_b8 hands a lane four bytes = 8 values of k of ONE column, each byte twice (the
//     B operand of a v_mfma_f32_32x32x16_f16): a byte's nibbles are where the two halves of a pair want them without a permutation.  Against
//     every byte once, eight of them a read, and permutations (64 instructions that unpack), HBM / cache, us: 16 rows of gate | up
//     4096 x 22016 19.1 / 18.3 -> 18.5 / 16.8, 50 rows 22.7 / 20.7 -> 22.5 / 19.4, 128 rows over 4096 x 12288 21.5 / 19.4 -> 20.7 / 19.5, over 11008 x 4096 in
//     four splits 23.3 / 21.7 -> 22.0 / 21.0; 17 products 1.022 / 1.029 times as fast;
//   * split-K without atomics (5.6 M float atomics cost 75 us on this chip): each K-split writes its fp32 tile to the
//     library workspace and a second small kernel adds the splits in a fixed order and rounds once to fp16 - results
//     do not depend on timing.
// Before (blocks of 256 columns, a k half of 64 columns per wavefront, x operands permuted instead of weights) and now, on one
// card, weights from memory: 64 rows over 4096 x 4096 / 4096 x 22016 / 11008 x 4096 13.6 / 28.6 / 18.2 us -> 11.2 / 22.4 / 16.9;
// 50 rows over 11008 x 4096 17.9 -> 16.2; 128 rows over 4096 x 12288 / 22016 28.1 / 40.0 -> 22.3 / 31.2; 16 rows over
// 1024 x 3072 7.4 -> 6.8.
// The end of a block: the k halves exchange halves of their sums as they lie in the registers, the K-splits' sums leave from
// there, SWIGLU pairs gate and up by lane exchange.  Against sums that meet as [row][column] by one half of the wavefronts and are
// read back by fours, half of the lanes without work in SWIGLU, on one card: 128 rows over 4096 x 22016 34.9 -> 32.5 us, SWIGLU
// 39.0 -> 35.3, 50 rows with SWIGLU 26.6 -> 25.2, six splits of 128 rows over 11008 x 4096 26.1 -> 25.5.
// q | k | v (kRope): a block is a head, its rows are rotated on the way out, with angles that are fetched before the loop.  Against the
// rotation in a launch of its own behind the product (4096 x 12288, both launches, one card): 16 rows 16.1 -> 15.0 us, 50 rows
// 21.2 -> 18.9, 128 rows 26.1 -> 22.4; blocks of 256 columns: 300 rows 47.4 -> 44.1, 1003 rows 104.7 -> 99.3 (the product alone
// 96.0).  A rotation of the sums in registers, its code unrolled, lost more in the wide blocks than the launch costs.
#include "art_w4_mfma.h"

#include <type_traits>

namespace {

using namespace art::w4;

template <int V> using Int = std::integral_constant<int, V>;

constexpr int kThreads = 512;                       // 8 wavefronts: 4 column quarters x 2 k halves
constexpr int BN = 128, GK = 128;                   // columns of a block, k of a quantisation group
constexpr int W_BYTES = (GK / 2) * BN;              // packed weights of a group: 64 byte-rows x 128 columns
constexpr int Q_BYTES = 2048;                       // scales (256 B) at 0, zero points (64 B) at 256; the rest takes the idle lanes
constexpr int stage_bytes(int MT) { return W_BYTES + Q_BYTES + MT * 32 * GK * 2; }
constexpr size_t lds_bytes(int MT) { return 3 * (size_t)stage_bytes(MT); }     // 55, 80 (two blocks per compute unit), 129 KB
static_assert(16 * 1024 + 32 * (BN + 8) * 2 <= 3 * stage_bytes(1) && 32 * 1024 + 64 * (BN + 8) * 2 <= 3 * stage_bytes(2) &&
                  64 * 1024 + 128 * (BN + 8) * 2 <= 3 * stage_bytes(4), "the sums that are handed over and the results fit the ring");

// How the (column tile, K split) pairs are laid out; worked out on the host, so that a block starts without divisions.
struct Work {
  Deal deal;
  int splits;
  unsigned int inv_splits;                          // ceil(2^32 / splits), 0 for one split: unit / splits = mulhi(unit, inv_splits) for units below 2^16
  int groups, longer;                               // groups of a K split; the first `longer` have one more
};

template <int MT, Tail TAIL, bool FAR = false>
__global__ __launch_bounds__(kThreads, MT == 4 ? 2 : 4) void gemm_w4a16_kernel(
    const _Float16* __restrict__ x, const unsigned char* __restrict__ qweight, const _Float16* __restrict__ scales,
    const unsigned char* __restrict__ qzeros, _Float16* y, float* __restrict__ partial, int M, int K, int N, Work work, Magic mg,
    const _Float16* residual, Rope rope) {          // residual may be y itself
  constexpr bool SWIGLU = TAIL == kSwiglu, ROPE = TAIL == kRope;
  constexpr int STAGE = stage_bytes(MT), BM = 32 * MT;
  constexpr int L = 2 + MT;                         // LDS-direct loads per wavefront and group: weights, scales, MT x
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = wave & 3, kh = wave >> 2;          // 32-column quarter of the tile, k half of every group

  int unit, m_block;                                // (tile, split) pair, block of rows
  if (!work.deal.take(unit, m_block)) return;
  const int m0 = m_block * BM;
  const int tile = work.inv_splits ? (int)__umulhi(unit, work.inv_splits) : unit, split = unit - tile * work.splits;
  const TileColumns<TAIL, BN> cols{tile * (SWIGLU ? BN / 2 : BN), N};
  const int g_begin = split * work.groups + (split < work.longer ? split : work.longer), groups = work.groups + (split < work.longer ? 1 : 0);
  const unsigned int lds0 = (unsigned int)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;

  // ---- what this lane fetches per group.  Columns past N and rows past M re-read valid memory; nothing of them is stored.
  unsigned int woff, xoff[MT], qoff = 0;
  {
    const int r = 8 * wave + (lane >> 3);
    woff = (unsigned int)r * N + cols.safe(((lane & 7) ^ ((r >> 1) & 7)) * 16);
  }
#pragma unroll
  for (int u = 0; u < MT; ++u) {
    const int r = 4 * (wave + 8 * u) + (lane >> 4), row = m0 + r < M ? r : M - 1 - m0;
    xoff[u] = (unsigned int)row * (2 * K) + (((lane & 15) ^ (r & 15)) * 16);
  }
  if (wave == 0) qoff = 2u * cols.safe(2 * lane);                        // scales of columns 2 lane, 2 lane + 1
  if (wave == 1 && lane < 16) qoff = (unsigned int)cols.safe(8 * lane) >> 1;      // zero points of 8 columns; idle lanes re-read the first
  const unsigned int qstep = wave == 1 ? N / 2 : 2 * N;
  Rows<FAR> w_rows(qweight + (size_t)g_begin * (GK / 2) * N, (GK / 2) * N, groups), x_rows(x + (size_t)m0 * K + (size_t)g_begin * GK, GK * 2, groups),
      q_rows(wave == 1 ? (const void*)(qzeros + (size_t)g_begin * qstep) : (const void*)(scales + (size_t)g_begin * N), qstep, groups);
  const unsigned int lds_w = lds0 + wave * 1024, lds_q = lds0 + wave * 256;
  // Load j for ring slot S: 0 packed weights, 1 scales and zero points, 2 .. MT + 1 x.  The slot of group i holds x of
  // group i and the weights of group i + 1.
  auto issue = [&](auto s_tag, auto j_tag) {
    constexpr unsigned int ST = decltype(s_tag)::value * STAGE;
    constexpr int J = decltype(j_tag)::value;
    if constexpr (J == 0) buffer_lds_x4<ST>(w_rows.buffer, woff, w_rows.at, lds_w);
    else if constexpr (J == 1) buffer_lds_x1<ST + W_BYTES>(q_rows.buffer, qoff, q_rows.at, lds_q);
    else buffer_lds_x4<ST + W_BYTES + Q_BYTES + 8 * (J - 2) * 1024>(x_rows.buffer, xoff[J - 2], x_rows.at, lds_w);
  };
  auto issue_x = [&](auto s_tag) {
    issue(s_tag, Int<2>{});
    if constexpr (MT >= 2) issue(s_tag, Int<3>{});
    if constexpr (MT >= 4) { issue(s_tag, Int<4>{}); issue(s_tag, Int<5>{}); }
  };
  auto next_weights = [&]() {
    w_rows.next();
    q_rows.next();
    if (w_rows.far()) { w_rows.rebase(); q_rows.rebase(); }
  };

  // ROPE: the block is one head.  The angles that this thread needs at the end are fetched first.
  const int head = cols.n0 / BN;
  const bool rotated = ROPE && work.splits == 1 && rope.rotated(head);
  constexpr int PIECES = ROPE ? (BM * 8 + kThreads - 1) / kThreads : 1;
  Angles<8> angles[PIECES];
  if (rotated)
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int row = m0 + ((tid + i * kThreads) >> 3);
      angles[i] = load_angles<8>(rope.angles + (size_t)(row < M ? row : M - 1) * 64 + (tid & 7) * 8);
    }

  // ---- operand roles.  A transposing read takes 8 byte-rows x 16 columns per 16 lanes: lane s16 supplies the
  // 8-byte piece (row s16 / 2, half s16 % 2) and receives the 8 bytes of column s16.  Lanes 16-31 take the chunk four
  // further on, whose swizzled positions are the other four (and, with SWIGLU, the up columns of the lanes' gates).
  const int s16 = lane & 15, hi16 = (lane >> 4) & 1, h = lane >> 5;
  const int chunk = cw + 4 * hi16, colpos = chunk * 16 + s16;              // the column (within the tile) this lane accumulates
  int b_off[4], a_off[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = kh * 32 + h * 16 + 4 * e + twice_row(s16 >> 1);
    b_off[e] = r * 128 + ((chunk ^ ((r >> 1) & 7)) * 16) + (s16 & 1) * 8;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) a_off[e] = W_BYTES + Q_BYTES + (lane & 31) * 256 + (((kh * 8 + h * 4 + e) ^ s16) * 16);     // + 8192 per row tile

  f16v acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

  i32x2 pk[4], pk_next[4];                          // packed weights of the group and of the next one: [round]
  _Float16 raw_s;
  unsigned int raw_z;
  h2 s2, zz2;                                       // scale, 1024 and 64 + zero point of this lane's column
  h8 fa[2][MT];                                     // operands of a round, double buffered: x
  h2 fb[2][4];                                      // ... weights, in pairs of k
  auto read_weights = [&](unsigned int slot, i32x2 (&to)[4], int e) {
    to[e] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*)(smem + slot + b_off[e]));
  };
  auto read_scales = [&](unsigned int slot) {
    const unsigned char* st = smem + slot + W_BYTES;
    raw_s = *reinterpret_cast<const _Float16*>(st + colpos * 2);
    raw_z = st[256 + (colpos >> 1)];
  };
  auto decode_scales = [&]() {
    const unsigned int z = (raw_z >> ((colpos & 1) * 4)) & 15u;
    const _Float16 s = cols.inside(colpos) ? raw_s : (_Float16)0.f;
    s2 = h2{s, s};
    zz2 = as_h2(z | (z << 20) | mg.bias);
  };
  auto read_x = [&](unsigned int slot, int e, int t) {
    fa[e & 1][t] = *reinterpret_cast<const h8*>(smem + slot + a_off[e] + t * 8192);
  };
  auto unpack = [&](const i32x2 (&from)[4], int e, int j) {       // k = 2 j, 2 j + 1 of round e
    fb[e & 1][j] = (as_h2(and_or(nibbles_of_twice((unsigned int)from[e][j >> 1], j), mg.mask, mg.bias)) - zz2) * s2;
  };
  auto multiply = [&](int slot, int t) {
    const h2* p = fb[slot];
    const h8 b = h8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[slot][t], b, acc[t], 0, 0, 0);
  };

  // ---- prologue: weights of group 0 into slot 2, then slots 0 and 1
  issue(Int<2>{}, Int<0>{});
  issue(Int<2>{}, Int<1>{});
  next_weights();
  issue(Int<0>{}, Int<0>{});
  issue(Int<0>{}, Int<1>{});
  issue_x(Int<0>{});
  next_weights();
  x_rows.next();
  issue(Int<1>{}, Int<0>{});
  issue(Int<1>{}, Int<1>{});
  issue_x(Int<1>{});
  next_weights();
  x_rows.next();
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");       // loads return in order
  art_lds_barrier();
#pragma unroll
  for (int e = 0; e < 4; ++e) read_weights(2 * STAGE, pk, e);
  read_scales(2 * STAGE);
  decode_scales();
#pragma unroll
  for (int t = 0; t < MT; ++t) read_x(0, 0, t);
#pragma unroll
  for (int j = 0; j < 4; ++j) unpack(pk, 0, j);
  art_lds_barrier();                                // slot 2 is free again: it takes the weights of group 3 first
  issue(Int<2>{}, Int<0>{});
  issue(Int<2>{}, Int<1>{});
  next_weights();

  // A round multiplies 16 values of k per lane half and prepares the operands of the round behind it, in MT chunks: one
  // MFMA, one read of x, 4 / MT unpacked pairs, at most two loads.  S: the slot of the group.
  auto chunk_of = [&](auto s_tag, auto e_tag, auto c_tag) {
    constexpr int S = decltype(s_tag)::value, E = decltype(e_tag)::value, c = decltype(c_tag)::value;
    constexpr int kPairs = 4 / MT;
    constexpr unsigned int s_cur = S * STAGE, s_next = (S + 1) % 3 * STAGE;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (E == 0) issue(Int<(S + 2) % 3>{}, Int<2 + c>{});         // x of the group two ahead
    if constexpr (E == 3 && c == 0) issue(s_tag, Int<0>{});                // weights of the group four ahead
    if constexpr (E == 3 && c == MT - 1) issue(s_tag, Int<1>{});
    if (E < 3 && c == 0) read_weights(s_cur, pk_next, E);                  // the weights of the next group came with x of this one
    if (E == 2 && c == 0) read_scales(s_cur);
    if (E == 2 && c == MT - 1) read_weights(s_cur, pk_next, 3);
    if (E == 3 && c == 0) decode_scales();
    E == 3 ? read_x(s_next, 0, c) : read_x(s_cur, (E + 1) & 3, c);
#pragma unroll
    for (int p = c * kPairs; p < (c + 1) * kPairs; ++p) unpack(E == 3 ? pk_next : pk, (E + 1) & 3, p);
    multiply(E & 1, c);
  };
  auto round = [&](auto s_tag, auto e_tag) {
    chunk_of(s_tag, e_tag, Int<0>{});
    if constexpr (MT >= 2) chunk_of(s_tag, e_tag, Int<1>{});
    if constexpr (MT >= 4) { chunk_of(s_tag, e_tag, Int<2>{}); chunk_of(s_tag, e_tag, Int<3>{}); }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto group = [&](auto s_tag) {
    round(s_tag, Int<0>{});
    x_rows.next();
    round(s_tag, Int<1>{});
    round(s_tag, Int<2>{});
    // The next slot is complete once only the loads of the slot behind it (weights, x) are outstanding, and everybody has read all of
    // this one, which then takes group i + 3.  Behind the last group the reads return old bytes; nothing uses them.
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");
    art_lds_barrier();
    round(s_tag, Int<3>{});
    next_weights();
#pragma unroll
    for (int e = 0; e < 4; ++e) pk[e] = pk_next[e];
  };
  for (int left = groups;;) {                       // the slots are constants
    group(Int<0>{});
    if (--left == 0) break;
    group(Int<1>{});
    if (--left == 0) break;
    group(Int<2>{});
    if (--left == 0) break;
  }

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing of the ring is on its way when its space is reused or given back

  // ---- the two k halves meet: wavefront (c, h) hands half of its sums to (c, 1 - h), by fours of rows, and keeps the other.
  // Accumulator elements 4 (q % 4) .. + 3 of tile q / 4 are rows (q / 4) * 32 + (q % 4) * 8 + (lane / 32) * 4 .. + 3.
  constexpr int KEEP = 2 * MT;
  f32x4* const meet = reinterpret_cast<f32x4*>(smem) + cw * KEEP * 64 + lane;
  auto quad = [&](int q) { return f32x4{acc[q >> 2][4 * (q & 3)], acc[q >> 2][4 * (q & 3) + 1], acc[q >> 2][4 * (q & 3) + 2], acc[q >> 2][4 * (q & 3) + 3]}; };
  f32x4 sum[KEEP];
  auto row_of = [&](int j) { return ((kh * KEEP + j) >> 2) * 32 + ((kh * KEEP + j) & 3) * 8 + h * 4; };
  __syncthreads();
  if (kh == 0) {
#pragma unroll
    for (int j = 0; j < KEEP; ++j) { meet[(4 * KEEP + j) * 64] = quad(KEEP + j); sum[j] = quad(j); }
  } else {
#pragma unroll
    for (int j = 0; j < KEEP; ++j) { meet[j * 64] = quad(j); sum[j] = quad(KEEP + j); }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KEEP; ++j) sum[j] += meet[(4 * KEEP * kh + j) * 64];
  if (work.splits > 1) {                            // 64 bytes and more of a row at a time
    if (!cols.inside(colpos)) return;
    const PartialTile to(partial, split, M, N);
    const unsigned int at = to.at(m0 + row_of(0), cols.at(colpos));
#pragma unroll
    for (int j = 0; j < KEEP; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) to.store(at, (j >> 2) * 32 + (j & 3) * 8 + i, sum[j][i]);
    return;
  }
  // fp16 results to LDS as [row][column], out in pieces of eight columns.
  constexpr int COLS = SWIGLU ? BN / 2 : BN, C_LD = COLS + 8;
  _Float16* const cs = reinterpret_cast<_Float16*>(smem + 8 * KEEP * 1024);
#pragma unroll
  for (int j = 0; j < KEEP; ++j) {
    if constexpr (SWIGLU) {                         // lanes 0-15 hold a gate column, lanes 16-31 its up column
#pragma unroll
      for (int i = 0; i < 4; i += 2) {              // exchanged: the former have both of one row, the latter both of the next
        const float here = sum[j][i], next = sum[j][i + 1];      // (a bit cast of an element of a vector takes its first one)
        const auto pair = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned int, here), __builtin_bit_cast(unsigned int, next), false, false);
        const float g = (float)(_Float16)__builtin_bit_cast(float, (unsigned int)pair[0]), u = (float)(_Float16)__builtin_bit_cast(float, (unsigned int)pair[1]);
        cs[(row_of(j) + i + hi16) * C_LD + cw * 16 + s16] = (_Float16)(art::silu(g) * u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) cs[(row_of(j) + i) * C_LD + colpos] = (_Float16)sum[j][i];
    }
  }
  __syncthreads();
  if constexpr (ROPE) {
    _Float16* const to = rope.at(head);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int row = (tid + i * kThreads) >> 3, c8 = (tid & 7) * 8;
      if (row >= BM || m0 + row >= M) break;
      h8 a = *reinterpret_cast<const h8*>(cs + row * C_LD + c8), b = *reinterpret_cast<const h8*>(cs + row * C_LD + c8 + 64);
      if (rotated) rotate(a, b, angles[i]);
      _Float16* const out = to + (size_t)(m0 + row) * (rope.heads * 128) + c8;
      *reinterpret_cast<h8*>(out) = a;
      *reinterpret_cast<h8*>(out + 64) = b;
    }
    return;
  }
#pragma unroll 1
  for (int e = tid; e < BM * (COLS / 8); e += kThreads) {
    const int row = e / (COLS / 8), c8 = (e % (COLS / 8)) * 8;
    if (m0 + row >= M || !cols.inside(c8)) continue;
    const size_t out = (size_t)(m0 + row) * (SWIGLU ? N / 2 : N) + cols.at(c8);
    h8 o = *reinterpret_cast<const h8*>(cs + row * C_LD + c8);
    if (TAIL == kPlain && residual) {                      // y = fp16(fp16(product) + residual); may alias y: same elements
      const h8 res = *reinterpret_cast<const h8_by_8*>(residual + out);
#pragma unroll
      for (int k = 0; k < 8; ++k) o[k] = (_Float16)((float)o[k] + (float)res[k]);
    }
    *reinterpret_cast<h8_by_8*>(y + out) = o;
  }
}

// Four neighbouring sums over the K-splits, in split order, all loads issued before the first is added (a loop of load-then-add
// runs one memory round trip per split).  SPLITS: their number, up to eight; 0: eight at a time, where past the last one a load
// repeats split 0 and is not added.  With the number known, product and pass together: 128 rows over 4096 x 4096 in three splits
// 15.0 -> 14.7 us, 50 rows in four 10.9 -> 10.7, 16 rows over 4096 x 12288 in two 13.6 -> 13.4.
template <int SPLITS>
__device__ __forceinline__ f32x4 sum_splits(const float* partial, long long split_stride, int splits) {
  f32x4 t = *reinterpret_cast<const f32x4*>(partial);
  if constexpr (SPLITS > 0) {
    f32x4 v[SPLITS];
#pragma unroll
    for (int j = 1; j < SPLITS; ++j) v[j] = *reinterpret_cast<const f32x4*>(partial + j * split_stride);
#pragma unroll
    for (int j = 1; j < SPLITS; ++j) t += v[j];
    return t;
  }
  for (int s0 = 1; s0 < splits; s0 += 8) {
    f32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const f32x4*>(partial + (s0 + j < splits ? s0 + j : 0) * split_stride);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < splits) t += v[j];
  }
  return t;
}

// Which part of a row the pass adds where: block b runs on XCD b % 8 and takes that eighth of the columns (by_eighths; else whole rows in
// order).  The product deals its column tiles, with all their K-splits, to the XCDs in the same order (Deal, art_gemm_w4_deep.hip), so that the
// sums are in the L2 that they were written to unless the weights have pushed them out.  With rows dealt whole, product and pass, HBM / cache, us: 50 rows over
// 4096 x 4096 in four splits 11.1 / 9.9, now 9.8 / 8.6, 64 over 8192 x 2048 in eight 11.2 / 10.3 and 10.0 / 9.0, 30 over 5504 x 2048 8.4 / 7.9 and 7.7 / 7.0; over
// 11008 x 4096 (3 MB of weights per XCD) 1 % either way.
struct Part {
  Div across;                                       // pieces of a row in a part: an eighth of them, or all
  int pieces;                                       // of a row
  // false: nothing to do
  __device__ __forceinline__ bool take(int rows, unsigned& row, unsigned& piece) const {
    const bool whole = (int)across.by == pieces;
    const unsigned i = (whole ? blockIdx.x : blockIdx.x >> 3) * 256 + threadIdx.x;
    row = over(i, across);
    piece = i - row * across.by + (whole ? 0 : (blockIdx.x & 7) * across.by);
    return (int)row < rows && (int)piece < pieces;
  }
};

// As numbers, which are in registers when a kernel starts; as a struct, which is not, 1 to 3 % slower.
#define ART_PART_PARAMS unsigned mul, unsigned shift, unsigned across, int pieces
#define ART_PART (Part{Div{mul, shift, across}, pieces})

// y[m,n] = fp16(sum over splits); four columns per thread (N % 4 == 0).
template <int SPLITS> __global__ __launch_bounds__(256) void gemm_w4a16_combine_kernel(const float* __restrict__ partial, _Float16* y,
                                                                  const _Float16* residual, long long split_stride,
                                                                  int splits, int rows, ART_PART_PARAMS) {
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if ((int)across == pieces) {
    if (i >= (long long)rows * pieces) return;
  } else {
    unsigned row, quad;
    if (!ART_PART.take(rows, row, quad)) return;
    i = (long long)row * pieces + quad;
  }
  const f32x4 t = sum_splits<SPLITS>(partial + i * 4, split_stride, splits);
  h4 out = h4{(_Float16)t[0], (_Float16)t[1], (_Float16)t[2], (_Float16)t[3]};
  if (residual) {                    // y = fp16(fp16(product) + residual); residual may be y itself
    const h4 res = *reinterpret_cast<const h4*>(residual + i * 4);
    out = h4{(_Float16)((float)out[0] + (float)res[0]), (_Float16)((float)out[1] + (float)res[1]),
             (_Float16)((float)out[2] + (float)res[2]), (_Float16)((float)out[3] + (float)res[3])};
  }
  *reinterpret_cast<h4*>(y + i * 4) = out;
}

// The same with the RMSNorm that follows (norm_out = fp16(y / rms(y) * weight), from the rounded y): a block owns a row, whose
// elements stay in registers, 8 per thread and turn (N % 8 == 0, N <= 8192; as many threads as a row of up to 4096 has
// pieces of 8).  Bound by the launch: instead of two launches of 2 us and more, one; a layer of the 32-layer model's prompt pass has
// two of them: 8 layers 608 -> 594 us at 8 tokens, 776 -> 750 at 50, 962 -> 925 at 100, 1345 -> 1337 at 200 (fewer K-splits meet).
// The sum over a row is bound by its steps: by DPP instead of six trips through LDS, the wavefronts' sums read at once, product and pass
// 9.1 -> 8.9 us at 8 rows over 4096 x 4096, 14.3 -> 14.0 at 128 rows, 2048 x 2048 6.5 -> 6.2 and 9.2 -> 8.9.
constexpr int kNormThreads = 512, kNormTurns = 2;
// Sum over the 64 lanes of a wavefront; every lane gets it.
__device__ __forceinline__ float wave_sum(float v) {
#define ART_DPP_ADD(ctrl) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, false))
  ART_DPP_ADD(0xB1);                                // quad_perm [1,0,3,2]
  ART_DPP_ADD(0x4E);                                // quad_perm [2,3,0,1]
  ART_DPP_ADD(0x141);                               // row_half_mirror
  ART_DPP_ADD(0x140);                               // row_mirror
#undef ART_DPP_ADD
  const int b = __builtin_bit_cast(int, v);
  return (__builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0)) + __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16))) +
         (__builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32)) + __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48)));
}
template <int SPLITS> __global__ __launch_bounds__(kNormThreads) void gemm_w4a16_combine_norm_kernel(const float* __restrict__ partial, const _Float16* residual,
                                                                                const _Float16* __restrict__ weight, _Float16* y, long long split_stride, int N,
                                                                                int splits, int threads, float eps, _Float16* __restrict__ norm_out) {
  __shared__ float s_part[kNormThreads / 64];
  const int tid = threadIdx.x, chunks = N >> 3;
  const size_t row = (size_t)blockIdx.x * N;
  // the norm's weights and the residual are asked for with the sums, not behind them (every lane asks: no branch around a load)
  h8 v[kNormTurns], w[kNormTurns], res[kNormTurns];
  f32x4 lo[kNormTurns], hi[kNormTurns];
  const bool second = chunks > threads;             // the same for the whole launch
#pragma unroll
  for (int i = 0; i < kNormTurns; ++i) {
    if (i > 0 && !second) break;
    const int c = tid + i * threads, at = 8 * (c < chunks ? c : chunks - 1);
    w[i] = *reinterpret_cast<const h8*>(weight + at);
    if (residual) res[i] = *reinterpret_cast<const h8*>(residual + row + at);
    lo[i] = sum_splits<SPLITS>(partial + row + at, split_stride, splits);
    hi[i] = sum_splits<SPLITS>(partial + row + at + 4, split_stride, splits);
  }
  float a = 0.f;
#pragma unroll
  for (int i = 0; i < kNormTurns; ++i) {
    const int c = tid + i * threads;
    if (c >= chunks) break;
#pragma unroll
    for (int k = 0; k < 8; ++k) v[i][k] = (_Float16)(k < 4 ? lo[i][k] : hi[i][k - 4]);
    if (residual) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[i][k] = (_Float16)((float)v[i][k] + (float)res[i][k]);
    }
    *reinterpret_cast<h8*>(y + row + 8 * (size_t)c) = v[i];
#pragma unroll
    for (int k = 0; k < 8; ++k) a = fmaf((float)v[i][k], (float)v[i][k], a);
  }
  a = wave_sum(a);
  if ((tid & 63) == 0) s_part[tid >> 6] = a;
  art_lds_barrier();                                // LDS only: y need not have landed
  const int waves = threads >> 6;
  float ss = 0.f;                                   // fixed length: one trip to LDS, not one for each wavefront
#pragma unroll
  for (int k = 0; k < kNormThreads / 64; ++k) {
    const float part = s_part[k];
    ss += k < waves ? part : 0.f;
  }
  const float r = 1.0f / sqrtf(ss * (1.0f / (float)N) + eps);
#pragma unroll
  for (int i = 0; i < kNormTurns; ++i) {
    const int c = tid + i * threads;
    if (c >= chunks) break;
    h8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = (_Float16)((float)v[i][k] * r * (float)w[i][k]);
    *reinterpret_cast<h8*>(norm_out + row + 8 * (size_t)c) = o;
  }
}

// The same for gate | up: y[m, n] of N / 2 columns from the sums of columns n and N / 2 + n.
template <int SPLITS> __global__ __launch_bounds__(256) void gemm_w4a16_combine_swiglu_kernel(const float* __restrict__ partial, _Float16* y, int rows, int N,
                                                                         int splits, ART_PART_PARAMS) {   // groups of four output columns
  unsigned m, quad;
  if (!ART_PART.take(rows, m, quad)) return;
  const long long row = m, col = quad * 4, stride = (long long)rows * N;
  const f32x4 g = sum_splits<SPLITS>(partial + row * N + col, stride, splits), u = sum_splits<SPLITS>(partial + row * N + N / 2 + col, stride, splits);
  *reinterpret_cast<h4*>(y + row * (N / 2) + col) = swiglu4(h4{(_Float16)g[0], (_Float16)g[1], (_Float16)g[2], (_Float16)g[3]},
                                                            h4{(_Float16)u[0], (_Float16)u[1], (_Float16)u[2], (_Float16)u[3]});
}

// The same for q | k | v: columns j .. j + 3 of a head and their partners 64 further on, rotated in q and k.
template <int SPLITS> __global__ __launch_bounds__(256) void gemm_w4a16_combine_rope_kernel(const float* __restrict__ partial, int rows, int splits, ART_PART_PARAMS, Rope rope) {      // 48 heads of them
  unsigned m, at;
  if (!ART_PART.take(rows, m, at)) return;
  const long long row = m, stride = (long long)rows * pieces * 8;
  const int head = at >> 4, j = (at & 15) * 4;
  const float* const from = partial + (row * pieces * 8 + head * 128 + j);
  const f32x4 first = sum_splits<SPLITS>(from, stride, splits), second = sum_splits<SPLITS>(from + 64, stride, splits);
  h4 a = h4{(_Float16)first[0], (_Float16)first[1], (_Float16)first[2], (_Float16)first[3]};
  h4 b = h4{(_Float16)second[0], (_Float16)second[1], (_Float16)second[2], (_Float16)second[3]};
  if (rope.rotated(head)) rotate(a, b, load_angles<4>(rope.angles + row * 64 + j));
  _Float16* const to = rope.at(head) + row * rope.heads * 128 + j;
  *reinterpret_cast<h4*>(to) = a;
  *reinterpret_cast<h4*>(to + 64) = b;
}

// ---- Which kernel, rows per block and K-splits.
struct Plan {
  bool wide;
  int row_tiles, splits;
  int deep;                                         // column tiles of a block of art_gemm_w4_deep.hip, 0: not that kernel
};
// What a launch takes, in microseconds.  K-splits: the second launch and the fp32 tiles on top.  A pass that also turns or gates costs a
// prompt more than it costs alone (q | k | v of 64 rows over 4096 x 12288, in a prompt's trace: one launch 18.8, two splits 16.1 and the pass 5.0; in a loop
// of its own 18.6 and 17.7), and waits twice for more than eight (8 rows, K = 3712, one head: 5.8 in seven splits, 9.3 in fifteen).
double splits_estimate(int M, int N, int splits, Tail tail) {
  return splits > 1 ? 1.8 + (8.0 * splits + 2.0) * M * N / 4.2e6 + (tail == kPlain ? 0.0 : splits > 8 ? 3.5 : 0.849) : 0.0;
}
// Where K-splits meet in a pass of their own, a norm is part of that pass, up to 256 rows: beyond them nothing is
// gained (8 layers of the same pass: 1384 -> 1368 us at 256 tokens, 1861 and 1854 at 300, 2178 and 2183 at 500).
bool norm_fits(int M, int N) { return M <= 256 && N % 8 == 0 && N <= 8 * kNormThreads * kNormTurns; }
// Else it is a launch of its own.  (Of more than eight splits the pass waits twice.)
double norm_estimate(int M, int N, int splits) { return splits == 1 ? 3.046 + 2.178e-6 * M * N : splits > 8 ? 1.0 : 0.0; }
// A fixed part, one or two co-resident blocks' time per group and round (one's: more with more of the compute units at work; either: more where
// several blocks of rows unpack the same weights; two's: more where rows are whole KiB apart, and for the halves of gate | up), the ramp and
// the meeting of the k halves again for every further round of blocks of 128 columns (4 rows over 4096 x 12288: 13.3 us with 480 blocks, i.e. 5 K-splits
// in one round, 14.6 with 768).  Constants of 128 columns x 128 rows and of 256 columns are from all forms over 6200 sizes of 4 to 1003 rows on MI355X, a
// quarter with weights that stay in the last-level cache.  The others and deep_estimate's are from 2678 sizes of 4 to 512 rows, each with
// weights from HBM and from the cache, the former counting 70 %, and from 3469 prompts of 4 to 620 tokens (models of 8 to 64 heads): for each product of a
// layer, what another form does to the layer's time.  The pick is 0.9 % (HBM) and 1.4 % (cache) slower than the fastest
// form, a layer of a prompt 0.8 %.  Before there were terms for blocks of rows, rows whole KiB apart and halves: 2.1, 1.6 and 1.4 %, and 20 to 40 % at some
// (weights from HBM, us: 8 rows over 4096 x 4096 10.1, now 7.8; 5120 x 5120 14.0, 9.2; 64 rows over 11008 x 4096 18.5, 15.9; 256 rows 34.4, 32.1).
// Products from the cache would rather keep the narrow blocks there (8 rows over 5120 x 5120 6.9, now 7.9).
double estimate(int M, int K, int N, const Plan& p, Tail tail, int compute_units) {
  struct Cost { double fixed, one, two; int per_cu; double busy, rows, whole_kib, halves; };
  const Cost c = p.wide ? (p.row_tiles == 8 ? Cost{8.5, 2.16, 1.94, 1, 0, 0, 0, 0} : Cost{5.2, 1.2, 2.3, 2, 0, 0, 0, 0})
                 : p.row_tiles == 4 ? Cost{4.8, 0.52, 0.82, 1, 0, 0, 0, 0}
                 : p.row_tiles == 2 ? Cost{4.419, 0.372, 0.915, 2, 0.1, 0.065, 0.005, 0.04} : Cost{3.697, 0.388, 0.831, 2, 0, 0.053, 0.011, 0};
  const int groups = (K / GK + p.splits - 1) / p.splits, m_blocks = (M + 32 * p.row_tiles - 1) / (32 * p.row_tiles);
  const int blocks = tile_count(N, false, p.wide ? 256 : BN) * m_blocks * p.splits, round = c.per_cu * compute_units, rest = blocks % round;
  const double busy = blocks < compute_units ? (double)blocks / compute_units : 1.0;
  double one = 0.0, two = blocks / round;           // rounds of each kind
  if (rest > compute_units) two += 1.0;
  else if (rest > 0) {
    one = c.per_cu == 2 || blocks > round ? 1.0 : 1.0 - (double)rest / compute_units;
    two += 1.0 - one;
  }
  const double waits = ((N % 1024 == 0 ? c.whole_kib : 0.0) + (tail == kSwiglu ? c.halves : 0.0)) / m_blocks;       // (blocks of rows share weights)
  const double per_group = (c.one + c.busy * busy) * one + (c.two + waits) * two + c.rows * busy * (1.0 - 1.0 / m_blocks) * (one + two);
  const double again = p.wide ? 0.0 : 0.73 * ((blocks - 1) / round);
  return c.fixed + again + groups * per_group + splits_estimate(M, N, p.splits, tail);
}
// art_gemm_w4_deep.hip: a fixed part and, for each group, what the load path of a compute unit needs for it (all eight wavefronts share it,
// so groups count, not rounds of them), more with more of the compute units at work and with each further block on one.  Narrow blocks
// have few bytes on their way to HBM, and wait longest where rows are whole KiB apart (4992 x 3808, one split: 9.5 us; 5120 x 5120: 13.9, from the
// cache 6.8) and for pieces of 16 columns of two halves (gate | up).
double deep_estimate(int M, int K, int N, const Plan& p, Tail tail, int compute_units) {
  struct Cost { double fixed, group, busy, further, again, whole_kib, halves; };
  const Cost c = p.deep == 2 ? (M <= 16 ? Cost{3.23, 0.178, 0.04, 0.257, 0.404, 0.036, 0.014} : Cost{3.21, 0.213, 0.064, 0.205, 1.88, 0.017, 0.035})
                 : p.row_tiles == 2 ? Cost{3.449, 0.2, 0.101, 0.219, 1.577, 0.02, 0.028}
                 : M <= 16 ? Cost{2.737, 0.102, 0.069, 0.148, 0.387, 0.04, 0.024} : Cost{2.943, 0.147, 0.051, 0.162, 1.471, 0.024, 0.028};
  const int groups = (K / GK + p.splits - 1) / p.splits, m_blocks = (M + 32 * p.row_tiles - 1) / (32 * p.row_tiles);
  const int blocks = deep_tiles(N, tail, p.deep) * m_blocks * p.splits, more = (blocks - 1) / compute_units;
  const double busy = blocks < compute_units ? (double)blocks / compute_units : 1.0;
  const double waits = (N % 1024 == 0 ? c.whole_kib : 0.0) + (tail == kSwiglu ? c.halves : 0.0);
  return c.fixed + groups * (c.group + c.busy * busy + c.further * more + waits * (1 + more)) + c.again * more + splits_estimate(M, N, p.splits, tail);
}
constexpr int kDeepBlocks = 8;                      // of rows
// What a form's 32-bit offsets (a block's rows of x and of the packed weights), its division by the number of column
// tiles and its grid hold.  Where the packed weights of a split do not fit 32 bits, two of the forms are left.  Offsets end below 4 GiB - 1,
// the limit of a descriptor: of a load that ends at it the last word comes back as zero.  (x: with K-splits a block's rows end before that.)
int groups_of(const Plan& p, int K) { return (K / GK + p.splits - 1) / p.splits; }
bool far(const Plan& p, int K, int N) { return 64LL * N * groups_of(p, K) >= 1LL << 32; }
bool holds(const Plan& p, int M, int K, int N, Tail tail) {
  const int rows = M < 32 * p.row_tiles ? M : 32 * p.row_tiles;
  const long long padded = (M + 32LL * p.row_tiles - 1) / (32 * p.row_tiles) * (32 * p.row_tiles);
  if (p.splits > 1 && 4LL * N * padded > 1LL << 32) return false;       // PartialTile
  const bool offsets = 64LL * p.row_tiles * K <= 1LL << 32 && 2LL * K * (rows - 1) + 256LL * groups_of(p, K) < 1LL << 32 && 64LL * N <= 1LL << 32;
  if (p.deep) return offsets && !far(p, K, N) && (long long)deep_tiles(N, tail, p.deep) * p.splits < 1 << 16 && M <= 32 * p.row_tiles * kDeepBlocks;
  const long long units = (long long)tile_count(N, tail == kSwiglu, p.wide ? 256 : BN) * p.splits;
  return offsets && units < (p.wide ? 1 << 19 : 1 << 16) && (!far(p, K, N) || p.row_tiles == (p.wide ? 4 : 1));
}
// What a caller's k_splits calls a form: rows of a block / 32, 5: 128 rows x 128 columns, 9, 10, 11: art_gemm_w4_deep.hip with 32 x 32, 32 x 64,
// 64 rows x 32 columns.
int code_of(const Plan& p) { return p.deep ? 7 + 2 * p.row_tiles + (p.deep == 2 ? 1 : 0) : !p.wide && p.row_tiles == 4 ? 5 : p.row_tiles; }
// False: no form takes these sizes.  `code` and `splits` are the caller's wishes (0: none; splits alone: not the deep kernel); a form that
// does not hold the sizes is replaced by one that does.  A product with a
// residual counts as one with a norm behind it, in its own call or the next: the bits of y are the same in both.
bool choose(Plan& best, int M, int K, int N, Tail tail, bool residual, size_t scratch_bytes, int compute_units, int code, int splits) {
  const int G = K / GK;
  const size_t per_split = (size_t)M * N * sizeof(float);
  const int cap = (int)(scratch_bytes / per_split), most = G < cap ? G : (cap < 1 ? 1 : cap);
  double t_best = 1e30;
  const bool norm_in_pass = residual && norm_fits(M, N);
  auto consider = [&](const Plan& p, double t) {
    if (norm_in_pass) t += norm_estimate(M, N, p.splits);
    if (t < t_best) { t_best = t; best = p; }
  };
  for (int pass = 0; pass < 3 && t_best == 1e30; ++pass) {        // the wishes; without the form; without the splits
    for (const Plan form : {Plan{false, 1, 1, 0}, Plan{false, 2, 1, 0}, Plan{false, 4, 1, 0}, Plan{true, 4, 1, 0}, Plan{true, 8, 1, 0},
                            Plan{false, 1, 1, 1}, Plan{false, 1, 1, 2}, Plan{false, 2, 1, 1}}) {
      if (form.deep && (pass > 0 || code == 0 && splits > 0)) continue;
      if (pass == 0 && (code != 0 ? code != code_of(form) : 16 * form.row_tiles >= M && form.row_tiles > 1)) continue;      // not over twice the rows
      for (int s = splits > 0 ? splits : 1; s <= (splits > 0 ? splits : form.deep ? 16 : 32); ++s) {
        if (splits == 0 && s > 1 && (s > most || 2 * s > G + 1)) break;
        const Plan p{form.wide, form.row_tiles, s > most ? most : s, form.deep};
        if (holds(p, M, K, N, tail)) consider(p, p.deep ? deep_estimate(M, K, N, p, tail, compute_units) : estimate(M, K, N, p, tail, compute_units));
      }
    }
    if (t_best == 1e30) splits = pass == 0 ? 1 : 0;
  }
  return t_best < 1e30;
}
// An RMSNorm of the result: out = fp16(y / rms(y) * weight).
struct Norm {
  const void* weight;
  void* out;
  float eps;
};

template <int SPLITS>
void launch_combine(const float* partial, _Float16* y, int rows, int N, int splits, const _Float16* residual, Tail tail, const Norm* norm,
                    const Rope& rope, hipStream_t stream) {
  const int pieces = tail == kPlain ? N / 4 : N / 8;
  const Div across = make_div((unsigned)(by_eighths(N, tail) ? (pieces + 7) / 8 : pieces));
  const unsigned blocks = (unsigned)(((long long)rows * across.by + 255) / 256) * ((int)across.by == pieces ? 1 : 8);
  if (norm) {
    const int threads = N < 8 * kNormThreads ? (N / 8 + 63) / 64 * 64 : kNormThreads;
    gemm_w4a16_combine_norm_kernel<SPLITS><<<dim3(rows), threads, 0, stream>>>(partial, residual, (const _Float16*)norm->weight, y, (long long)rows * N, N, splits,
                                                                               threads, norm->eps, (_Float16*)norm->out);
  } else if (tail == kRope) {
    gemm_w4a16_combine_rope_kernel<SPLITS><<<blocks, 256, 0, stream>>>(partial, rows, splits, across.mul, across.shift, across.by, pieces, rope);
  } else if (tail == kSwiglu) {
    gemm_w4a16_combine_swiglu_kernel<SPLITS><<<blocks, 256, 0, stream>>>(partial, y, rows, N, splits, across.mul, across.shift, across.by, pieces);
  } else {
    gemm_w4a16_combine_kernel<SPLITS><<<blocks, 256, 0, stream>>>(partial, y, residual, (long long)rows * N, splits, rows, across.mul, across.shift, across.by, pieces);
  }
}
int combine(const float* partial, _Float16* y, int rows, int N, int splits, const _Float16* residual, Tail tail, const Norm* norm, const Rope& rope,
            hipStream_t stream) {
  static const decltype(&launch_combine<0>) by_splits[9] = {launch_combine<0>, launch_combine<0>, launch_combine<2>, launch_combine<3>, launch_combine<4>,
                                                            launch_combine<5>, launch_combine<6>, launch_combine<7>, launch_combine<8>};
  by_splits[splits <= 8 ? splits : 0](partial, y, rows, N, splits, residual, tail, norm, rope, stream);
  ART_LAUNCH_CHECK();
  return 0;
}

// One launch of the product (and of the pass behind it) over up to kMaxRows rows.
constexpr int kMaxRows = 1 << 18;                   // 8192 blocks of 32 rows
int run_rows(const _Float16* xs, const unsigned char* qweight, const _Float16* scales, const unsigned char* qzeros, _Float16* ys, const _Float16* res,
             int M, int K, int N, int code, int splits, Tail tail, const Norm* norm, const Rope& rope, float* scratch, size_t scratch_bytes, hipStream_t st) {
  const bool swiglu = tail == kSwiglu;
  Plan p;
  ART_REQUIRE(choose(p, M, K, N, tail, res != nullptr, scratch_bytes, art::compute_units(), code, splits), "art_gemm_w4a16: K=%d N=%d are too large", K, N);
  const bool norm_there = norm && p.splits > 1 && norm_fits(M, N) &&
                          (((uintptr_t)ys | (uintptr_t)res | (uintptr_t)norm->weight | (uintptr_t)norm->out) % 16) == 0;
  if (p.deep) {
    if (art::w4::gemm_deep(xs, qweight, scales, qzeros, ys, scratch, M, K, N, p.splits, p.row_tiles, p.deep, res, tail, rope, st)) return 1;
  } else if (p.wide) {
    if (art::w4::gemm_wide(xs, qweight, scales, qzeros, ys, scratch, M, K, N, p.splits, p.row_tiles, far(p, K, N), res, tail, rope, st)) return 1;
  } else {
    static const decltype(&gemm_w4a16_kernel<1, kPlain>) kernels[4][3] = {
        {gemm_w4a16_kernel<1, kPlain>, gemm_w4a16_kernel<1, kSwiglu>, gemm_w4a16_kernel<1, kRope>},
        {gemm_w4a16_kernel<2, kPlain>, gemm_w4a16_kernel<2, kSwiglu>, gemm_w4a16_kernel<2, kRope>},
        {gemm_w4a16_kernel<4, kPlain>, gemm_w4a16_kernel<4, kSwiglu>, gemm_w4a16_kernel<4, kRope>},
        {gemm_w4a16_kernel<1, kPlain, true>, gemm_w4a16_kernel<1, kSwiglu, true>, gemm_w4a16_kernel<1, kRope, true>}};
    static bool configured = false;
    if (!configured) {
      for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 3; ++j)
          ART_HIP(hipFuncSetAttribute((const void*)kernels[i][j], hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes(i == 3 ? 1 : 1 << i)));
      configured = true;
    }
    const int col_tiles = tile_count(N, swiglu, BN), m_blocks = (M + 32 * p.row_tiles - 1) / (32 * p.row_tiles);
    const int units = col_tiles * p.splits, G = K / GK;
    dim3 grid;
    const Work work{deal(units, m_blocks, grid), p.splits, (unsigned int)((0x100000000ull + p.splits - 1) / p.splits), G / p.splits, G % p.splits};
    const auto kernel = kernels[far(p, K, N) ? 3 : p.row_tiles == 4 ? 2 : p.row_tiles - 1][tail];
    kernel<<<grid, kThreads, lds_bytes(p.row_tiles), st>>>(xs, qweight, scales, qzeros, ys, scratch, M, K, N, work, kMagic, res, rope);
    ART_LAUNCH_CHECK();
  }
  if (p.splits > 1 && combine(scratch, ys, M, N, p.splits, res, tail, norm_there ? norm : nullptr, rope, st)) return 1;
  return norm && !norm_there ? art_rmsnorm(ys, nullptr, norm->weight, norm->out, M, N, 1.0f / (float)N, norm->eps, 1, 1, 1, st) : 0;
}

bool code_taken(int k_splits) {
  const int code = k_splits >> 8;
  return k_splits >= 0 && (code <= 2 || code == 4 || code == 5 || code >= 8 && code <= 11);
}

int run(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev, void* y_dev, const void* residual_dev,
        int M, int K, int N, int k_splits, Tail tail, const Norm* norm, const Rope* rope, void* stream) {
  const int n_out = tail == kSwiglu ? N / 2 : tail == kRope ? N / 3 : N;
  const int code = k_splits >> 8;                   // 0: library's choice; else code_of
  ART_REQUIRE(code_taken(k_splits),
              "art_gemm_w4a16: k_splits must be 0 (library's choice) or 1..255, plus 256 x the rows-per-block code 1, 2, 4, 5 or 8 to 11 (got %d)", k_splits);
  ART_REQUIRE(((uintptr_t)residual_dev % 8) == 0, "art_gemm_w4a16: the residual must be 8-byte aligned");
  ART_REQUIRE(!art::overlaps(x_dev, (size_t)M * K * 2, y_dev, (size_t)M * n_out * 2), "art_gemm_w4a16: y must not overlap x");
  ART_REQUIRE(x_dev && qweight_dev && scales_dev && qzeros_dev && y_dev, "art_gemm_w4a16: null pointer");
  ART_REQUIRE(M >= 1, "art_gemm_w4a16: M must be positive (got %d)", M);
  ART_REQUIRE(K > 0 && N > 0 && K % 128 == 0 && N % 16 == 0, "art_gemm_w4a16: need K %% 128 == 0 and N %% 16 == 0 (K=%d N=%d)", K, N);
  ART_REQUIRE(((uintptr_t)qweight_dev % 16) == 0 && ((uintptr_t)x_dev % 16) == 0 && ((uintptr_t)qzeros_dev % 8) == 0 &&
                  ((uintptr_t)y_dev % 8) == 0 && ((uintptr_t)scales_dev % 4) == 0,
              "art_gemm_w4a16: x and qweight must be 16-byte aligned, qzeros and y 8-byte aligned, scales 4-byte aligned");
  art::Workspace* ws = art::workspace((hipStream_t)stream);
  if (!ws) return 1;
  float* scratch = reinterpret_cast<float*>((char*)ws->base + art::kScratchOffset);
  const size_t scratch_bytes = ws->bytes - art::kScratchOffset;
  for (int m0 = 0; m0 < M; m0 += kMaxRows) {
    const size_t out = (size_t)m0 * n_out;
    const Norm rows_norm = norm ? Norm{norm->weight, (_Float16*)norm->out + out, norm->eps} : Norm{};
    const size_t d = (size_t)N / 3 * m0;
    const Rope rows_rope = rope ? Rope{rope->angles + 64 * (size_t)m0, rope->q + d, rope->k + d, rope->v + d, rope->heads} : Rope{};
    if (run_rows((const _Float16*)x_dev + (size_t)m0 * K, (const unsigned char*)qweight_dev, (const _Float16*)scales_dev, (const unsigned char*)qzeros_dev,
                 (_Float16*)y_dev + out, residual_dev ? (const _Float16*)residual_dev + out : nullptr, M - m0 < kMaxRows ? M - m0 : kMaxRows, K, N, code,
                 k_splits & 0xff, tail, norm ? &rows_norm : nullptr, rows_rope, scratch, scratch_bytes, (hipStream_t)stream))
      return 1;
    if (M - m0 <= kMaxRows) break;                  // m0 does not pass the largest int
  }
  return 0;
}

}  // namespace

extern "C" int art_gemm_w4a16_form(int M, int K, int N, int tail, int residual, int k_splits) {
  Plan p;
  if (M < 1 || K < 1 || N < 1 || K % GK != 0 || N % 16 != 0 || tail < kPlain || tail > kRope || !code_taken(k_splits)) return 0;
  if (!choose(p, M < kMaxRows ? M : kMaxRows, K, N, (Tail)tail, residual != 0, art_workspace_bytes() - art::kScratchOffset, 256, k_splits >> 8, k_splits & 0xff)) return 0;
  return 256 * code_of(p) + p.splits;
}

extern "C" int art_gemm_w4a16(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev,
                              void* y_dev, int M, int K, int N, void* stream) {
  return art_gemm_w4a16_tuned(x_dev, qweight_dev, scales_dev, qzeros_dev, y_dev, M, K, N, 0, stream);
}

extern "C" int art_gemm_w4a16_tuned(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev,
                                    void* y_dev, int M, int K, int N, int k_splits, void* stream) {
  return art_gemm_w4a16_residual(x_dev, qweight_dev, scales_dev, qzeros_dev, y_dev, nullptr, M, K, N, k_splits, stream);
}

extern "C" int art_gemm_w4a16_residual(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev,
                                       void* y_dev, const void* residual_dev, int M, int K, int N, int k_splits, void* stream) {
  return run(x_dev, qweight_dev, scales_dev, qzeros_dev, y_dev, residual_dev, M, K, N, k_splits, kPlain, nullptr, nullptr, stream);
}

extern "C" int art_gemm_w4a16_swiglu(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev,
                                     void* y_dev, int M, int K, int N, int k_splits, void* stream) {
  ART_REQUIRE(N % 32 == 0, "art_gemm_w4a16_swiglu: the gate and up halves must be multiples of 16 columns (N=%d)", N);
  return run(x_dev, qweight_dev, scales_dev, qzeros_dev, y_dev, nullptr, M, K, N, k_splits, kSwiglu, nullptr, nullptr, stream);
}

extern "C" int art_gemm_w4a16_residual_norm(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev,
                                            void* y_dev, const void* residual_dev, const void* norm_weight_dev, void* norm_out_dev, int M, int K,
                                            int N, float eps, int k_splits, void* stream) {
  ART_REQUIRE(norm_weight_dev && norm_out_dev, "art_gemm_w4a16_residual_norm: null pointer");
  ART_REQUIRE((((uintptr_t)norm_weight_dev | (uintptr_t)norm_out_dev) % 2) == 0, "art_gemm_w4a16_residual_norm: misaligned tensor");
  ART_REQUIRE(!art::overlaps(norm_out_dev, (size_t)M * N * 2, y_dev, (size_t)M * N * 2) &&
                  !art::overlaps(norm_out_dev, (size_t)M * N * 2, residual_dev, residual_dev ? (size_t)M * N * 2 : 0) &&
                  !art::overlaps(norm_out_dev, (size_t)M * N * 2, norm_weight_dev, (size_t)N * 2) &&
                  !art::overlaps(norm_out_dev, (size_t)M * N * 2, x_dev, (size_t)M * K * 2),
              "art_gemm_w4a16_residual_norm: the normalised result must not overlap an operand or the result");
  const Norm norm{norm_weight_dev, norm_out_dev, eps};
  return run(x_dev, qweight_dev, scales_dev, qzeros_dev, y_dev, residual_dev, M, K, N, k_splits, kPlain, &norm, nullptr, stream);
}

extern "C" int art_gemm_w4a16_rope_store(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev,
                                         const void* angles_dev, void* q_out_dev, void* key_cache_dev, void* val_cache_dev, int M, int K, int heads,
                                         int first_pos, int max_positions, int k_splits, void* stream) {
  ART_REQUIRE(angles_dev && q_out_dev && key_cache_dev && val_cache_dev, "art_gemm_w4a16_rope_store: null pointer");
  ART_REQUIRE(heads >= 1 && heads < 1 << 22, "art_gemm_w4a16_rope_store: bad shape");
  ART_REQUIRE(M >= 1 && first_pos >= 0 && max_positions >= M && first_pos <= max_positions - M,
              "art_gemm_w4a16_rope_store: positions %d.. of %d rows do not fit caches of %d", first_pos, M, max_positions);
  ART_REQUIRE((((uintptr_t)q_out_dev | (uintptr_t)key_cache_dev | (uintptr_t)val_cache_dev | (uintptr_t)angles_dev) % 16) == 0,
              "art_gemm_w4a16_rope_store: the angles, q and the caches must be 16-byte aligned");
  const size_t row = (size_t)heads * 128, rows = (size_t)M * row * 2, first = (size_t)first_pos * row;
  const Rope rope{(const float2*)angles_dev, (_Float16*)q_out_dev, (_Float16*)key_cache_dev + first, (_Float16*)val_cache_dev + first, heads};
  const void* outs[3] = {rope.q, rope.k, rope.v};
  for (int i = 0; i < 3; ++i)
    ART_REQUIRE(!art::overlaps(x_dev, (size_t)M * K * 2, outs[i], rows) && !art::overlaps(angles_dev, (size_t)M * 512, outs[i], rows) &&
                    !art::overlaps(outs[i], rows, outs[(i + 1) % 3], rows),
                "art_gemm_w4a16_rope_store: q, keys and values must not overlap an operand or each other");
  return run(x_dev, qweight_dev, scales_dev, qzeros_dev, q_out_dev, nullptr, M, K, 3 * heads * 128, k_splits, kRope, nullptr, &rope, stream);
}
