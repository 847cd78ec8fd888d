// Weight-only int4 GEMM for a batch of rows (prefill, four rows and more): the same arithmetic as the GEMV of
// art_gemv_w4.hip,
//     y[m,n] = sum_k x[m,k] * w[k,n],   w[k,n] = fp16(s[g,n] * fp16(q[k,n] - z[g,n])),   group g = k / 128,
// on the matrix cores with fp32 accumulation; w is rounded exactly as the reference's dequant + matmul program
// does (samples/05_llama2_7b_int4.py:135-144 exported with a batch axis).
//
// Design for MI355X:
//   * a block of eight wavefronts owns 256 columns, up to 64 rows and a contiguous range of quantisation groups; it
//     works one group (128 k) per loop iteration;
//   * everything a group needs - 16 KiB of packed weights, 16 KiB of x, 512 B of scales, 128 B of zero points - goes
//     from global memory straight into LDS (global_load_lds_dwordx4 / _dword: no registers hold data in flight), into
//     a ring of four stages, so three groups (100 KiB per compute unit) are on their way while one is multiplied.
//     Register staging two groups ahead held a compute unit to about 45 GB/s; this ring sustains over 100 GB/s;
//   * each lane chooses which 16-byte chunk it fetches, and LDS position (row r, chunk c) holds chunk c ^ (r & 7) of
//     the weights (c ^ (r & 15) of x): the reads below then touch every bank once although rows are 256 bytes apart;
//   * the packed bytes stay packed in LDS.  ds_read_b64_tr_b8 hands a lane the 8 bytes = 16 values of k of ONE column,
//     i.e. the B operand of two v_mfma_f32_32x32x16_f16; a lane unpacks only the columns it multiplies (one shift,
//     four v_bitop3_b32, four packed subtractions of the zero point, four packed multiplications by the scale per
//     word).  The nibble extraction leaves k in the order 0 4 1 5 2 6 3 7; the A operand is permuted the same way
//     (four v_perm_b32 per 16 bytes of x);
//   * wavefront (c, h) multiplies 64 columns (c = 0..3) by the k half h of every group: per group 16 bytes of x and
//     of packed weights per lane and MFMA, 112 KiB of LDS traffic per group instead of 280 KiB with fp16 weights in
//     LDS; the two k halves meet in LDS once, after the loop;
//   * the loop is rolled (one group per iteration, one barrier): the whole kernel is 7 KiB of code.  A launch fetches
//     its code cold - straight-line code costs about 0.3 us per KiB executed - so unrolled stages are not free;
//   * split-K without atomics (5.6 M float atomics cost 75 us on this chip): each K-split writes its fp32 tile to the
//     library workspace and a second small kernel adds the splits in a fixed order and rounds once to fp16 - results
//     do not depend on timing.
#include "art_w4_mfma.h"

namespace {

using namespace art::w4;


constexpr int kThreads = 512;                       // 8 wavefronts: 4 column quarters x 2 k halves
constexpr int BM = 64, BN = 256, GK = 128;          // rows and columns of a block, k of a quantisation group
constexpr int NS = 4;                               // stages of the LDS ring, one quantisation group each
constexpr int W_BYTES = (GK / 2) * BN;              // packed weights of a group: 64 byte-rows x 256 columns
constexpr int X_BYTES = BM * GK * 2;                // x of a group: 64 rows x 128 k, fp16
constexpr int Q_BYTES = 2048;                       // scales (512 B) at 0, zero points (128 B) at 512; the rest takes the idle lanes
constexpr int STAGE = W_BYTES + X_BYTES + Q_BYTES;
constexpr int RLD = BN + 4;                         // floats per row of a result tile in LDS
constexpr size_t kLdsBytes = (size_t)NS * STAGE;    // 139264; the two result tiles of the epilogue (133120) reuse it
static_assert(2 * BM * RLD * sizeof(float) <= kLdsBytes, "the result tiles fit the ring");

// 64 lanes x 16 (4) bytes from global memory straight into LDS: lane l's bytes land at lds_dst + 16 l (4 l); the lane
// chooses its global address freely.  The instruction takes the LDS address from m0, which is put back afterwards.
// Counted by vmcnt like any load; the compiler does not see these loads, so every wait for them below is written by
// hand (the compiler's own builtin for this instruction makes it wait for vmcnt(0) before every LDS read).
__device__ __forceinline__ void load_lds_x4(const void* g, unsigned int lds_dst) {
  unsigned int keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(g), "s"(lds_dst) : "memory");
}
__device__ __forceinline__ void load_lds_x1(const void* g, unsigned int lds_dst) {
  unsigned int keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(g), "s"(lds_dst) : "memory");
}

// MT accumulator tiles of 32 rows: a block owns 32 MT rows.  SWIGLU: see art_gemm_w4_wide.hip
template <int MT, bool SWIGLU>
__global__ __launch_bounds__(kThreads) void gemm_w4a16_kernel(const _Float16* __restrict__ x, const unsigned char* __restrict__ qweight,
                                                              const _Float16* __restrict__ scales,
                                                              const unsigned char* __restrict__ qzeros, _Float16* y,
                                                              float* __restrict__ partial, int M_total, int K, int N, int splits,
                                                              int col_tiles, int m_blocks, Magic mg,
                                                              const _Float16* residual) {       // residual may be y itself
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = wave & 3, kh = wave >> 2;          // 64-column quarter of the tile, k half of every group

  // block -> (column tile, K split, block of 64 rows).  The row blocks of one (tile, split) stream the same weights:
  // they get block ids that are 8 apart, which the dispatcher places on the same XCD at the same time, so that the
  // weights come from HBM once and from that XCD's L2 for the others.
  const int G = K / GK;
  const int unit = (int)(blockIdx.x / (8 * m_blocks)) * 8 + (int)(blockIdx.x % 8);      // (tile, split) pair
  const int m_block = (int)(blockIdx.x % (8 * m_blocks)) / 8;
  if (unit >= col_tiles * splits) return;
  const int split = unit / col_tiles;
  const TileColumns<SWIGLU> cols{(unit % col_tiles) * (SWIGLU ? BN / 2 : BN), N};
  constexpr int RB = 32 * MT;                       // rows of a block
  constexpr int kLoadsPerGroup = 3 + MT;            // LDS-direct loads per wavefront and group: 2 weights, MT x, 1 scales / zero points
  const int m0 = m_block * RB;
  const int M = M_total - m0 < RB ? M_total - m0 : RB;          // rows of this block
  x += (size_t)m0 * K;
  y += (size_t)m0 * (SWIGLU ? N / 2 : N);
  if (residual) residual += (size_t)m0 * N;
  const int g_begin = (int)((long long)G * split / splits), g_end = (int)((long long)G * (split + 1) / splits);
  const int groups = g_end - g_begin;
  const unsigned int lds0 = (unsigned int)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;

  // ---- what this lane fetches per group: two 16-byte chunks of packed weights, two of x, one dword of scales or
  // zero points.  Wavefront w fills LDS bytes [1024 j, 1024 j + 1024), j = w and w + 8, of the weight and the x area:
  // rows 4 j .. 4 j + 3 of 256 bytes.  Columns past N and rows past M re-read valid memory; nothing of them is stored.
  const unsigned char* wsrc[2];
  const _Float16* xsrc[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = 4 * (wave + 8 * u) + (lane >> 4);
    wsrc[u] = qweight + ((size_t)g_begin * (GK / 2) + r) * N + cols.safe(((lane & 15) ^ (r & 7)) * 16);
    xsrc[u] = x + (size_t)(r < M ? r : M - 1) * K + (size_t)g_begin * GK + ((lane & 15) ^ (r & 15)) * 8;
  }
  const unsigned char* qsrc;
  int qstep;                                        // bytes from one group to the next
  {
    const int d = wave * 64 + lane;                 // dword of the 2 KiB area
    if (d < 128) {                                  // scales of columns 2 d, 2 d + 1
      qsrc = reinterpret_cast<const unsigned char*>(scales + (size_t)g_begin * N + cols.safe(2 * d));
      qstep = 2 * N;
    } else if (d < 160) {                           // zero points of columns 8 (d - 128) .. + 7
      qsrc = qzeros + (size_t)g_begin * (N / 2) + (cols.safe(8 * (d - 128)) >> 1);
      qstep = N / 2;
    } else {                                        // idle lanes re-read the first scales into the padding
      qsrc = reinterpret_cast<const unsigned char*>(scales + (size_t)g_begin * N);
      qstep = 2 * N;
    }
  }
  // batch b (group g_begin + b) goes to stage b % NS: kLoadsPerGroup loads per wavefront
  auto issue = [&](int b) {
    const unsigned int st = lds0 + (unsigned int)(b % NS) * STAGE;
#pragma unroll
    for (int u = 0; u < 2; ++u) load_lds_x4(wsrc[u] + (size_t)b * (GK / 2) * N, st + (wave + 8 * u) * 1024);
#pragma unroll
    for (int u = 0; u < MT; ++u) load_lds_x4(xsrc[u] + (size_t)b * GK, st + W_BYTES + (wave + 8 * u) * 1024);    // 32 rows each
    load_lds_x1(qsrc + (size_t)b * qstep, st + W_BYTES + X_BYTES + wave * 256);
  };

  // ---- operand roles.  A transposing read takes 8 byte-rows x 16 columns per 16 lanes: lane s16 supplies the
  // 8-byte piece (row s16 / 2, half s16 % 2) and receives the 8 bytes of column s16.  Lanes 16-31 of a column tile
  // take the chunk 8 further on, so that the 32 lanes of a pass touch 16 different chunk positions.
  const int s16 = lane & 15, hi16 = (lane >> 4) & 1, h = lane >> 5;
  int b_off[2], colpos[2];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int chunk = cw * 2 + ct + 8 * hi16;       // this lane's 16-column chunk of column tile ct
    b_off[ct] = (kh * 32 + h * 16 + (s16 >> 1)) * 256 + ((chunk ^ (s16 >> 1)) * 16) + (s16 & 1) * 8;
    colpos[ct] = chunk * 16 + s16;                  // the column (within the tile) this lane accumulates
  }
  int a_off[4];                                     // x chunk kh * 8 + h * 4 + e of row lane % 32 (+ 32 per accumulator tile)
#pragma unroll
  for (int e = 0; e < 4; ++e) a_off[e] = W_BYTES + (lane & 31) * 256 + (((kh * 8 + h * 4 + e) ^ s16) * 16);

  f16v acc[MT][2];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][c][r] = 0.f;

  for (int b = 0; b < NS - 1; ++b)
    if (b < groups) issue(b);
#pragma unroll 1
  for (int i = 0; i < groups; ++i) {
    // loads return in order: batch i is complete when at most the batches issued after it are outstanding
    const int later = groups - 1 - i;
    if (later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kLoadsPerGroup) : "memory");
    else if (later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoadsPerGroup) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                   // batch i is in LDS for everybody; everybody has left stage (i - 1) % NS
    asm volatile("" ::: "memory");
    if (i + NS - 1 < groups) issue(i + NS - 1);     // ... which the batch three groups ahead overwrites
    const unsigned char* st = smem + (size_t)(i % NS) * STAGE;
    h2 s2[2], zlo[2], zhi[2];                       // scale, zero point on the two nibble biases, of this lane's two columns
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      const _Float16 sc = *reinterpret_cast<const _Float16*>(st + W_BYTES + X_BYTES + colpos[ct] * 2);
      const unsigned int zb = st[W_BYTES + X_BYTES + 512 + (colpos[ct] >> 1)];
      const _Float16 s = cols.inside(colpos[ct]) ? sc : (_Float16)0.f;
      s2[ct] = h2{s, s};
      const unsigned int z = (zb >> ((colpos[ct] & 1) * 4)) & 15u;
      const unsigned int zz = z | (z << 16);
      zlo[ct] = as_h2(zz | mg.bias_lo);             // 1024 + z
      zhi[ct] = as_h2((zz << 4) | mg.bias_hi);      // 64 + z
    }
    // every LDS operand of the group goes to registers first: 4 transposing reads (q x column tile), 4 MT reads of x
    i32x2 pk[2][2];
    u32x4 ax[4][MT];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) pk[q][ct] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*)(st + b_off[ct] + q * 2048));
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < MT; ++t) ax[e][t] = *reinterpret_cast<const u32x4*>(st + a_off[e] + t * 32 * 256);
    // round e = (q, dword of the 8 bytes): 16 values of k for each lane half; its operands are built while the
    // MFMAs of round e - 1 run
    h8 fa[2][MT], fb[2][2];
    auto build = [&](int e, int slot) {
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const unsigned int w = (unsigned int)pk[e >> 1][ct][e & 1], w8 = w >> 8;
        const h2 p0 = (as_h2(and_or(w, mg.mask_lo, mg.bias_lo)) - zlo[ct]) * s2[ct];      // k0 k4
        const h2 p1 = (as_h2(and_or(w, mg.mask_hi, mg.bias_hi)) - zhi[ct]) * s2[ct];      // k1 k5
        const h2 p2 = (as_h2(and_or(w8, mg.mask_lo, mg.bias_lo)) - zlo[ct]) * s2[ct];     // k2 k6
        const h2 p3 = (as_h2(and_or(w8, mg.mask_hi, mg.bias_hi)) - zhi[ct]) * s2[ct];     // k3 k7
        fb[slot][ct] = h8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) fa[slot][t] = permute_k(ax[e][t]);
    };
    auto multiply = [&](int slot) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
          acc[t][ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[slot][t], fb[slot][ct], acc[t][ct], 0, 0, 0);
    };
    build(0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      multiply(e & 1);
      build(e + 1, (e + 1) & 1);
      // one MFMA (mask 0x008), then a share of the vector work (mask 0x002) of the next round: 26 + 4 MT instructions
#pragma unroll
      for (int m = 0; m < 2 * MT; ++m) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (26 + 4 * MT + 2 * MT - 1) / (2 * MT), 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    multiply(1);
  }

  // ---- the two k halves meet in LDS as [k half][row][column]; then every thread owns four neighbouring columns.
  // Accumulator element r of tile t is row t*32 + (r/4)*8 + (lane/32)*4 + r%4.
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = t * 32 + (r >> 2) * 8 + h * 4 + (r & 3);
        red[((size_t)kh * BM + row) * RLD + colpos[ct]] = acc[t][ct][r];
      }
  __syncthreads();
  if (groups == 0) return;
#pragma unroll 1
  for (int e = tid; e < MT * 32 * (BN / 4); e += kThreads) {
    const int row = e >> 6, c4 = (e & 63) * 4;
    if (row >= M || !cols.inside(c4)) continue;
    const size_t at = (size_t)row * N + cols.at(c4);
    const f32x4 v = *reinterpret_cast<const f32x4*>(red + (size_t)row * RLD + c4) +
                    *reinterpret_cast<const f32x4*>(red + ((size_t)BM + row) * RLD + c4);
    if (SWIGLU && splits == 1) {                    // the gate half of the tile works, with the up half 128 columns further on
      if (c4 >= 128) continue;
      const f32x4 u = *reinterpret_cast<const f32x4*>(red + (size_t)row * RLD + 128 + c4) +
                      *reinterpret_cast<const f32x4*>(red + ((size_t)BM + row) * RLD + 128 + c4);
      *reinterpret_cast<h4*>(y + (size_t)row * (N / 2) + cols.at(c4)) =
          swiglu4(h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]}, h4{(_Float16)u[0], (_Float16)u[1], (_Float16)u[2], (_Float16)u[3]});
    } else if (splits == 1) {
      h4 o = h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
      if (residual) {                               // y = fp16(fp16(product) + residual); may alias y: same elements
        const h4 res = *reinterpret_cast<const h4*>(residual + at);
        o = h4{(_Float16)((float)o[0] + (float)res[0]), (_Float16)((float)o[1] + (float)res[1]),
               (_Float16)((float)o[2] + (float)res[2]), (_Float16)((float)o[3] + (float)res[3])};
      }
      *reinterpret_cast<h4*>(y + at) = o;
    } else {
      *reinterpret_cast<f32x4*>(partial + ((size_t)split * M_total + m0) * N + at) = v;
    }
  }
}

// Four neighbouring sums over the K-splits, in split order: eight splits at a time, all eight loads issued before the
// first is added (a loop of load-then-add runs one memory round trip per split).  Past the last split a load repeats
// split 0 and is not added.
__device__ __forceinline__ f32x4 sum_splits(const float* partial, long long split_stride, int splits) {
  f32x4 t = *reinterpret_cast<const f32x4*>(partial);
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

// y[m,n] = fp16(sum over splits); four columns per thread (N % 4 == 0).
__global__ __launch_bounds__(256) void gemm_w4a16_combine_kernel(const float* __restrict__ partial, _Float16* y,
                                                                  long long count4, long long split_stride, int splits,
                                                                  const _Float16* residual) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= count4) return;
  const f32x4 t = sum_splits(partial + i * 4, split_stride, splits);
  h4 out = h4{(_Float16)t[0], (_Float16)t[1], (_Float16)t[2], (_Float16)t[3]};
  if (residual) {                    // y = fp16(fp16(product) + residual); residual may be y itself
    const h4 res = *reinterpret_cast<const h4*>(residual + i * 4);
    out = h4{(_Float16)((float)out[0] + (float)res[0]), (_Float16)((float)out[1] + (float)res[1]),
             (_Float16)((float)out[2] + (float)res[2]), (_Float16)((float)out[3] + (float)res[3])};
  }
  *reinterpret_cast<h4*>(y + i * 4) = out;
}

// The same for gate | up: y[m, n] of N / 2 columns from the sums of columns n and N / 2 + n.
__global__ __launch_bounds__(256) void gemm_w4a16_combine_swiglu_kernel(const float* __restrict__ partial, _Float16* y, int rows, int N,
                                                                         int splits) {
  const int quads = N / 8;           // groups of four output columns
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)rows * quads) return;
  const long long row = i / quads, col = (i % quads) * 4, stride = (long long)rows * N;
  const f32x4 g = sum_splits(partial + row * N + col, stride, splits), u = sum_splits(partial + row * N + N / 2 + col, stride, splits);
  *reinterpret_cast<h4*>(y + row * (N / 2) + col) = swiglu4(h4{(_Float16)g[0], (_Float16)g[1], (_Float16)g[2], (_Float16)g[3]},
                                                            h4{(_Float16)u[0], (_Float16)u[1], (_Float16)u[2], (_Float16)u[3]});
}

// Number of K-splits: as many blocks as the chip holds at once (one per compute unit), but at least
// two groups per block, no more partial-tile bytes than twice the weight bytes (every split adds an fp32 copy of
// the output to the traffic; 256 rows over 4096 x 4096: 4 splits 23.1 us, the 2 that the weight bytes allow 28.3),
// and no more than the scratch space allows.  The rule lands on the measured
// optimum at M = 64 on MI355X: 8 splits for 4096x4096 and 11008x4096 (two 32-row blocks each), 5 for 4096x11008,
// 2 for 4096x32000.
int choose_splits(int rows, int N, int K, size_t scratch_bytes, int compute_units) {
  const int col_tiles = (N + BN - 1) / BN, G = K / GK;
  int s = (512 / kThreads) * compute_units / col_tiles;      // blocks that are resident at once
  if (s > G / 2) s = G / 2;
  const size_t per_split = (size_t)rows * N * sizeof(float);
  const size_t weight_bytes = (size_t)K * N / 2;
  if ((size_t)s * per_split > 2 * weight_bytes) s = (int)(2 * weight_bytes / per_split);
  const int cap = (int)(scratch_bytes / per_split);
  if (s > cap) s = cap;
  return s < 1 ? 1 : s;
}

// Rows per block of this file's kernel at the library's choice.  32 rows where twice the blocks fill the chip better than
// twice the K-splits do - a block of 32 rows unpacks the same weights for half the matrix instructions, but every K-split
// it saves is an fp32 copy of the output less to write and read back.  Measured at M = 64 and 128 on MI355X: 32-row
// blocks win where one block per compute unit then covers at least four K-splits' worth of (column tile, row block)
// pairs (M = 64: up to 8192 columns, M = 128: 4096), and lose where they would need a second round of blocks; beyond
// 64 rows also where the loop over K is long (128 rows over 11008 x 4096: 27.2 us against 25.8 with 64-row blocks; over
// 4096 x 4096: 17.3 against 19.7).
int choose_block_rows(int M, int K, int N, int compute_units) {
  if (M <= 32) return 32;
  const int col_tiles = (N + BN - 1) / BN;
  return (M <= 64 || (M <= 128 && K <= 8192)) && col_tiles * ((M + 31) / 32) * 4 <= compute_units ? 32 : BM;
}

constexpr int kMaxRowBlocks = 8;                    // row blocks of one launch: they share the weight stream through L2

// ---- What a launch takes, in microseconds, from sweeps of 48 to 1003 rows over eight weight shapes (1024 x 3072 to
// 4096 x 22016 and 11008 x 4096) on MI355X; within 10 % of the measured times above 96 rows.
double split_cost(double rows, double N, int splits) {     // the second launch, and the fp32 tiles at 6 TB/s
  return splits == 1 ? 0.0 : 2.5 + (8.0 * splits + 2.0) * rows * N / 6.0e6;
}
double estimate_narrow(int M, int K, int N, size_t scratch_bytes, int compute_units) {
  const int block_rows = choose_block_rows(M, K, N, compute_units), col_tiles = (N + BN - 1) / BN, G = K / GK;
  double t = 0;
  for (int m0 = 0; m0 < M; m0 += block_rows * kMaxRowBlocks) {
    const int rows = M - m0 < block_rows * kMaxRowBlocks ? M - m0 : block_rows * kMaxRowBlocks;
    const int m_blocks = (rows + block_rows - 1) / block_rows;
    const int splits = choose_splits(rows, N, K, scratch_bytes, compute_units / m_blocks);
    const int rounds = (col_tiles * m_blocks * splits + compute_units - 1) / compute_units;
    t += 5.0 + rounds * ((G + splits - 1) / splits) * (block_rows == BM ? 1.05 : 0.8) + split_cost(rows, N, splits);
  }
  return t;
}
double estimate_wide(int M, int K, int N, int row_tiles, int splits, int compute_units) {
  const int col_tiles = (N + 255) / 256, m_blocks = (M + 32 * row_tiles - 1) / (32 * row_tiles), G = K / GK;
  const double stages = 2 * ((G + splits - 1) / splits), blocks = (double)col_tiles * m_blocks * splits;
  double t = 6.0 + split_cost(M, N, splits);
  if (row_tiles == 8) {             // one block per compute unit; a fuller chip clocks lower
    const int rounds = (int)((blocks + compute_units - 1) / compute_units);
    t += rounds * stages * (1.05 + 0.25 * blocks / ((double)rounds * compute_units));
  } else {                          // two
    const int full = (int)(blocks / (2 * compute_units));
    const double rest = blocks - 2.0 * full * compute_units;
    t += full * stages * 1.62;
    if (rest > compute_units) t += stages * 1.62;
    else if (rest > 0) t += stages * (0.70 + 0.15 * rest / compute_units);
  }
  return t;
}
// Row tiles and K-splits for art_gemm_w4_wide.hip, or 0 where this file's kernel is the better one: blocks of 32 and 64
// rows start sooner and fill the chip at smaller sizes, those of 128 and 256 rows multiply faster (M = 1003 over
// 4096 x 12288: 93 against 156 us, 4096 x 22016: 166 against 248; M = 128 over 4096 x 4096: 21 against 17).
int choose_wide(int M, int K, int N, size_t scratch_bytes, int compute_units, int* splits) {
  if (M <= 64) return 0;
  double best = estimate_narrow(M, K, N, scratch_bytes, compute_units) - 1.5;
  int row_tiles = 0;
  for (int rt = 4; rt <= 8; rt += 4)
    for (int s = 1; s <= 16 && s <= K / (2 * GK); ++s) {
      if (s > 1 && (size_t)s * M * N * sizeof(float) > scratch_bytes) break;
      const double t = estimate_wide(M, K, N, rt, s, compute_units);
      if (t < best) { best = t; row_tiles = rt; *splits = s; }
    }
  return row_tiles;
}

int combine(const float* partial, _Float16* y, int rows, int N, int splits, const _Float16* residual, bool swiglu, hipStream_t stream) {
  if (swiglu) {
    gemm_w4a16_combine_swiglu_kernel<<<dim3((unsigned)(((long long)rows * (N / 8) + 255) / 256)), 256, 0, stream>>>(partial, y, rows, N, splits);
    ART_LAUNCH_CHECK();
    return 0;
  }
  const long long count4 = (long long)rows * N / 4;
  gemm_w4a16_combine_kernel<<<dim3((unsigned)((count4 + 255) / 256)), 256, 0, stream>>>(partial, y, count4, (long long)rows * N, splits, residual);
  ART_LAUNCH_CHECK();
  return 0;
}

int run(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev, void* y_dev, const void* residual_dev,
        int M, int K, int N, int k_splits, bool swiglu, void* stream) {
  const int n_out = swiglu ? N / 2 : N;
  const int want_rows = k_splits >> 8;              // 0: library's choice; else rows of a block / 32
  ART_REQUIRE(k_splits >= 0 && (want_rows <= 2 || want_rows == 4 || want_rows == 8),
              "art_gemm_w4a16: k_splits must be 0 (library's choice) or 1..255, plus 256 x the rows-per-block code 1, 2, 4 or 8 (got %d)", k_splits);
  ART_REQUIRE(((uintptr_t)residual_dev % 8) == 0, "art_gemm_w4a16: the residual must be 8-byte aligned");
  ART_REQUIRE(!art::overlaps(x_dev, (size_t)M * K * 2, y_dev, (size_t)M * n_out * 2), "art_gemm_w4a16: y must not overlap x");
  ART_REQUIRE(x_dev && qweight_dev && scales_dev && qzeros_dev && y_dev, "art_gemm_w4a16: null pointer");
  ART_REQUIRE(M >= 1, "art_gemm_w4a16: M must be positive (got %d)", M);
  ART_REQUIRE(K > 0 && N > 0 && K % 128 == 0 && N % 16 == 0, "art_gemm_w4a16: need K %% 128 == 0 and N %% 16 == 0 (K=%d N=%d)", K, N);
  ART_REQUIRE(((uintptr_t)qweight_dev % 16) == 0 && ((uintptr_t)x_dev % 16) == 0 && ((uintptr_t)qzeros_dev % 8) == 0 &&
                  ((uintptr_t)y_dev % 8) == 0 && ((uintptr_t)scales_dev % 4) == 0,
              "art_gemm_w4a16: x and qweight must be 16-byte aligned, qzeros and y 8-byte aligned, scales 4-byte aligned");
  art::Workspace* wsp = art::workspace((hipStream_t)stream);
  if (!wsp) return 1;
  art::Workspace& ws = *wsp;
  float* scratch = reinterpret_cast<float*>((char*)ws.base + art::kScratchOffset);
  const size_t scratch_bytes = ws.bytes - art::kScratchOffset;
  static int compute_units = 0;
  if (compute_units == 0) {
    int dev = 0;
    ART_HIP(hipGetDevice(&dev));
    ART_HIP(hipDeviceGetAttribute(&compute_units, hipDeviceAttributeMultiprocessorCount, dev));
    for (const auto kernel : {gemm_w4a16_kernel<1, false>, gemm_w4a16_kernel<2, false>, gemm_w4a16_kernel<1, true>, gemm_w4a16_kernel<2, true>})
      ART_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
  }
  hipStream_t st = (hipStream_t)stream;
  const int G = K / GK, col_tiles = tile_count(N, swiglu);
  // Up to kMaxRowBlocks row blocks of this file's kernel go into one launch; longer batches take several passes over the
  // weights.  The caller's choice of kernel and rows per block arrives in the upper bits of k_splits.
  k_splits &= 0xff;
  int row_tiles = want_rows >= 4 ? want_rows : 0, wide_splits = k_splits;
  if (want_rows == 0 && k_splits == 0) row_tiles = choose_wide(M, K, N, scratch_bytes, compute_units, &wide_splits);
  if (row_tiles) {
    const size_t per_split = (size_t)M * N * sizeof(float);
    if (wide_splits > G) wide_splits = G;
    if ((size_t)wide_splits * per_split > scratch_bytes) wide_splits = (int)(scratch_bytes / per_split);
    if (wide_splits < 1) wide_splits = 1;
    if (art::w4::gemm_wide((const _Float16*)x_dev, (const unsigned char*)qweight_dev, (const _Float16*)scales_dev,
                           (const unsigned char*)qzeros_dev, (_Float16*)y_dev, scratch, M, K, N, wide_splits, row_tiles,
                           (const _Float16*)residual_dev, swiglu, st))
      return 1;
    return wide_splits > 1 ? combine(scratch, (_Float16*)y_dev, M, N, wide_splits, (const _Float16*)residual_dev, swiglu, st) : 0;
  }
  const int block_rows = want_rows == 1 ? 32 : want_rows == 2 ? (M <= 32 ? 32 : BM) : choose_block_rows(M, K, N, compute_units);
  for (int m0 = 0; m0 < M; m0 += block_rows * kMaxRowBlocks) {
    const int rows = M - m0 < block_rows * kMaxRowBlocks ? M - m0 : block_rows * kMaxRowBlocks;
    const int m_blocks = (rows + block_rows - 1) / block_rows;
    int splits = choose_splits(rows, N, K, scratch_bytes, compute_units / m_blocks);
    if (k_splits > 0) {           // the caller's choice, within what the kernel and the scratch space take
      const int cap = (int)(scratch_bytes / ((size_t)rows * N * sizeof(float)));
      splits = k_splits > G ? G : k_splits;
      if (splits > cap) splits = cap < 1 ? 1 : cap;
    }
    const _Float16* xs = (const _Float16*)x_dev + (size_t)m0 * K;
    _Float16* ys = (_Float16*)y_dev + (size_t)m0 * n_out;
    const _Float16* rs = residual_dev ? (const _Float16*)residual_dev + (size_t)m0 * N : nullptr;
    const dim3 grid((unsigned)((col_tiles * splits + 7) / 8 * 8 * m_blocks));
    const auto kernel = block_rows == 32 ? (swiglu ? gemm_w4a16_kernel<1, true> : gemm_w4a16_kernel<1, false>)
                                         : (swiglu ? gemm_w4a16_kernel<2, true> : gemm_w4a16_kernel<2, false>);
    kernel<<<grid, kThreads, kLdsBytes, st>>>(xs, (const unsigned char*)qweight_dev, (const _Float16*)scales_dev,
                                              (const unsigned char*)qzeros_dev, ys, scratch, rows, K, N, splits, col_tiles, m_blocks,
                                              kMagic, rs);
    ART_LAUNCH_CHECK();
    if (splits > 1 && combine(scratch, ys, rows, N, splits, rs, swiglu, st)) return 1;
  }
  return 0;
}

}  // namespace

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
  return run(x_dev, qweight_dev, scales_dev, qzeros_dev, y_dev, residual_dev, M, K, N, k_splits, false, stream);
}

extern "C" int art_gemm_w4a16_swiglu(const void* x_dev, const void* qweight_dev, const void* scales_dev, const void* qzeros_dev,
                                     void* y_dev, int M, int K, int N, int k_splits, void* stream) {
  ART_REQUIRE(N % 32 == 0, "art_gemm_w4a16_swiglu: the gate and up halves must be multiples of 16 columns (N=%d)", N);
  return run(x_dev, qweight_dev, scales_dev, qzeros_dev, y_dev, nullptr, M, K, N, k_splits, true, stream);
}
