// What the int4 GEMM kernels share: operand types, the nibble -> fp16 extraction and the order of k it leaves.
#pragma once
#include "art_common.h"

namespace art {
namespace w4 {

using ::art::Div;
using ::art::make_div;
using ::art::over;

using ::art::buffer_lds_x1;
using ::art::buffer_lds_x4;
using ::art::buffer_of;
using ::art::u32x4_t;

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef h8 h8_by_8 __attribute__((aligned(8)));      // rows that are 8-byte aligned
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) i32x2 lds_i32x2;

struct Magic {
  unsigned int mask, bias;
};

__device__ __forceinline__ h2 as_h2(unsigned int v) { return __builtin_bit_cast(h2, v); }

// (w & mask) | bias in one v_bitop3_b32 (truth table 0xEA = (a & b) | c).
__device__ __forceinline__ unsigned int and_or(unsigned int w, unsigned int mask, unsigned int bias) {
  return __builtin_amdgcn_bitop3_b32(w, mask, bias, 0xEA);
}

constexpr Magic kMagic{0x00F0000Fu, 0x54006400u};

// Byte j of a word holds k = 2 j (low nibble) and 2 j + 1 (high nibble).  Masked and biased as kMagic, the result is fp16 (1024 + the
// first, 64 + the second): the low nibble is the last bits of 1024 + q, the high one those of 64 + q where it lies.  Two of
// four byte permutations are shifts, which issue faster (one card, against a shift and four permutations per word: 1003 rows over
// 4096 x 22016 161.0 -> 158.8 us).
__device__ __forceinline__ unsigned int nibble_pair(unsigned int w, int j) {
  const unsigned int twice = __builtin_amdgcn_perm(w, w, j < 2 ? 0x01000100u : 0x03020302u);      // a half word in both halves
  return j & 1 ? twice >> 8 : twice;
}

// No permutation is left where a transposing read brings every byte in both halves of a word: of the eight rows that it takes, row i is
// twice_row(i) of four, and the words hold rows (0, 1, 0, 1) and (2, 3, 2, 3).  Twice the reads for a sixth less vector work; blocks of 128
// columns take it (art_gemm_w4.hip).  The small blocks wait for their loads either way and spill in one form (16 rows over 4096 x 4096 7.8 -> 8.3 us),
// the wide ones have the permutations in the shadow of their products (0 to 1 %).
__device__ __forceinline__ int twice_row(int i) { return (i & 1) + ((i >> 2) & 1) * 2; }
__device__ __forceinline__ unsigned int nibbles_of_twice(unsigned int w, int j) { return j & 1 ? w >> 8 : w; }

// What becomes of the product: stored (a residual added), SwiGLU of its gate | up halves, or, of q | k | v with heads of
// 128 columns, q and k rotated and all three stored where the attention reads them.
enum Tail { kPlain, kSwiglu, kRope };

// The BN columns of a block: neighbours, or (kSwiglu) BN / 2 of the gate half and the matching ones of the up half.
// N % 16 == 0 (kSwiglu: N % 32), so a piece of 16 columns is inside or outside as a whole.
template <Tail TAIL, int BN>
struct TileColumns {
  int n0, N;
  static constexpr bool SWIGLU = TAIL == kSwiglu;
  __device__ __forceinline__ int at(int pos) const { return SWIGLU && pos >= BN / 2 ? N / 2 + n0 + pos - BN / 2 : n0 + pos; }
  __device__ __forceinline__ bool inside(int pos) const { return SWIGLU ? n0 + (pos & (BN / 2 - 1)) < N / 2 : n0 + pos < N; }
  __device__ __forceinline__ int safe(int pos) const { return inside(pos) ? at(pos) : 0; }
};
inline int tile_count(int N, bool swiglu, int bn) { return swiglu ? (N / 2 + bn / 2 - 1) / (bn / 2) : (N + bn - 1) / bn; }

// Rows of memory that a block fetches one after another, `step` bytes apart: a descriptor and the offset of the next.  Behind the last
// row it stays there: that one is fetched again, into slots that nobody reads, and the loop needs neither branches nor a varying
// count of loads.  Offsets are 32 bits; FAR, for more than that: wherever one has passed 2 GiB, the descriptor moves on (rebase; in
// every kernel it would cost 2 to 3 %).  A step is at most 2 GiB (67108864 columns of a stage of the wide kernel) and far() is asked
// behind every next(): an offset of less than 2 GiB and a step stay below 4 GiB, two steps need not.
template <bool FAR> struct Rows {
  u32x4_t buffer;
  unsigned int at, step, last;
  unsigned long long end;                           // FAR: from the descriptor's base to the last row
  __device__ __forceinline__ Rows(const void* base, unsigned int bytes, int count) : buffer(buffer_of(base)), at(0), step(bytes), last(bytes * (count - 1)) {
    if constexpr (FAR) {
      end = (unsigned long long)bytes * (unsigned int)(count - 1);
      set_last();
    }
  }
  __device__ __forceinline__ void set_last() { last = end > 0xffffffffull ? 0xffffffffu : (unsigned int)end; }
  __device__ __forceinline__ void next() { at = at + step < last ? at + step : last; }
  __device__ __forceinline__ bool far() const { return FAR && (int)at < 0; }
  __device__ __forceinline__ void rebase() {
    const unsigned long long base = ((unsigned long long)buffer[1] << 32 | buffer[0]) + at;
    buffer[0] = (unsigned int)base;
    buffer[1] = (unsigned int)(base >> 32);
    end -= at;
    at = 0;
    set_last();
  }
};

// The M x N sums of a K split on their way to the pass that adds them: a buffer of exactly that many bytes, so that what is stored to
// rows past M is dropped on the way out, without a comparison and a branch for each store.  Offsets are 32 bits: 4 N times the rows of
// all blocks is at most 4 GiB, or what is past M comes round to the first rows.
struct PartialTile {
  __amdgpu_buffer_rsrc_t buffer;
  unsigned int row;                                 // bytes
  __device__ __forceinline__ PartialTile(float* partial, int split, int M, int N)
      : buffer(__builtin_amdgcn_make_buffer_rsrc(partial + (size_t)split * M * N, 0, M * N * 4, art::kBufferFlags)), row(4u * N) {}
  __device__ __forceinline__ unsigned int at(int m, int n) const { return m * row + 4u * n; }
  __device__ __forceinline__ void store(unsigned int at, int rows_on, float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), buffer, (int)(at + rows_on * row), 0, 0);
  }
};

// kRope: sine and cosine of row m, column j < 64 of a head at angles[64 m + j]; row m of q, k and v holds `heads` heads of 128.
struct Rope {
  const float2* angles;
  _Float16 *q, *k, *v;
  int heads;
  // where head h of q | k | v has its first row, and whether it is rotated
  __device__ __forceinline__ _Float16* at(int h) const {
    return h < heads ? q + h * 128 : h < 2 * heads ? k + (h - heads) * 128 : v + (h - 2 * heads) * 128;
  }
  __device__ __forceinline__ bool rotated(int h) const { return h < 2 * heads; }
};
// Neighbouring columns of the first half of a head and their partners 64 further on, with their angles (sine, cosine).
template <int COUNT> struct Angles {
  f32x4 of[COUNT / 2];
};
template <int COUNT> __device__ __forceinline__ Angles<COUNT> load_angles(const float2* from) {
  Angles<COUNT> a;
#pragma unroll
  for (int k = 0; k < COUNT / 2; ++k) a.of[k] = reinterpret_cast<const f32x4*>(from)[k];
  return a;
}
template <int COUNT, class V> __device__ __forceinline__ void rotate(V& a, V& b, const Angles<COUNT>& angles) {
#pragma unroll
  for (int k = 0; k < COUNT; ++k) {
    const float sine = angles.of[k >> 1][2 * (k & 1)], cosine = angles.of[k >> 1][2 * (k & 1) + 1];
    const float x = (float)a[k], y = (float)b[k];
    a[k] = (_Float16)(x * cosine - y * sine);
    b[k] = (_Float16)(y * cosine + x * sine);
  }
}

// How units - (column tile, K split) pairs - x blocks of rows are dealt out.  A launch is a grid of 8 m_blocks x ceil(units / 8)
// blocks, and block b runs on XCD b % 8: the row blocks of a unit, which stream the same weights, go to one XCD at the same time,
// so that the weights come from HBM once and from that XCD's L2 for the others.  So do neighbouring tiles (units are numbered by tile, then
// by split, and an XCD has a run of them): pieces of 64 columns of the gate and of the up half are half a line of memory, which two XCDs
// would fetch both.  Dealt in turn instead, us: 16 rows of gate | up 4096 x 22016 23.7, now 19.7, 50 rows 25.3 and 22.9, 128 rows 34.4 and 32.5;
// blocks whose pieces are whole lines 1 % either way.  Numbered by split, then by tile, an XCD's blocks ask for the same lines of x at
// once: 12 to 19 % slower with K-splits.  The last units % 8 units are dealt to all XCDs by
// their row blocks: else some XCDs have a unit more than others, and 264 blocks on 256 compute units take as long as 512
// (87 rows over 4352 x 10816 30.4 -> 19.8 us, 842 over 3840 x 4176 54.5 -> 33.8).
struct Deal {
  int whole, m_blocks;                              // units / 8
  int left, each;                                   // row blocks of the last units % 8 units, and how many of them an XCD has
  // false: nothing to do
  __device__ __forceinline__ bool take(int& unit, int& m_block) const {
    const int xcd = blockIdx.x & 7, i = blockIdx.x >> 3;
    unit = xcd * whole + blockIdx.y;
    m_block = i;
    if ((int)blockIdx.y < whole) return true;
    unit = whole * 8;
    m_block = xcd * each + i;
    const bool some = i < each && m_block < left;
    while (m_block >= m_blocks) { m_block -= m_blocks; ++unit; }      // at most seven times
    return some;
  }
};
inline Deal deal(int units, int m_blocks, dim3& grid) {
  grid = dim3(8 * m_blocks, (units + 7) / 8);
  const int left = units % 8 * m_blocks;
  return Deal{units / 8, m_blocks, left, (left + 7) / 8};
}

// Whether the pass that adds K-splits takes each row by eighths, on the XCDs that wrote them, and art_gemm_w4_deep.hip numbers its units by
// column tile for that; else whole rows in order, and units by split: an XCD then reads one split's part of x, not all of them.  By eighths
// from 2560 columns on, and below where an eighth of a row's sums (pieces of 16 bytes, two of them where a gate and its up
// projection or the two halves of a head meet) is whole lines of memory: else two XCDs fetch the lines between.  Against rows dealt whole, in the mean over 4 to
// 1000 rows and K of 2048 to 11008 (weights in the cache): 16 to 208 columns 0.87 to 0.95 times as fast (400 rows of 11008 over 64 columns 9.4 us, whole 7.2),
// 256 1.07, 384 0.99, 512 1.04, 640 0.99, 1024 1.07, 1152 0.98, 1536 1.03, 2320 0.98, 2768 1.01, 3024 1.02, 4096 1.03, 5520 1.03; gate | up of 320 columns 0.89, 512 1.01,
// 768 0.97, 1024 1.04, 1088 0.98, 2048 1.04, 4128 1.01, 4992 1.02; q | k | v of one head 0.92, 3 0.98, 4 1.02, 6 0.99, 8 1.01, 9 1.01, 11 1.03.
inline bool by_eighths(int N, Tail tail) { return N >= 2560 || (tail == kPlain ? N / 4 : N / 8) % 64 == 0; }

// fp16(silu(gate) * up) of fp16 operands in fp32.  silu is half as many instructions as expf and a division (every fp16 gate gives
// the same fp16 value): 1003 rows over 4096 x 22016 with SWIGLU 186.4 -> 184.1 us.
__device__ __forceinline__ h4 swiglu4(h4 g, h4 u) {
  h4 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = (_Float16)(silu((float)g[k]) * (float)u[k]);
  return o;
}

// Large batches (art_gemm_w4_wide.hip): one launch over blocks of 32 row_tiles rows x 256 columns, K cut into `splits`;
// with splits > 1 the fp32 tiles go to `partial` [splits][M][N].  row_tiles is 4 or 8; far (the packed weights of a split are 4 GiB and
// more): 4.  No residual but with kPlain.
int gemm_wide(const _Float16* x, const unsigned char* qweight, const _Float16* scales, const unsigned char* qzeros, _Float16* y,
              float* partial, int M, int K, int N, int splits, int row_tiles, bool far, const _Float16* residual, Tail tail, const Rope& rope, hipStream_t stream);

// Small products (art_gemm_w4_deep.hip): one launch over blocks of 32 row_tiles rows (1 or 2; 16 where there are no more) and 32 col_tiles columns (1, or
// 2 with one row tile).
// Partial sums as above; tiles x splits below 2^16, the packed weights of a split below 4 GiB.
inline int deep_tiles(int N, Tail tail, int col_tiles) { return tail == kPlain ? (N + 32 * col_tiles - 1) / (32 * col_tiles) : (N / 2 + 16 * col_tiles - 1) / (16 * col_tiles); }
int gemm_deep(const _Float16* x, const unsigned char* qweight, const _Float16* scales, const unsigned char* qzeros, _Float16* y,
              float* partial, int M, int K, int N, int splits, int row_tiles, int col_tiles, const _Float16* residual, Tail tail, const Rope& rope, hipStream_t stream);

}  // namespace w4
}  // namespace art
