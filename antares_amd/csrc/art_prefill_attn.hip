// Causal attention over a whole prompt on the gfx950 matrix cores (fp16 in, fp32 accumulation, fp16 out):
//
//   a[t,h,s] = att_f * sum_m q[t,h,m] k[s,h,m]   for s <= t;   p = softmax_s(a);   out[t,h,m] = sum_s p[t,h,s] v[s,h,m]
//
// i.e. the attention of samples/03_llama_tiny.py:94-99 / samples/05_llama2_7b_int4.py:161-165 for T query positions at
// once, position t attending to cache rows 0..t.  It replaces the two generated contraction kernels (scores, then
// softmax times V) that the reference's tiled schedule would produce for a prompt
// (backends/c-rocm/schedule/standard/algo_tiling.py:35-98).
//
// One block of four wavefronts per (head, tile of 32 queries).  The key tiles 0 .. the block's own are dealt out to the
// wavefronts in turn, each keeps an online softmax of its share, and the four states are merged through LDS at the end:
// nothing is computed above the diagonal, no barrier exists in the loop, and the longest chain of tiles - which bounds the
// launch, 1.0 us a tile with one wavefront per SIMD - is a quarter of the tiles.  With four wavefronts the L2 has to serve the
// key tiles: the blocks of a head run on one XCD, those of the heads past a multiple of eight on all.  One wavefront per query
// tile / four with the blocks of a head wherever they fall / four as here, us: 1003 tokens of 32 heads 50 / 63 / 26, of 31
// heads 49 / 39 / 27; 4000 tokens of 31 heads 456 / 547 / 276, of 71 heads 917 / 1247 / 653; 128 tokens of 32 heads 8.0 / - / 5.2.
// A prompt of one query tile has one key tile: one wavefront, which stores its own outputs (32 tokens: 4.2 us, 4.6 with four).
// Everything is kept transposed so that a lane owns ONE query:
//   * S^T = K Q^T on v_mfma_f32_32x32x16_f16: A = a K tile as it lies in the cache (32 rows of 128 dims, staged in LDS
//     with coalesced 16-byte loads, read back as 16-byte rows), B = the lane's query row from registers.  The 32 x 32
//     result has query lane % 32 in every lane, 16 keys per lane: the running maximum and sum of the online softmax
//     are per-lane scalars, completed with one exchange between lanes l and l ^ 32.
//   * O^T += V^T P^T: the probabilities go from the accumulator layout straight into the B operand (the order of
//     the summed index is free as long as both operands agree), V^T comes out of the row-major V tile through the
//     transposing LDS read ds_read_b64_tr_b16, with the row quadruples chosen to match that order.
//   * key tiles come through buffer descriptors: a lane's eight offsets into a tile never change, and rows past the prompt's end read as
//     zeros.  What bounds a step is its vector instructions, and a comparison and a 64-bit product for each of eight rows were a quarter
//     of their time: 32 heads, 400 tokens 9.6 -> 9.1 us, 1003 24.8 -> 23.2, 4000 256 -> 236; 8 heads 8.1 -> 7.5, 14.0 -> 12.4, 71 -> 65; up to 256
//     tokens 1 to 2 %.  Not kept: 64 queries to a block, which share every key tile but leave one wavefront to a SIMD (1003 tokens 25 -> 37 us);
//     maxima that stay until they have grown by 2^8 (another 4 %, but 3 to 14 % more error: the largest weight is no longer an exact 1);
//   * the rescaling by 2^(m_old - m_new) is one multiplication per accumulator register, skipped where no maximum grew;
//     exponentials are of base 2, log2(e) being folded into the scale; only the diagonal tile is masked.
#include "art_common.h"

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr int D = 128;                 // head dimension
constexpr int QT = 32, KT = 32;        // queries per block, keys per step
constexpr int kMaxWaves = 4;
constexpr int K_LD = D + 8;            // halves per K row in LDS (272 bytes)
constexpr int O_LD = D + 4;            // floats per output row of the merge
constexpr int V_LD = D + 32;           // halves per V row in LDS (320 bytes: the four rows of a transposing read fall on disjoint banks)

__device__ __forceinline__ float max_with_lane_xor_32(float v) {
  const unsigned int u = __builtin_bit_cast(unsigned int, v);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__builtin_bit_cast(float, (unsigned int)r[0]), __builtin_bit_cast(float, (unsigned int)r[1]));
}
__device__ __forceinline__ float sum_with_lane_xor_32(float v) {
  const unsigned int u = __builtin_bit_cast(unsigned int, v);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (unsigned int)r[0]) + __builtin_bit_cast(float, (unsigned int)r[1]);
}

// q: [T, heads, 128]; k, v: rows of kv_stride halves, row s holding [heads, 128]; out: [T, heads, 128]
// FAR: the 32 rows of a key tile take 4 GiB and more.
template <int kWaves, bool FAR>
__global__ __launch_bounds__(64 * kWaves, 2) void prefill_attention_kernel(const _Float16* __restrict__ q, const _Float16* __restrict__ k,
                                                                const _Float16* __restrict__ v, _Float16* __restrict__ out, int T,
                                                                int heads, long long kv_stride, const float* __restrict__ att_f,
                                                                int q_tiles) {
  constexpr int TILE = KT * (K_LD + V_LD);           // halves of a wavefront's K and V tile
  static_assert(TILE * 2 >= QT * O_LD * 4, "a wavefront's outputs take the place of its tiles");
  __shared__ __align__(16) _Float16 tiles[kWaves][TILE];
  __shared__ float s_m[kWaves][QT], s_l[kWaves][QT];
  const int lane = threadIdx.x & 63, half = lane >> 5, qi = lane & 31, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  _Float16* const Ks = tiles[wave];
  _Float16* const Vs = Ks + KT * K_LD;
  // The longest walks (last query tiles) are handed out first, in chunks (grid y, z) of eight query tiles of all heads.
  // Workgroups go to the eight XCDs round robin: in a chunk, the tiles of heads & ~7 heads lie that many blocks apart, a head
  // on one XCD, whose L2 then holds its keys and values; the tiles of the other heads & 7 are dealt to all XCDs, in front.
  const int chunk = blockIdx.y + blockIdx.z * gridDim.y, ranks = q_tiles - 8 * chunk < 8 ? q_tiles - 8 * chunk : 8;
  if (ranks <= 0) return;
  const unsigned whole = heads & ~7, others = heads & 7, dealt = (ranks * others + 7) & ~7u;
  const bool is_dealt = blockIdx.x < dealt;
  const unsigned at = is_dealt ? blockIdx.x : blockIdx.x - dealt, per = is_dealt ? others : whole;
  if (at >= ranks * per) return;
  const int qt = q_tiles - 1 - (8 * chunk + (int)(at / per)), h = (int)((is_dealt ? whole : 0) + at % per);
  const int query = qt * QT + qi;
  const int qrow = query < T ? query : T - 1;                    // rows past T repeat the last one and are never stored
  const float scale = att_f[0] * 1.44269504088896341f;            // scores in units of log2(e)

  // B operand of S^T = K Q^T: query lane % 32, dims 16 s + 8 half .. + 8 of step s
  h8 bq[D / 16];
  {
    const _Float16* qp = q + ((size_t)qrow * heads + h) * D + 8 * half;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) bq[s] = *reinterpret_cast<const h8*>(qp + 16 * s);
  }
  // staging of a K / V tile: 32 rows x 16 chunks of 16 bytes = 8 chunks per lane and matrix
  const int st_row = lane >> 4, st_col = (lane & 15) * 8;      // + 4 rows per i
  u32x4 kreg[8], vreg[8];
  const unsigned row_bytes = (unsigned)kv_stride * 2u, lane_off = (unsigned)st_row * row_bytes + st_col * 2u;
  auto load_tile = [&](int kt) {
    if constexpr (FAR) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = kt * KT + st_row + 4 * i;
        const size_t off = (size_t)(key < T ? key : T - 1) * kv_stride + (size_t)h * D + st_col;
        kreg[i] = *reinterpret_cast<const u32x4*>(k + off);
        vreg[i] = *reinterpret_cast<const u32x4*>(v + off);
      }
    } else {
      // Buffers that end with the head's last row: what lies behind it reads as zeros.
      const int rows = T - kt * KT < KT ? T - kt * KT : KT;
      const size_t from = (size_t)(kt * KT) * kv_stride + (size_t)h * D;
      const unsigned bytes = (unsigned)(rows - 1) * row_bytes + D * 2;
      const auto kb = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(k + from), 0, (int)bytes, art::kBufferFlags);
      const auto vb = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(v + from), 0, (int)bytes, art::kBufferFlags);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        kreg[i] = __builtin_amdgcn_raw_buffer_load_b128(kb, (int)(lane_off + 4u * i * row_bytes), 0, 0);
        vreg[i] = __builtin_amdgcn_raw_buffer_load_b128(vb, (int)(lane_off + 4u * i * row_bytes), 0, 0);
      }
    }
  };
  if (wave <= qt) load_tile(wave);

  float m_run = -INFINITY, l_run = 0.f;
  f16v o[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;

  // per-lane constants of the transposing read of V^T: 16 lanes cover 4 rows x 16 columns
  const int s16 = lane & 15;
  const int tr_row = s16 >> 2, tr_col = ((lane & 31) >> 4) * 16 + (s16 & 3) * 4;

  for (int kt = wave; kt <= qt; kt += kWaves) {
    // registers -> LDS (a wavefront's LDS operations execute in order: the reads of the previous tile are done)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      *reinterpret_cast<u32x4*>(&Ks[(st_row + 4 * i) * K_LD + st_col]) = kreg[i];
      *reinterpret_cast<u32x4*>(&Vs[(st_row + 4 * i) * V_LD + st_col]) = vreg[i];
    }
    if (kt + kWaves <= qt) load_tile(kt + kWaves);                // next tile's loads fly during this tile's arithmetic
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // ---- S^T tile: rows = keys of the tile, columns = queries
    f16v st;
#pragma unroll
    for (int r = 0; r < 16; ++r) st[r] = 0.f;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      const h8 a = *reinterpret_cast<const h8*>(&Ks[qi * K_LD + 16 * s + 8 * half]);      // key row lane % 32
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bq[s], st, 0, 0, 0);
    }
    // element r of the accumulator: key (r / 4) * 8 + 4 * half + r % 4 of the tile, query lane % 32
    float mx = -INFINITY;
    if (kt == qt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kt * KT + (r >> 2) * 8 + 4 * half + (r & 3);
        st[r] = key <= query ? st[r] * scale : -INFINITY;
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) st[r] *= scale;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[r]);
    mx = max_with_lane_xor_32(mx);
    // The maximum may stay -infinity (a tile of infinitely negative scores is all that a wavefront has had so far): its terms
    // are then 2^(-inf - 0) = 0.
    const float m_new = fmaxf(m_run, mx), base = m_new == -INFINITY ? 0.f : m_new;
    if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {       // first tile: 2^(-inf) = 0
      const float alpha = __builtin_amdgcn_exp2f(m_run - base);
      l_run *= alpha;
#pragma unroll
      for (int t = 0; t < D / 32; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
    }
    float lsum = 0.f;
    float p[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      p[r] = __builtin_amdgcn_exp2f(st[r] - base);              // masked: 2^(-inf) = 0
      lsum += p[r];
    }
    l_run += sum_with_lane_xor_32(lsum);
    m_run = m_new;

    // ---- O^T += V^T P^T.  Step j sums over 16 keys; lane half `half` supplies, as elements 0..7, the keys
    // (2j) * 8 + 4 half + 0..3 and (2j + 1) * 8 + 4 half + 0..3 - exactly p[8j .. 8j + 7] - and V^T is read with the same
    // two row quadruples.
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const h8 bp = {(_Float16)p[8 * j], (_Float16)p[8 * j + 1], (_Float16)p[8 * j + 2], (_Float16)p[8 * j + 3],
                     (_Float16)p[8 * j + 4], (_Float16)p[8 * j + 5], (_Float16)p[8 * j + 6], (_Float16)p[8 * j + 7]};
      const int row_lo = 16 * j + 4 * half + tr_row, row_hi = row_lo + 8;
#pragma unroll
      for (int t = 0; t < D / 32; ++t) {
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(&Vs[row_lo * V_LD + t * 32 + tr_col]));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(&Vs[row_hi * V_LD + t * 32 + tr_col]));
        const h4 l4 = __builtin_bit_cast(h4, lo), h4v = __builtin_bit_cast(h4, hi);
        const h8 a = {l4[0], l4[1], l4[2], l4[3], h4v[0], h4v[1], h4v[2], h4v[3]};      // dim t * 32 + lane % 32, eight keys
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bp, o[t], 0, 0, 0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");      // the LDS reads above precede the next tile's writes
    __builtin_amdgcn_wave_barrier();
  }

  typedef float f32x4 __attribute__((ext_vector_type(4)));
  // element r of tile t: dim t * 32 + (r / 4) * 8 + 4 * half + r % 4
  if constexpr (kWaves == 1) {
    if (query >= T) return;
    const float mine = 1.0f / l_run;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<h4*>(out + ((size_t)query * heads + h) * D + t * 32 + g * 8 + 4 * half) =
            h4{(_Float16)(o[t][4 * g] * mine), (_Float16)(o[t][4 * g + 1] * mine), (_Float16)(o[t][4 * g + 2] * mine), (_Float16)(o[t][4 * g + 3] * mine)};
    return;
  }
  // ---- merge: every wavefront scales its outputs to the common maximum and leaves them in LDS, where its tiles were
  if (half == 0) { s_m[wave][qi] = m_run; s_l[wave][qi] = l_run; }
  __syncthreads();
  float m_all = s_m[0][qi], l_all = 0.f;
#pragma unroll
  for (int w = 1; w < kWaves; ++w) m_all = fmaxf(m_all, s_m[w][qi]);
#pragma unroll
  for (int w = 0; w < kWaves; ++w) l_all += s_l[w][qi] * __builtin_amdgcn_exp2f(s_m[w][qi] - m_all);
  const float mine = __builtin_amdgcn_exp2f(m_run - m_all) / l_all;
  float* const O = reinterpret_cast<float*>(tiles[wave]);
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(O + qi * O_LD + t * 32 + g * 8 + 4 * half) =
          f32x4{o[t][4 * g] * mine, o[t][4 * g + 1] * mine, o[t][4 * g + 2] * mine, o[t][4 * g + 3] * mine};
  __syncthreads();
#pragma unroll
  for (int i = 0; i < QT * D / 4 / (64 * kWaves); ++i) {
    const int e = threadIdx.x + i * 64 * kWaves, row = e >> 5, c = (e & 31) * 4;
    if (qt * QT + row >= T) break;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) v += *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(tiles[w]) + row * O_LD + c);
    *reinterpret_cast<h4*>(out + ((size_t)(qt * QT + row) * heads + h) * D + c) = h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
  }
}

}  // namespace

extern "C" int art_prefill_attention(const void* q_dev, const void* k_dev, const void* v_dev, const void* att_f_dev, void* out_dev,
                                     int T, int heads, int head_dim, long long kv_row_stride, void* stream) {
  ART_REQUIRE(q_dev && k_dev && v_dev && att_f_dev && out_dev, "art_prefill_attention: null pointer");
  ART_REQUIRE(head_dim == D, "art_prefill_attention: head_dim must be 128 (got %d)", head_dim);
  ART_REQUIRE(T >= 1 && heads >= 1 && kv_row_stride >= (long long)heads * D, "art_prefill_attention: bad sizes (T=%d heads=%d stride=%lld)",
              T, heads, kv_row_stride);
  ART_REQUIRE(((uintptr_t)q_dev % 16) == 0 && ((uintptr_t)k_dev % 16) == 0 && ((uintptr_t)v_dev % 16) == 0 && ((uintptr_t)out_dev % 8) == 0 &&
                  kv_row_stride % 8 == 0,
              "art_prefill_attention: q, k, v must be 16-byte aligned (row stride a multiple of 8 halves), out 8-byte aligned");
  const int q_tiles = (T + QT - 1) / QT;
  const long long blocks = (long long)q_tiles * heads;
  ART_REQUIRE(blocks <= 0x7fffffffLL, "art_prefill_attention: too many blocks");
  const unsigned chunks = (q_tiles + 7) / 8, rows = chunks < 32768 ? chunks : 32768;
  const unsigned a_chunk = chunks > 1 ? 8 * heads : (q_tiles * (heads & 7) + 7) / 8 * 8 + q_tiles * (heads & ~7);
  // one key tile: one wavefront, and no merge
  const bool far = kv_row_stride >= 1LL << 26;
  const auto kernel = q_tiles == 1 ? (far ? prefill_attention_kernel<1, true> : prefill_attention_kernel<1, false>)
                                   : (far ? prefill_attention_kernel<kMaxWaves, true> : prefill_attention_kernel<kMaxWaves, false>);
  kernel<<<dim3(a_chunk, rows, (chunks + rows - 1) / rows), dim3(q_tiles == 1 ? 64 : 64 * kMaxWaves), 0, (hipStream_t)stream>>>(
      (const _Float16*)q_dev, (const _Float16*)k_dev, (const _Float16*)v_dev, (_Float16*)out_dev, T, heads, kv_row_stride,
      (const float*)att_f_dev, q_tiles);
  ART_LAUNCH_CHECK();
  return 0;
}
