// Attention over a latent cache: every position keeps one normed latent vector c (rank floats'
// worth, shared by all heads) and one rotated key part (rot floats' worth, shared too).  A head's
// unrotated key is Wuk c and its value Wuv c; neither is ever built.  The query's unrotated part
// is carried into the latent space instead (q_lat = Wuk^T q, a per-head product), so that
//     score(i, j) = (q_lat_i . c_j + q_rot_i . k_rot_j) scale,      o_lat_i = sum_j p_ij c_j,
// and the head's output is Wuv o_lat (another per-head product).  A page of the cache holds its
// positions twice: [page_size][rank + rot] rows (the latent and the rotated key part: what scores
// read), then [rank][page_size], the latents again with the positions of one dim side by side
// (what the matrix cores want as the operand of the weighted sum; the same layout as the values of
// the grouped-query attention's pages).  Scores, weights and sums are 32-bit.
#include <type_traits>

#include "api.h"
#include "common.h"
#include "instances.h"

namespace {

// One block per token.  fused [T, stride] float32 holds the down projections' results:
//   [q_at, q_at + q_rank): the query latent -> RMS norm with q_gain -> cq [T, q_rank] (compute dtype);
//   [kv_at, kv_at + rank): the key/value latent -> RMS norm with kv_gain -> the page;
//   [kv_at + rank, + rot): the shared key part -> its first rot_dims dims rotated -> the page; the pairs are
//   (i, i + rot_dims / 2), or (2i, 2i + 1) with `neighbours`, and cos and sin are multiplied by `magnitude`.
// The sums of squares: a strided chain per thread, a butterfly per wave, the four waves in order.
__global__ void __launch_bounds__(256)
latent_prepare_kernel(const float* __restrict__ fused, long stride, int q_at, int q_rank, int kv_at, int rank, int rot,
                      int rot_dims, int neighbours, float magnitude, const void* __restrict__ q_gain, int q_gain_is_f32,
                      const void* __restrict__ kv_gain, int kv_gain_is_f32, float eps, const float* __restrict__ table, const int32_t* __restrict__ positions,
                      const int32_t* __restrict__ seq_rows, const int32_t* __restrict__ block_table, int table_stride,
                      elem_t* __restrict__ cache, int page_size, elem_t* __restrict__ cq, int write_kv) {
  __shared__ float partial[4];
  const int t = blockIdx.x;
  const float* row = fused + (long)t * stride;
  if (q_rank > 0) {
    float ss = 0.0f;
    for (int i = threadIdx.x; i < q_rank; i += 256) ss = fmaf(row[q_at + i], row[q_at + i], ss);
    const float inv = 1.0f / sqrtf(block_sum_256(ss, partial) / (float)q_rank + eps);
    for (int i = threadIdx.x; i < q_rank; i += 256)
      cq[(long)t * q_rank + i] = from_float((row[q_at + i] * inv) * load_vec(q_gain, q_gain_is_f32, i));
    __syncthreads();
  }
  if (!write_kv) return;
  const int pos = positions[t];
  const int page = block_table[(long)seq_rows[t] * table_stride + pos / page_size];
  elem_t* page_base = cache + (long)page * page_size * (2 * rank + rot);
  elem_t* dst = page_base + (long)(pos % page_size) * (rank + rot);
  elem_t* by_dim = page_base + (long)page_size * (rank + rot) + pos % page_size;      // [rank][page_size]
  float ss = 0.0f;
  for (int i = threadIdx.x; i < rank; i += 256) ss = fmaf(row[kv_at + i], row[kv_at + i], ss);
  const float inv = 1.0f / sqrtf(block_sum_256(ss, partial) / (float)rank + eps);
  for (int i = threadIdx.x; i < rank; i += 256) {
    const elem_t v = from_float((row[kv_at + i] * inv) * load_vec(kv_gain, kv_gain_is_f32, i));
    dst[i] = v;
    by_dim[(long)i * page_size] = v;
  }
  const float* kr = row + kv_at + rank;
  const int half = rot_dims / 2;
  const float* tab = table + (long)t * half * 2;
  for (int i = threadIdx.x; i < half; i += 256) {
    const float s = tab[2 * i] * magnitude, c = tab[2 * i + 1] * magnitude;
    const int ia = neighbours ? 2 * i : i, ib = neighbours ? 2 * i + 1 : i + half;
    const float a = kr[ia], b = kr[ib];
    dst[rank + ia] = from_float(__fsub_rn(__fmul_rn(a, c), __fmul_rn(b, s)));
    dst[rank + ib] = from_float(__fadd_rn(__fmul_rn(b, c), __fmul_rn(a, s)));
  }
  for (int i = rot_dims + threadIdx.x; i < rot; i += 256) dst[rank + i] = from_float(kr[i]);
}

// The rotated part of every head's query: q [T, heads, dim + rot] float32 (rows q_stride apart) -> q_full
// [T, heads, rank + rot] float32, places rank .. rank + rot - 1 (the first `rank` are the per-head
// product's).  Pairs and magnitude as in latent_prepare_kernel.
__global__ void latent_query_rope_kernel(const float* __restrict__ q, long q_stride, int dim, int rot, int rot_dims, int neighbours,
                                         float magnitude, const float* __restrict__ table, float* __restrict__ q_full, int rank,
                                         int heads) {
  const int t = blockIdx.x;
  const int half = rot_dims / 2;
  const float* tab = table + (long)t * half * 2;
  for (int idx = threadIdx.x; idx < heads * rot; idx += blockDim.x) {
    const int h = idx / rot, i = idx % rot;
    const float* src = q + (long)t * q_stride + (long)h * (dim + rot) + dim;
    float v = src[i];
    if (i < rot_dims) {
      const bool first = neighbours ? !(i & 1) : i < half;
      const int pair = neighbours ? i >> 1 : (first ? i : i - half);
      const int other = neighbours ? i ^ 1 : (first ? i + half : i - half);
      const float s = tab[2 * pair] * magnitude, c = tab[2 * pair + 1] * magnitude;
      v = first ? __fsub_rn(__fmul_rn(src[i], c), __fmul_rn(src[other], s)) : __fadd_rn(__fmul_rn(src[i], c), __fmul_rn(src[other], s));
    }
    q_full[((long)t * heads + h) * (rank + rot) + rank + i] = v;
  }
}

// One wave per (token, head), four waves a block.  Positions lo ..= pos in blocks of 64 aligned
// to absolute position, ascending; in a block lane j scores position 64 b + j (walking its key
// row against the query in LDS), the block's maximum and sum are butterflies, and the running
// (m, l, o) are rescaled block by block.  For the values lane d owns the latent dims d, d + 64, ...
// and walks the block's positions, taking each weight from its lane.  `sink` (a number a head, or null):
// the sum of the weights also holds exp(sink) once, which has no key and no value: the running
// (m, l) start at (sink, 1).
#define LA_WAVES 4
__global__ void __launch_bounds__(LA_WAVES * 64)
latent_attention_kernel(const float* __restrict__ q_full, const elem_t* __restrict__ cache,
                        const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ positions,
                        const int32_t* __restrict__ seq_rows, float* __restrict__ o_lat, int n_tokens, int heads, int rank,
                        int rot, int page_size, int window, float scale, const float* __restrict__ sink) {
  extern __shared__ float smem[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int width = rank + rot;
  const long page_elems = (long)page_size * (width + rank);
  const long item = (long)blockIdx.x * LA_WAVES + wave;
  const bool active = item < (long)n_tokens * heads;
  const int t = active ? (int)(item / heads) : 0, h = active ? (int)(item % heads) : 0;
  float* qs = smem + (long)wave * width;
  const float* qsrc = q_full + ((long)t * heads + h) * width;
  if (active)
    for (int i = lane; i < width; i += 64) qs[i] = qsrc[i];
  __syncthreads();
  if (!active) return;
  const int pos = positions[t];
  const int lo = window > 0 ? max(0, pos + 1 - window) : 0;
  const int32_t* pages = block_table + (long)seq_rows[t] * table_stride;
  constexpr int MAX_OWN = 16;                      // latent dims a lane owns: rank up to 1024
  float acc[MAX_OWN];
#pragma unroll
  for (int i = 0; i < MAX_OWN; ++i) acc[i] = 0.0f;
  float m = sink ? sink[h] : -INFINITY, l = sink ? 1.0f : 0.0f;
  for (int b = lo / 64; b <= pos / 64; ++b) {
    const int p = b * 64 + lane;
    const bool seen = p >= lo && p <= pos;
    float s = -INFINITY;
    if (seen) {
      const elem_t* key = cache + (long)pages[p / page_size] * page_elems + (long)(p % page_size) * width;
      float dot = 0.0f;
      for (int i = 0; i < width; ++i) dot = fmaf(qs[i], to_float(key[i]), dot);
      s = dot * scale;
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float w = seen ? expf(s - m_new) : 0.0f;
    const float fold = expf(m - m_new);            // 0 at the first block (m = -inf)
    l = fmaf(l, fold, wave_sum(w));
    m = m_new;
#pragma unroll
    for (int i = 0; i < MAX_OWN; ++i) acc[i] *= fold;
    const int j_lo = max(lo, b * 64) - b * 64, j_hi = min(pos, b * 64 + 63) - b * 64;
    for (int j = j_lo; j <= j_hi; ++j) {
      const float wj = __shfl(w, j, 64);
      const int pj = b * 64 + j;
      const elem_t* val = cache + (long)pages[pj / page_size] * page_elems + (long)(pj % page_size) * width;
#pragma unroll
      for (int i = 0; i < MAX_OWN; ++i) {
        const int d = lane + 64 * i;
        if (d < rank) acc[i] = fmaf(wj, to_float(val[d]), acc[i]);
      }
    }
  }
  const float inv = 1.0f / l;
  float* dst = o_lat + ((long)t * heads + h) * rank;
#pragma unroll
  for (int i = 0; i < MAX_OWN; ++i) {
    const int d = lane + 64 * i;
    if (d < rank) dst[d] = acc[i] * inv;
  }
}

#if AXON_BF16
typedef __attribute__((ext_vector_type(8))) __bf16 la_bf16x8;
typedef __attribute__((ext_vector_type(4))) float la_f32x4;
__device__ inline la_bf16x8 la_frag(uint4 v) { return __builtin_bit_cast(la_bf16x8, v); }

// The same attention on the matrix cores.  One wave per (token, sixteen heads), two waves a block,
// each on its own: the sixteen heads of a token see the same positions, so a block of 64 positions is
//   S^T [position, head] = K [position, dims] Q^T           (rank + rot dims in chunks of 32),
//   a maximum, weights and their sum per head (a lane holds 16 positions of its head; the four
//   lanes of a head meet by lane permutation), the running (m, l) and O^T rescaled, then
//   O^T [dim, head] += C^T [dim, position] P^T              (positions in two chunks of 32),
// with K rows and the rows of C^T straight from the page into the first operand (16 or 8 bytes a
// lane) and the rounded weights, as they lie in the accumulators, as the second.  RT: tiles of 16
// latent dims at most; QC: chunks of 32 key dims at most.  Pages hold a multiple of 64 positions.
#define LAM_WAVES 2
#define LAP_TOKENS 8                                  // tokens a block of the kernel for steps of many tokens
// What the kernel for steps of many tokens walks of the tokens first .. last of a tile: up to two runs of neighbours of one
// request, [from0, end0) and [from1, end1).  All of them where the tile holds no more than two requests; else those of
// portions of two tokens or more (decoding rows beside them are left out), unless there are three of these.
struct LatentRuns {
  int from0, end0, from1, end1;
  __device__ __forceinline__ bool hold(int t) const { return (t >= from0 && t < end0) || (t >= from1 && t < end1); }
};
__device__ __forceinline__ LatentRuns latent_runs(const int32_t* __restrict__ seq_rows, int n_tokens, int first, int last) {
  const int n = last + 1 - first, whole = (1 << n) - 1;
  int slot[LAP_TOKENS + 2];                             // of the tile's tokens and their neighbours, all asked for at once
#pragma unroll
  for (int i = 0; i < LAP_TOKENS + 2; ++i) slot[i] = seq_rows[min(max(first + i - 1, 0), n_tokens - 1)];
  int same = 0;                                         // bit i: token i is of the request of the one before
#pragma unroll
  for (int i = 0; i <= LAP_TOKENS; ++i)
    same |= (slot[i] == slot[i + 1] && first + i > 0 && first + i < n_tokens ? 1 : 0) << i;
  const int starts = (~same | 1) & whole, portions = starts & (same | same >> 1);
  auto behind = [&](int i) {                            // where the run that starts at i ends
    const int later = starts & ~((2 << i) - 1);
    return later ? __builtin_ctz(later) : n;
  };
  int a, b;                                             // the runs' first tokens (n: none)
  if (__builtin_popcount(starts) <= 2) {
    a = 0;
    b = behind(0);
  } else if (__builtin_popcount(portions) <= 2) {
    const int second = portions & (portions - 1);
    a = portions ? __builtin_ctz(portions) : n;
    b = second ? __builtin_ctz(second) : n;
  } else {
    a = b = n;
  }
  return LatentRuns{first + a, first + (a < n ? behind(a) : n), first + b, first + (b < n ? behind(b) : n)};
}

template <int RT, int QC, bool SINK>
__global__ void __launch_bounds__(LAM_WAVES * 64)
latent_attention_mfma_kernel(const float* __restrict__ q_full, const bf16_t* __restrict__ cache,
                             const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ positions,
                             const int32_t* __restrict__ seq_rows, float* __restrict__ o_lat, int n_tokens, int heads, int rank,
                             int rot, int page_size, int window, float scale, const float* __restrict__ sink, bool mixed_only) {
  // the sixteen heads' queries as bfloat16 in LDS, rows 16 bytes longer than their chunks so that the
  // sixteen rows a product's operand is read from fall into different banks
  constexpr int QROW = QC * 32 + 8;
  __shared__ __align__(16) bf16_t qs_all[LAM_WAVES][16 * QROW];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int groups = heads / 16;
  // without a window the step's last tokens first: they see the most positions, and the waves that start last
  // should be the short ones; over a window most rows are equally long, and the tokens go in their order
  const long n_items = (long)n_tokens * groups, at = (long)blockIdx.x * LAM_WAVES + wave;
  const long item = window > 0 ? at : n_items - 1 - at;
  bool active = at < n_items;
  const int t = active ? (int)(item / groups) : 0, hg = active ? (int)(item % groups) : 0;
  if (mixed_only && active) {                         // beside the kernel for steps of many tokens: what it leaves
    const int t_first = t / LAP_TOKENS * LAP_TOKENS;
    active = !latent_runs(seq_rows, n_tokens, t_first, min(t_first + LAP_TOKENS, n_tokens) - 1).hold(t);
  }
  const int width = rank + rot, qc = width / 32, rt = rank / 16;
  const int j = lane & 15, g = lane >> 4;
  bf16_t* qs = qs_all[wave];
  if (active) {
    const int per_row = width / 8;
    for (int idx = lane; idx < 16 * per_row; idx += 64) {
      const int row = idx / per_row, part = idx % per_row;
      const float* src = q_full + ((long)t * heads + hg * 16 + row) * width + 8 * part;
      const float4 a = *reinterpret_cast<const float4*>(src), b = *reinterpret_cast<const float4*>(src + 4);
      *reinterpret_cast<uint4*>(qs + row * QROW + 8 * part) =
          make_uint4(pack2_bf16(a.x, a.y), pack2_bf16(a.z, a.w), pack2_bf16(b.x, b.y), pack2_bf16(b.z, b.w));
    }
  }
  __syncthreads();
  if (!active) return;
  const bf16_t* qlane = qs + j * QROW + 8 * g;
  const int pos = positions[t];
  const int lo = window > 0 ? max(0, pos + 1 - window) : 0;
  const int32_t* pages = block_table + (long)seq_rows[t] * table_stride;
  const long page_elems = (long)page_size * (width + rank);
  la_f32x4 acc[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) acc[i] = la_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // a sink is counted once a row (an instance of its own: without a sink the running pair starts from constants)
  float m = SINK ? sink[hg * 16 + j] : -INFINITY, l = SINK ? 1.0f : 0.0f;
  for (int b = lo / 64; b <= pos / 64; ++b) {
    const int p0 = b * 64, in0 = p0 % page_size;
    const bf16_t* page = cache + (long)pages[p0 / page_size] * page_elems;
    const bf16_t* kbase = page + (long)in0 * width + 8 * g;
    const bf16_t* vbase = page + (long)page_size * width + in0 + 4 * g;
    la_f32x4 s[4];
#pragma unroll
    for (int pt = 0; pt < 4; ++pt) {
      s[pt] = la_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      const bf16_t* krow = kbase + (long)(16 * pt + j) * width;
      constexpr int QB = QC < 10 ? QC : 10;         // chunks of a row asked for before the first product waits for any
#pragma unroll
      for (int k0 = 0; k0 < QC; k0 += QB) {
        uint4 kf[QB];
#pragma unroll
        for (int e = 0; e < QB; ++e)
          if (k0 + e < qc) kf[e] = *reinterpret_cast<const uint4*>(krow + 32 * (k0 + e));
#pragma unroll
        for (int e = 0; e < QB; ++e)
          if (k0 + e < qc) s[pt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(la_frag(kf[e]), la_frag(*reinterpret_cast<const uint4*>(qlane + 32 * (k0 + e))), s[pt], 0, 0, 0);
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int pt = 0; pt < 4; ++pt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = p0 + 16 * pt + 4 * g + i;
        const float v = (p >= lo && p <= pos) ? s[pt][i] * scale : -INFINITY;
        s[pt][i] = v;
        mx = fmaxf(mx, v);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float fold = expf(m - m_new);
    float sum = 0.0f;
#pragma unroll
    for (int pt = 0; pt < 4; ++pt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float w = expf(s[pt][i] - m_new);        // 0 where the position is not seen
        s[pt][i] = w;
        sum += w;
      }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    l = fmaf(l, fold, sum);
    m = m_new;
    uint4 pf[2];
#pragma unroll
    for (int c = 0; c < 2; ++c)
      pf[c] = make_uint4(pack2_bf16(s[2 * c][0], s[2 * c][1]), pack2_bf16(s[2 * c][2], s[2 * c][3]),
                         pack2_bf16(s[2 * c + 1][0], s[2 * c + 1][1]), pack2_bf16(s[2 * c + 1][2], s[2 * c + 1][3]));
    constexpr int VB = 4;                         // tiles of 16 dims whose rows are asked for together
#pragma unroll
    for (int d0 = 0; d0 < RT; d0 += VB) {
      uint2 v[VB][4];
#pragma unroll
      for (int e = 0; e < VB; ++e) {
        if (d0 + e < rt) {
          const bf16_t* vrow = vbase + (long)(16 * (d0 + e) + j) * page_size;
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            v[e][2 * c] = *reinterpret_cast<const uint2*>(vrow + 32 * c);
            v[e][2 * c + 1] = *reinterpret_cast<const uint2*>(vrow + 32 * c + 16);
          }
        }
      }
#pragma unroll
      for (int e = 0; e < VB; ++e) {
        if (d0 + e < rt) {
          acc[d0 + e] *= fold;
#pragma unroll
          for (int c = 0; c < 2; ++c)
            acc[d0 + e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                la_frag(make_uint4(v[e][2 * c].x, v[e][2 * c].y, v[e][2 * c + 1].x, v[e][2 * c + 1].y)), la_frag(pf[c]), acc[d0 + e],
                0, 0, 0);
        }
      }
    }
  }
  const float inv = 1.0f / l;
  float* dst = o_lat + ((long)t * heads + hg * 16 + j) * rank + 4 * g;
#pragma unroll
  for (int dt = 0; dt < RT; ++dt)
    if (dt < rt) *reinterpret_cast<float4*>(dst + 16 * dt) = make_float4(acc[dt][0] * inv, acc[dt][1] * inv, acc[dt][2] * inv, acc[dt][3] * inv);
}

// Few tokens (a decoding step): a block of four waves per (token, sixteen heads, block of 64 positions).  Each wave scores sixteen of
// the positions, the scores meet in LDS, every wave works out the same weights from all of them, and each sums a quarter of the
// latent dims; (o, m, l) are left unscaled for the kernel that folds a token's blocks.  All that a wave reads of the page is asked
// for before its first product: such a step is 136 blocks of eight tokens over a window of 1,024, and a wave that had the block to
// itself waited for memory sixteen times one after the other.  The chains, their order and so the bits are those of the kernel
// above.  16 heads, latents of 512 + 64, eight tokens at 200 to 2,500 positions over a window of 1,024: 32.3 -> 12.5 us.  Of a smaller
// latent only what it has is asked for, and by all four waves: 32 heads of 256 + 64, 60 tokens over a window of 1,024, us, the walk / all that the
// instance has room for / here 54 / 70 / 49.5, 16 heads of 208 + 16 28 / 37 / 25.
template <int RT, int QC>
__global__ void __launch_bounds__(256)
latent_attention_blocks_kernel(const float* __restrict__ q_full, const bf16_t* __restrict__ cache,
                               const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ positions,
                               const int32_t* __restrict__ seq_rows, int heads, int rank, int rot, int page_size, int window, float scale,
                               float* __restrict__ partial, int n_chunks) {
  constexpr int QROW = QC * 32 + 8, OWN = RT / 4;
  __shared__ __align__(16) bf16_t qs[16 * QROW];
  __shared__ __align__(16) la_f32x4 scores[4][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, g = lane >> 4;
  const int groups = heads / 16, t = blockIdx.x / groups, hg = blockIdx.x % groups;
  const int pos = positions[t], lo = window > 0 ? max(0, pos + 1 - window) : 0, b = lo / 64 + (int)blockIdx.y;
  float* dst = partial + (((long)t * heads + hg * 16 + j) * n_chunks + blockIdx.y) * (rank + 2);
  if (b > pos / 64) {                                   // no such block: nothing seen
    if (threadIdx.x < 16) { dst[rank] = -INFINITY; dst[rank + 1] = 0.0f; }
    return;
  }
  const int width = rank + rot, qc = width / 32, rt = rank / 16, p0 = b * 64, in0 = p0 % page_size;
  const bf16_t* page = cache + (long)block_table[(long)seq_rows[t] * table_stride + p0 / page_size] * ((long)page_size * (width + rank));
  const bf16_t* krow = page + (long)(in0 + 16 * wave + j) * width + 8 * g;
  const bf16_t* vbase = page + (long)page_size * width + in0 + 4 * g;
  const int per_row = width / 8;                        // of the queries eight numbers a load, up to QC / 4 of these a lane
  float4 qv[(QC + 3) / 4][2];
#pragma unroll
  for (int i = 0; i < (QC + 3) / 4; ++i) {
    const int idx = min((int)threadIdx.x + 256 * i, 16 * per_row - 1);
    const float* src = q_full + ((long)t * heads + hg * 16 + idx / per_row) * width + idx % per_row * 8;
    qv[i][0] = *reinterpret_cast<const float4*>(src);
    qv[i][1] = *reinterpret_cast<const float4*>(src + 4);
  }
  __builtin_amdgcn_sched_barrier(0);
  uint4 kf[QC];                                         // (chunks and tiles that the sizes lack are not asked for: the same for the wave)
#pragma unroll
  for (int c = 0; c < QC; ++c)
    if (c < qc) kf[c] = *reinterpret_cast<const uint4*>(krow + 32 * c);
  uint2 v[OWN][4];
#pragma unroll
  for (int e = 0; e < OWN; ++e) {
    if (4 * e + wave >= rt) continue;                   // a wave has every fourth tile: of a small latent as many as the others
    const bf16_t* vrow = vbase + (long)(16 * (4 * e + wave) + j) * page_size;
#pragma unroll
    for (int c = 0; c < 4; ++c) v[e][c] = *reinterpret_cast<const uint2*>(vrow + 16 * c);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < (QC + 3) / 4; ++i) {
    const int idx = threadIdx.x + 256 * i;
    const float4 x = qv[i][0], y = qv[i][1];
    if (idx < 16 * per_row)
      *reinterpret_cast<uint4*>(qs + idx / per_row * QROW + idx % per_row * 8) =
          make_uint4(pack2_bf16(x.x, x.y), pack2_bf16(x.z, x.w), pack2_bf16(y.x, y.y), pack2_bf16(y.z, y.w));
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");       // the page's loads stay under way
  const bf16_t* qlane = qs + j * QROW + 8 * g;
  la_f32x4 mine = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < QC; ++c)
    if (c < qc) mine = __builtin_amdgcn_mfma_f32_16x16x32_bf16(la_frag(kf[c]), la_frag(*reinterpret_cast<const uint4*>(qlane + 32 * c)), mine, 0, 0, 0);
  scores[wave][lane] = mine;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  float mx = -INFINITY;
  la_f32x4 s[4];
#pragma unroll
  for (int pt = 0; pt < 4; ++pt) {
    s[pt] = scores[pt][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = p0 + 16 * pt + 4 * g + i;
      const float x = (p >= lo && p <= pos) ? s[pt][i] * scale : -INFINITY;
      s[pt][i] = x;
      mx = fmaxf(mx, x);
    }
  }
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  float l = 0.0f;
#pragma unroll
  for (int pt = 0; pt < 4; ++pt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float w = expf(s[pt][i] - mx);              // 0 where the position is not seen
      s[pt][i] = w;
      l += w;
    }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  uint4 pf[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
    pf[c] = make_uint4(pack2_bf16(s[2 * c][0], s[2 * c][1]), pack2_bf16(s[2 * c][2], s[2 * c][3]),
                       pack2_bf16(s[2 * c + 1][0], s[2 * c + 1][1]), pack2_bf16(s[2 * c + 1][2], s[2 * c + 1][3]));
#pragma unroll
  for (int e = 0; e < OWN; ++e) {
    la_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < 2; ++c)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(la_frag(make_uint4(v[e][2 * c].x, v[e][2 * c].y, v[e][2 * c + 1].x, v[e][2 * c + 1].y)),
                                                    la_frag(pf[c]), acc, 0, 0, 0);
    const int dt = 4 * e + wave;
    if (dt < rt) *reinterpret_cast<float2*>(dst + 16 * dt + 4 * g) = make_float2(acc[0], acc[1]),
                 *reinterpret_cast<float2*>(dst + 16 * dt + 4 * g + 2) = make_float2(acc[2], acc[3]);
  }
  if (wave == 0 && g == 0) { dst[rank] = mx; dst[rank + 1] = l; }
}

#define LATENT_PROMPT_KERNEL_FROM 256           // (token, sixteen heads) items of a step from which eight tokens share a block
typedef __attribute__((ext_vector_type(2))) unsigned la_u32x2;
typedef const __attribute__((address_space(1))) void* la_global_t;
typedef __attribute__((address_space(3))) void* la_lds_t;

template <int OFFSET>
__device__ __forceinline__ void la_read8(la_u32x2& dst, unsigned at) {
  asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(at), "n"(OFFSET));
}

// body(0) .. body(N - 1), each with its number as a constant.
template <int N, int I = 0, typename F>
__device__ __forceinline__ void la_for(F&& body) {
  if constexpr (I < N) {
    body(std::integral_constant<int, I>());
    la_for<N, I + 1>(body);
  }
}

// Steps of many tokens: a block takes eight neighbouring tokens (and the same sixteen heads), a wave each, its
// queries in registers.  Where the eight belong to one request (a prompt's portion) a block of 64 positions goes
// through LDS once for all of them, by direct loads: its K rows [64][rank + rot] while the block before is
// summed, its C^T rows [rank][64] while the scores are worked out.  16-byte slots of a staged row are permuted by
// slot ^ (row / 2 % 8), so that the sixteen rows of a read fall into different banks.  Each wave keeps its own
// mask, running pair and accumulators and runs the chain of products of the kernels above: the same bits (sums
// whose maximum stays are not multiplied by 1).  A tile that lies across two requests walks the blocks of one and then
// of the other; what `latent_runs` leaves out is left to a launch of the kernel above (`mixed_only`).  Bound by
// no one unit: at 2,048 tokens over a window of 1,024 (118 us) the matrix cores are busy a fifth of the time, a wave issues in 33 % of
// its cycles, waits for the unit it wants in 35 % (for LDS in 9 %, no bank conflicts; it reads the block's 136 KB for 2,176
// cycles of products) and for loads and barriers in 32 %.
// 16 heads, latents of 512 and 64 rotated dims, 2,048 tokens over a window of 1,024: 638 -> 123 us (four tokens a
// block, stages through registers, queries read from LDS beside the keys); three requests of 701, 523 and 301 tokens
// 232 -> 82, with the tiles across two of them left to the launch behind 260; two portions of 301 tokens at 6,000
// positions 2,280 -> 839.  The launch behind comes after this one, not beside it: 64 decoding rows at 1,000 positions and a
// prompt of 512 tokens 400 -> 335, but with latents of 64 dims 87 -> 92.
template <int RT, int QC, bool EXACT, bool SINK>
__global__ void __launch_bounds__(LAP_TOKENS * 64, 2)
latent_attention_prompt_kernel(const float* __restrict__ q_full, const bf16_t* __restrict__ cache,
                               const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ positions,
                               const int32_t* __restrict__ seq_rows, float* __restrict__ o_lat, int n_tokens, int heads, int rank,
                               int rot, int page_size, int window, float scale, const float* __restrict__ sink) {
  extern __shared__ __align__(256) unsigned char lap_lds[];                       // K [64][width], C^T [rank][64]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int groups = heads / 16, n_tiles = (n_tokens + LAP_TOKENS - 1) / LAP_TOKENS;
  // without a window the step's last tokens first (see above)
  const int at = (int)blockIdx.x / groups, hg = (int)blockIdx.x % groups;
  const int tile = window > 0 ? at : n_tiles - 1 - at;
  if (EXACT) { rank = 16 * RT; rot = 32 * QC - 16 * RT; }
  const int width = rank + rot, qc = width / 32, rt = rank / 16;
  const long page_elems = (long)page_size * (width + rank);
  const int t_first = tile * LAP_TOKENS, t_last = min(t_first + LAP_TOKENS, n_tokens) - 1;
  const LatentRuns runs = latent_runs(seq_rows, n_tokens, t_first, t_last);       // (the same for the whole block)
  const bool active = runs.hold(t_first + wave);
  const int t = min(t_first + wave, t_last), j = lane & 15, g = lane >> 4;
  const int pos = positions[t], lo = window > 0 ? max(0, pos + 1 - window) : 0;
  const int32_t* pages = nullptr;                                  // of the request whose blocks are walked
  // Q^T: a lane's head j, 8 consecutive dims from 32 kc + 8 g, rounded
  u32x4 qf[QC];
  const float* qsrc = q_full + ((long)t * heads + hg * 16 + j) * width + 8 * g;
#pragma unroll
  for (int kc = 0; kc < QC; ++kc)
    if (kc < qc) {
      const float4 a = *reinterpret_cast<const float4*>(qsrc + 32 * kc), b = *reinterpret_cast<const float4*>(qsrc + 32 * kc + 4);
      qf[kc] = u32x4{pack2_bf16(a.x, a.y), pack2_bf16(a.z, a.w), pack2_bf16(b.x, b.y), pack2_bf16(b.z, b.w)};
    }
  la_f32x4 acc[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) acc[i] = la_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m = SINK ? sink[hg * 16 + j] : -INFINITY, l = SINK ? 1.0f : 0.0f;

  // scores of a block (lane: positions p0 + 16 pt + 4 g + i of head j) to weights, the running pair, the operand
  la_f32x4 s[4];
  uint4 pf[2];
  auto weigh = [&](int p0) {
    float mx = -INFINITY;
#pragma unroll
    for (int pt = 0; pt < 4; ++pt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = p0 + 16 * pt + 4 * g + i;
        const float v = (p >= lo && p <= pos) ? s[pt][i] * scale : -INFINITY;
        s[pt][i] = v;
        mx = fmaxf(mx, v);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float fold = expf(m - m_new);
    float sum = 0.0f;
#pragma unroll
    for (int pt = 0; pt < 4; ++pt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float w = expf(s[pt][i] - m_new);        // 0 where the position is not seen
        s[pt][i] = w;
        sum += w;
      }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    l = fmaf(l, fold, sum);
    m = m_new;
#pragma unroll
    for (int c = 0; c < 2; ++c)
      pf[c] = make_uint4(pack2_bf16(s[2 * c][0], s[2 * c][1]), pack2_bf16(s[2 * c][2], s[2 * c][3]),
                         pack2_bf16(s[2 * c + 1][0], s[2 * c + 1][1]), pack2_bf16(s[2 * c + 1][2], s[2 * c + 1][3]));
    if (!__all(fold == 1.0f)) {
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[i] *= fold;
    }
  };

  const int per_row = width / 8, k_mask = per_row % 8 == 0 ? 7 : 3;
  unsigned char* vstage = lap_lds + 128 * width;
  const int first_slot = wave * 64 + lane, step_rows = LAP_TOKENS * 64 / per_row, step_slots = LAP_TOKENS * 64 % per_row;
  const int row0 = first_slot / per_row, slot0 = first_slot % per_row;
  auto ask_k = [&](int b) {
    const int p0 = b * 64;
    const bf16_t* src = cache + (long)pages[p0 / page_size] * page_elems + (long)(p0 % page_size) * width;
    int row = row0, slot = slot0;
    for (int n = wave; n < per_row; n += LAP_TOKENS) {
      __builtin_amdgcn_global_load_lds((la_global_t)(src + row * width + 8 * (slot ^ ((row >> 1) & k_mask))), (la_lds_t)(lap_lds + n * 1024), 16, 0, 0);
      row += step_rows;
      slot += step_slots;
      if (slot >= per_row) { slot -= per_row; ++row; }
    }
  };
  auto ask_v = [&](int b) {
    const int p0 = b * 64;
    const bf16_t* src = cache + (long)pages[p0 / page_size] * page_elems + (long)page_size * width + p0 % page_size +
                        8 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4))) + (long)(lane >> 3) * page_size;
    for (int n = wave; n < rank / 8; n += LAP_TOKENS)
      __builtin_amdgcn_global_load_lds((la_global_t)(src + (long)n * 8 * page_size), (la_lds_t)(vstage + n * 1024), 16, 0, 0);
  };
  const int f = j >> 1;
  const unsigned base = EXACT ? (unsigned)(size_t)(la_lds_t)lap_lds : 0u;       // (reads written as instructions: an LDS address)
  const unsigned k_row = base + j * 2 * width;
  // chunk kc of row j: k_at[kc % 2] + 128 (kc / 2); positions 16 x + 4 g .. + 3 of dim j: v_at[x].  Rows start at multiples
  // of 64 bytes and of 128, so the second address differs from the first by a bit of it.
  const unsigned k_first = k_row + ((k_mask == 7 ? g ^ f : g ^ (f & 3)) << 4);
  const unsigned v_first = base + 128 * width + j * 128 + 8 * (g & 1) + (((g >> 1) ^ f) << 4);
  for (int run = 0; run < 2; ++run) {
    const int u0 = run ? runs.from1 : runs.from0, u1 = (run ? runs.end1 : runs.end0) - 1;
    if (u0 > u1) continue;
    int b_from = 1 << 30, b_to = -1;
    for (int u = u0; u <= u1; ++u) {
      const int p = positions[u];
      b_from = min(b_from, (window > 0 ? max(0, p + 1 - window) : 0) / 64);
      b_to = max(b_to, p / 64);
    }
    pages = block_table + (long)seq_rows[u0] * table_stride;
    const bool walks = t_first + wave >= u0 && t_first + wave <= u1;
    ask_k(b_from);
    for (int b = b_from; b <= b_to; ++b) {
      wait_vmcnt<0>();
      __syncthreads();                                // K of this block is there, C^T of the block before is read
      ask_v(b);
      const bool mine = walks && b >= lo / 64 && b <= pos / 64;
      if (mine) {
#pragma unroll
        for (int pt = 0; pt < 4; ++pt) s[pt] = la_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        unsigned k_base = k_first;
        asm volatile("" : "+v"(k_base));              // (the others are worked out here: no registers of theirs across the loop)
        const unsigned k_at[2] = {k_base, k_mask == 7 ? k_base ^ 64 : k_base + 64};
        if constexpr (EXACT) {
          u32x4 kf[2][2];                             // two of the four tiles of 16 positions, read one pair ahead
          auto read_k = [&](auto u) {
            constexpr int U = decltype(u)::value, KC = U / 2;
            lds_read16<128 * (KC / 2) + 2 * (U & 1) * 1024 * QC>(kf[U & 1][0], k_at[KC & 1]);
            lds_read16<128 * (KC / 2) + (2 * (U & 1) + 1) * 1024 * QC>(kf[U & 1][1], k_at[KC & 1]);
          };
          read_k(std::integral_constant<int, 0>());
          la_for<2 * QC>([&](auto u) {
            constexpr int U = decltype(u)::value;
            if constexpr (U + 1 < 2 * QC) {
              read_k(std::integral_constant<int, U + 1>());
              wait_lgkmcnt<2>();
            } else {
              wait_lgkmcnt<0>();
            }
            use_frags<2>(kf[U & 1]);
#pragma unroll
            for (int e = 0; e < 2; ++e)
              s[2 * (U & 1) + e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(la_bf16x8, kf[U & 1][e]), __builtin_bit_cast(la_bf16x8, qf[U / 2]),
                                                                           s[2 * (U & 1) + e], 0, 0, 0);
          });
        } else {
#pragma unroll
          for (int kc = 0; kc < QC; ++kc)
            if (kc < qc)
#pragma unroll
              for (int pt = 0; pt < 4; ++pt) {
                const uint4 kf = *reinterpret_cast<const uint4*>(lap_lds + k_at[kc & 1] + 128 * (kc / 2) + pt * 32 * width);
                s[pt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(la_frag(kf), __builtin_bit_cast(la_bf16x8, qf[kc]), s[pt], 0, 0, 0);
              }
        }
        weigh(b * 64);
      }
      wait_vmcnt<0>();
      __syncthreads();                                // C^T of this block is there, its K is read
      if (b < b_to) ask_k(b + 1);
      if (mine) {
        unsigned v_base = v_first;
        asm volatile("" : "+v"(v_base));
        const unsigned v_at[4] = {v_base, v_base ^ 32, v_base ^ 64, v_base ^ 96};
        if constexpr (EXACT) {
          la_u32x2 vf[2][4];                          // a tile of 16 dims, read one ahead
          auto read_v = [&](auto d) {
            constexpr int D = decltype(d)::value;
#pragma unroll
            for (int x = 0; x < 4; ++x) la_read8<2048 * D>(vf[D & 1][x], v_at[x]);
          };
          read_v(std::integral_constant<int, 0>());
          la_for<RT>([&](auto d) {
            constexpr int D = decltype(d)::value;
            if constexpr (D + 1 < RT) {
              read_v(std::integral_constant<int, D + 1>());
              wait_lgkmcnt<4>();
            } else {
              wait_lgkmcnt<0>();
            }
#pragma unroll
            for (int x = 0; x < 4; ++x) asm volatile("" : "+v"(vf[D & 1][x]));
#pragma unroll
            for (int c = 0; c < 2; ++c)
              acc[D] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  la_frag(make_uint4(vf[D & 1][2 * c][0], vf[D & 1][2 * c][1], vf[D & 1][2 * c + 1][0], vf[D & 1][2 * c + 1][1])),
                  la_frag(pf[c]), acc[D], 0, 0, 0);
          });
        } else {
#pragma unroll
          for (int d = 0; d < RT; ++d)
            if (d < rt)
#pragma unroll
              for (int c = 0; c < 2; ++c) {
                const uint2 a = *reinterpret_cast<const uint2*>(lap_lds + v_at[2 * c] + 2048 * d);
                const uint2 e = *reinterpret_cast<const uint2*>(lap_lds + v_at[2 * c + 1] + 2048 * d);
                acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(la_frag(make_uint4(a.x, a.y, e.x, e.y)), la_frag(pf[c]), acc[d], 0, 0, 0);
              }
        }
      }
    }
  }
  if (!active) return;
  const float inv = 1.0f / l;
  float* dst = o_lat + ((long)t * heads + hg * 16 + j) * rank + 4 * g;
#pragma unroll
  for (int dt = 0; dt < RT; ++dt)
    if (dt < rt) *reinterpret_cast<float4*>(dst + 16 * dt) = make_float4(acc[dt][0] * inv, acc[dt][1] * inv, acc[dt][2] * inv, acc[dt][3] * inv);
}

// o_lat[row, :] = sum_c exp(m_c - M) o_c / sum_c exp(m_c - M) l_c over a row's blocks in ascending order
// (M the largest m_c; a block that saw nothing has l = 0 and weighs nothing).  One block per (token,
// head): the blocks' (m, l) once into LDS, all loads in flight together, their weights from there, then
// a thread a dim whose chain over the blocks has eight loads in flight.  With a sink, M is at least the
// head's sink and the sum of the weights holds exp(sink - M) as well.
__global__ void __launch_bounds__(512)
latent_attention_fold_kernel(const float* __restrict__ partial, float* __restrict__ o_lat, int rank, int n_chunks,
                             const float* __restrict__ sink, int heads) {
  extern __shared__ float fold_lds[];
  float* weight = fold_lds;
  float* ms = fold_lds + n_chunks;
  float* ls = ms + n_chunks;
  const float* src = partial + (long)blockIdx.x * n_chunks * (rank + 2);
  for (int c = threadIdx.x; c < n_chunks; c += blockDim.x) {
    ms[c] = src[(long)c * (rank + 2) + rank];
    ls[c] = src[(long)c * (rank + 2) + rank + 1];
  }
  __syncthreads();
  float M = sink ? sink[blockIdx.x % heads] : -INFINITY;
  int live = 0;                                         // the rows of blocks behind the last that saw something were not written
  for (int c = 0; c < n_chunks; ++c)
    if (ls[c] > 0.0f) {
      M = fmaxf(M, ms[c]);
      live = c + 1;
    }
  for (int c = threadIdx.x; c < n_chunks; c += blockDim.x) weight[c] = ls[c] > 0.0f ? expf(ms[c] - M) : 0.0f;
  __syncthreads();
  float L = sink ? expf(sink[blockIdx.x % heads] - M) : 0.0f;
  for (int c = 0; c < n_chunks; ++c) L = fmaf(weight[c], ls[c], L);
  const float inv = 1.0f / L;
  for (int d = threadIdx.x; d < rank; d += blockDim.x) {
    float o = 0.0f;
#pragma unroll 8
    for (int c = 0; c < live; ++c) o = fmaf(weight[c], src[(long)c * (rank + 2) + d], o);
    o_lat[(long)blockIdx.x * rank + d] = o * inv;
  }
}

// Steps of many tokens (no blocks side by side): eight tokens a block, their pages staged in LDS once.
#define LATENT_LDS_MOST (160 * 1024)

template <int RT, int QC, bool EXACT>
static int launch_latent_prompt(const float* q_full, const void* cache, const int32_t* block_table, int table_stride,
                                const int32_t* positions, const int32_t* seq_rows, float* o_lat, int n_tokens, int heads, int rank,
                                int rot, int page_size, int window, float scale, const float* sink, hipStream_t stream) {
  const int lds = 128 * (rank + rot) + 128 * rank;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attention_prompt_kernel<RT, QC, EXACT, true>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, LATENT_LDS_MOST);
    if (e == hipSuccess)
      e = hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attention_prompt_kernel<RT, QC, EXACT, false>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, LATENT_LDS_MOST);
    if (e != hipSuccess) {
      axk_set_error("latent_attention: cannot reserve %d bytes of LDS: %s", LATENT_LDS_MOST, hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  const unsigned grid = (unsigned)(((n_tokens + LAP_TOKENS - 1) / LAP_TOKENS) * (heads / 16));
  if (sink) { AXK_INSTANCE(INST_LATENT_PROMPT, RT, QC, EXACT, 1); } else { AXK_INSTANCE(INST_LATENT_PROMPT, RT, QC, EXACT, 0); }
  if (sink)
    latent_attention_prompt_kernel<RT, QC, EXACT, true><<<grid, LAP_TOKENS * 64, lds, stream>>>(
        q_full, (const bf16_t*)cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot, page_size, window,
        scale, sink);
  else
    latent_attention_prompt_kernel<RT, QC, EXACT, false><<<grid, LAP_TOKENS * 64, lds, stream>>>(
        q_full, (const bf16_t*)cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot, page_size, window,
        scale, sink);
  return 0;
}

template <int RT, int QC>
static void launch_latent_mfma(const float* q_full, const void* cache, const int32_t* block_table, int table_stride,
                               const int32_t* positions, const int32_t* seq_rows, float* o_lat, int n_tokens, int heads, int rank,
                               int rot, int page_size, int window, float scale, const float* sink, float* partial, int n_chunks,
                               bool mixed_only, hipStream_t stream) {
  const long items = (long)n_tokens * (heads / 16);
  if (partial) {
    AXK_INSTANCE(INST_LATENT_BLOCKS, RT, QC);
    latent_attention_blocks_kernel<RT, QC><<<dim3((unsigned)items, n_chunks), 256, 0, stream>>>(
        q_full, (const bf16_t*)cache, block_table, table_stride, positions, seq_rows, heads, rank, rot, page_size, window, scale, partial,
        n_chunks);
    latent_attention_fold_kernel<<<n_tokens * heads, min(512, (rank + 63) / 64 * 64), 3 * n_chunks * sizeof(float), stream>>>(
        partial, o_lat, rank, n_chunks, sink, heads);
    return;
  }
  if (sink) { AXK_INSTANCE(INST_LATENT_TOKENS, RT, QC, 1); } else { AXK_INSTANCE(INST_LATENT_TOKENS, RT, QC, 0); }
  const unsigned grid = (unsigned)((items + LAM_WAVES - 1) / LAM_WAVES);
  if (sink)
    latent_attention_mfma_kernel<RT, QC, true><<<grid, LAM_WAVES * 64, 0, stream>>>(
        q_full, (const bf16_t*)cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot, page_size,
        window, scale, sink, mixed_only);
  else
    latent_attention_mfma_kernel<RT, QC, false><<<grid, LAM_WAVES * 64, 0, stream>>>(
        q_full, (const bf16_t*)cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot, page_size,
        window, scale, sink, mixed_only);
}
#endif

}  // namespace

// 1 where axk_latent_attention runs on the matrix cores (the bfloat16 build, heads in sixteens,
// a latent in sixteens up to 512, key rows in chunks of 32 up to 640, pages of a multiple of 64).
extern "C" int axk_latent_attention_uses_mfma(int heads, int rank, int rot, int page_size) {
#if AXON_BF16
  return heads % 16 == 0 && rank % 16 == 0 && (rank + rot) % 32 == 0 && page_size % 64 == 0 && rank <= 512 && rank + rot <= 640;
#else
  return 0;
#endif
}

extern "C" int axk_latent_prepare(const float* fused, long stride, int q_at, int q_rank, int kv_at, int rank, int rot,
                                  int rot_dims, int neighbours, float magnitude, const void* q_gain, int q_gain_is_f32, const void* kv_gain,
                                  int kv_gain_is_f32, float eps, const float* table, const int32_t* positions,
                                  const int32_t* seq_rows, const int32_t* block_table, int table_stride, void* cache,
                                  int page_size, void* cq, int n_tokens, int write_kv, void* stream) {
  AXK_REQUIRE(n_tokens >= 0 && q_rank >= 0 && rank > 0 && rot >= 0 && page_size > 0, "latent_prepare: bad sizes T=%d q_rank=%d "
              "rank=%d rot=%d page=%d", n_tokens, q_rank, rank, rot, page_size);
  AXK_REQUIRE(rot_dims >= 0 && rot_dims <= rot && rot_dims % 2 == 0, "latent_prepare: %d rotated dims of %d", rot_dims, rot);
  AXK_REQUIRE(q_at >= 0 && kv_at >= 0 && q_at + q_rank <= stride && kv_at + rank + rot <= stride,
              "latent_prepare: the parts do not fit rows of %ld", stride);
  if (n_tokens == 0) return 0;
  latent_prepare_kernel<<<n_tokens, 256, 0, (hipStream_t)stream>>>(fused, stride, q_at, q_rank, kv_at, rank, rot, rot_dims,
      neighbours, magnitude, q_gain, q_gain_is_f32, kv_gain, kv_gain_is_f32, eps, table, positions, seq_rows, block_table, table_stride,
      (elem_t*)cache, page_size, (elem_t*)cq, write_kv);
  AXK_LAUNCH_CHECK("latent_prepare");
  return 0;
}

extern "C" int axk_latent_query_rope(const float* q, long q_stride, int dim, int rot, int rot_dims, int neighbours, float magnitude,
                                     const float* table, float* q_full, int rank, int heads, int n_tokens, void* stream) {
  AXK_REQUIRE(q_stride >= (long)heads * (dim + rot), "latent_query_rope: rows %ld apart hold no %d heads of %d", q_stride, heads,
              dim + rot);
  AXK_REQUIRE(n_tokens >= 0 && dim >= 0 && rot >= 0 && rank > 0 && heads > 0 && rot_dims % 2 == 0 && rot_dims <= rot,
              "latent_query_rope: bad sizes T=%d dim=%d rot=%d (%d rotated) rank=%d heads=%d", n_tokens, dim, rot, rot_dims,
              rank, heads);
  if (n_tokens == 0 || rot == 0) return 0;
  latent_query_rope_kernel<<<n_tokens, 256, 0, (hipStream_t)stream>>>(q, q_stride, dim, rot, rot_dims, neighbours, magnitude, table, q_full,
                                                                      rank, heads);
  AXK_LAUNCH_CHECK("latent_query_rope");
  return 0;
}

// Few tokens (a decoding step): a wave per block of 64 positions, so that the blocks of a token run side
// by side; the floats of the workspace this takes (0: the tokens' waves walk their blocks themselves).
// A window of w positions touches at most (w + 62) / 64 + 1 blocks; without a window the caller says how
// many positions the longest row of the step sees (`span`; 0: not known, no blocks side by side).
static int latent_blocks_side_by_side(int window, int span) {
  if (window > 0 && (span <= 0 || span > window)) return (window + 62) / 64 + 1;
  return span > 0 ? (span + 63) / 64 : 0;
}

extern "C" long axk_latent_attention_workspace(int n_tokens, int heads, int rank, int rot, int page_size, int window, int span) {
  if (!axk_latent_attention_uses_mfma(heads, rank, rot, page_size)) return 0;
  const int blocks = latent_blocks_side_by_side(window, span);
  if (blocks < 2 || (long)n_tokens * (heads / 16) >= 512) return 0;
  return (long)n_tokens * heads * blocks * (rank + 2);
}

extern "C" int axk_latent_attention(const float* q_full, const void* cache, const int32_t* block_table, int table_stride,
                                    const int32_t* positions, const int32_t* seq_rows, float* o_lat, int n_tokens, int heads,
                                    int rank, int rot, int page_size, int window, int span, float scale, const float* sink,
                                    float* partial, long partial_floats, void* stream) {
  AXK_REQUIRE(n_tokens >= 0 && heads > 0 && rank > 0 && rot >= 0 && page_size > 0 && window >= 0,
              "latent_attention: bad sizes T=%d heads=%d rank=%d rot=%d page=%d window=%d", n_tokens, heads, rank, rot,
              page_size, window);
  AXK_REQUIRE(rank <= 1024, "latent_attention: a latent of %d dims (at most 1024)", rank);
  AXK_REQUIRE((long)(rank + rot) * LA_WAVES * 4 <= 64 * 1024, "latent_attention: keys of %d dims do not fit LDS", rank + rot);
  if (n_tokens == 0) return 0;
#if AXON_BF16
  if (axk_latent_attention_uses_mfma(heads, rank, rot, page_size) && ((uintptr_t)q_full & 15) == 0 && ((uintptr_t)cache & 15) == 0 &&
      ((uintptr_t)o_lat & 15) == 0) {
    hipStream_t s = (hipStream_t)stream;
    const long need = axk_latent_attention_workspace(n_tokens, heads, rank, rot, page_size, window, span);
    AXK_REQUIRE(partial == nullptr || partial_floats >= need, "latent_attention: a workspace of %ld floats, %ld needed",
                partial_floats, need);
    if (need == 0) partial = nullptr;
    const int n_chunks = latent_blocks_side_by_side(window, span);
    const bool many = partial == nullptr && (long)n_tokens * (heads / 16) >= LATENT_PROMPT_KERNEL_FROM;
    if (many) {
#define LATENT_PROMPT(RT, QC, EXACT)                                                                                                      \
  launch_latent_prompt<RT, QC, EXACT>(q_full, cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot, page_size, \
                               window, scale, sink, s)
      int rc;
      const int rt = rank / 16, qc = (rank + rot) / 32;
      // Latents of a power of two from 64 to 512 beside 32, 64 or 128 rotated dims: every bound known when compiled, so that a
      // block's reads of LDS can be one stretch of instructions (no branch may stand between such a read and its wait).
      // 2,048 tokens of 16 heads, bounds known when launched against here: 512 + 32 283 / 194 us, 512 + 128 299 / 227, 256 +
      // 64 (32 heads) 242 / 162, 256 + 32 197 / 130, 128 + 64 118 / 96, 64 + 64 98 / 83, 64 + 32 85 / 77.
#define LATENT_EXACT(RT, QC) if (rt == RT && qc == QC) rc = LATENT_PROMPT(RT, QC, true); else
      LATENT_EXACT(32, 17) LATENT_EXACT(32, 18) LATENT_EXACT(32, 20)
      LATENT_EXACT(16, 9) LATENT_EXACT(16, 10) LATENT_EXACT(16, 12)
      LATENT_EXACT(8, 5) LATENT_EXACT(8, 6) LATENT_EXACT(8, 8)
      LATENT_EXACT(4, 3) LATENT_EXACT(4, 4) LATENT_EXACT(4, 6)
#undef LATENT_EXACT
      if (rank <= 64 && rank + rot <= 128) rc = LATENT_PROMPT(4, 4, false);
      else if (rank <= 128 && rank + rot <= 256) rc = LATENT_PROMPT(8, 8, false);
      else rc = LATENT_PROMPT(32, 20, false);
#undef LATENT_PROMPT
      if (rc) return rc;
    }
    if (rank <= 64 && rank + rot <= 128)
      launch_latent_mfma<4, 4>(q_full, cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot,
                               page_size, window, scale, sink, partial, n_chunks, many, s);
    else if (rank <= 128 && rank + rot <= 256)
      launch_latent_mfma<8, 8>(q_full, cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot,
                               page_size, window, scale, sink, partial, n_chunks, many, s);
    else
      launch_latent_mfma<32, 20>(q_full, cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot,
                                 page_size, window, scale, sink, partial, n_chunks, many, s);
    AXK_LAUNCH_CHECK("latent_attention");
    return 0;
  }
#endif
  const long items = (long)n_tokens * heads;
  const size_t lds = (size_t)(rank + rot) * LA_WAVES * sizeof(float);
  latent_attention_kernel<<<(unsigned)((items + LA_WAVES - 1) / LA_WAVES), LA_WAVES * 64, lds, (hipStream_t)stream>>>(
      q_full, (const elem_t*)cache, block_table, table_stride, positions, seq_rows, o_lat, n_tokens, heads, rank, rot,
      page_size, window, scale, sink);
  AXK_LAUNCH_CHECK("latent_attention");
  return 0;
}
