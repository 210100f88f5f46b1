// Paged causal attention on the 32-bit matrix cores (float32 build only): a kernel for prompt portions
// and one for decoding tokens, called as the bfloat16 build's (attention_mfma.hip) are, with the
// arithmetic of attention_rows (attention.hip), bit for bit:
//   s_p = (chain over the dims, ascending) scale;  m = max;  e_p = expf(s_p - m), 0 where the token does not see p;
//   l = the butterfly of attention_rows over the block's 64 places;  o = chain over the positions, ascending;
//   blocks of 64 positions folded in ascending order; out = O / L.
// A 16x16x4 product of 32-bit operands rounds as four fmaf in ascending k, and a position that a token
// does not see adds 0 times a finite value, which changes nothing.  (Values that are not finite are
// dealt with apart: see `spoiled`.)
//
// Both compute S^T = K Q^T and O^T = V^T P^T.  A lane of a product holds k = 4 i + q of its row for
// step i (q = lane / 16): where the operand comes from memory a lane loads k = 4 q .. 4 q + 3 and four
// lanes exchange (f32_operand); what S^T leaves in a lane, positions 4 q .. 4 q + 3 of one column, becomes
// the B operand of O^T by the same exchange.
#include <math.h>

#include "api.h"
#include "common.h"
#include "instances.h"

#define ATT_BLOCK 64
#define DC_CHUNK 256
#define CMB_MAX_CHUNKS 1024

#if !AXON_BF16

#define F32_STEP(acc, a, b, j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32((a)[j], (b)[j], acc, 0, 0, 0)
#define F32_ZERO (f32x4{0.0f, 0.0f, 0.0f, 0.0f})

// A block's raw scores (tile t, register e: position p0 + 16 t + 4 q + e of the lane's column) to weights;
// m_b and l_b in every lane of the column.
__device__ __forceinline__ void f32_weights(f32x4 (&s)[4], int p0, int lo, int pos, float scale, int q, float& m_b, float& l_b) {
  float m = -INFINITY;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int p = p0 + 16 * t + 4 * q + e;
      s[t][e] = p >= lo && p <= pos ? s[t][e] * scale : -INFINITY;
      m = fmaxf(m, s[t][e]);
    }
  m = fmaxf(m, __shfl_xor(m, 32, AXON_WAVE));
  m = fmaxf(m, __shfl_xor(m, 16, AXON_WAVE));
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int p = p0 + 16 * t + 4 * q + e;
      s[t][e] = p >= lo && p <= pos ? expf(s[t][e] - m) : 0.0f;
    }
  // the butterfly over places 0 .. 63 at distances 32, 16, 8, 4, 2, 1
  float b[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    b[e] = (s[0][e] + s[2][e]) + (s[1][e] + s[3][e]);
    b[e] += __shfl_xor(b[e], 32, AXON_WAVE);
    b[e] += __shfl_xor(b[e], 16, AXON_WAVE);
  }
  m_b = m;
  l_b = (b[0] + b[2]) + (b[1] + b[3]);
}

__device__ __forceinline__ int page_index(int p, int page_size) { return p >> (31 - __builtin_clz(page_size)); }
__device__ __forceinline__ int page_offset(int p, int page_size) { return p & (page_size - 1); }

// ============================================================================ prompt portions
// A block takes 64 or 32 tokens of a tile and one query head and walks their blocks of
// positions; a block's K [64][HD] and V^T [HD][64] go through LDS, rows in the order [16 k][q][i] so that
// a 16-byte read is a lane's operand of four products, rows a multiple of 16 bytes and an odd number
// of them apart (16 rows fall into 16 slots of the 64 banks).  The next block's numbers are asked for
// while this one is multiplied.  A wave has sixteen tokens, or with SHARED two waves have: each scores half of the positions, the
// scores meet in LDS, both work out the weights and each sums half of the dims, so that the tokens that see most, which a prompt waits
// for, take half as long.  grid (pairs of tiles, heads, 4 or 8): which tile of the pair and which part of it.
// Bound by the tokens that see most where all blocks have a place on the chip: a wave's 128 products of 32 cycles a block of positions (head
// size 128) are a third of its time, behind them stand the stage's writes, the exponentials and three barriers; and where blocks
// wait for places by what they stage, which with SHARED is twice as much (launch_attention_f32_prefill).
template <int HD, bool SHARED>
__global__ void __launch_bounds__(256, 2)
attention_f32_prefill_kernel(const float* __restrict__ q, int q_stride, const float* __restrict__ k_cache,
                             const float* __restrict__ v_cache, const int32_t* __restrict__ block_table, int table_stride,
                             const int32_t* __restrict__ positions, const int32_t* __restrict__ seq_rows,
                             float* __restrict__ out, const int32_t* __restrict__ tiles, int n_heads, int n_kv_heads,
                             int page_size, int window, float scale) {
  constexpr int KG = HD / 16, DT = HD / 16, K_LD = HD + 4, V_LD = ATT_BLOCK + 4, LOADS = ATT_BLOCK * HD / 4 / 256;
  constexpr int WAVES = SHARED ? 2 : 1, TOKENS = 64 / WAVES, PT = 4 / WAVES, DH = DT / WAVES;      // of sixteen tokens; a block's; a wave's tiles of positions, of dims
  constexpr int DS = DH < 4 ? DH : 4;                // tiles of dims whose numbers are read together
  extern __shared__ __align__(16) float smem[];      // K [64][K_LD], V^T [HD][V_LD], SHARED: the scores of the waves' tiles [4][2][64][4]
  float* ks = smem;
  float* vs = smem + ATT_BLOCK * K_LD;
  f32x4* scores = reinterpret_cast<f32x4*>(vs + HD * V_LD);
  const int32_t* mine = tiles + 4 * blockIdx.x + 2 * (blockIdx.z / (2 * WAVES));
  const int skip = TOKENS * (blockIdx.z % (2 * WAVES)), count = mine[1] - skip, t0 = mine[0] + skip;
  if (count <= 0) return;                            // the same for the whole block
  const int head = blockIdx.y, kvh = head / (n_heads / n_kv_heads);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g4 = lane >> 4;
  const int group = wave / WAVES, half = SHARED ? __builtin_amdgcn_readfirstlane(wave & 1) : 0, d0 = half * DH;
  const int n = min(count, TOKENS), first_pos = positions[t0], last_pos = positions[t0 + n - 1];
  const bool wave_live = 16 * group < n;
  const int row = t0 + min(16 * group + r16, n - 1), pos = positions[row];
  const int lo = window > 0 ? max(0, pos + 1 - window) : 0;
  const int from = window > 0 ? max(0, first_pos + 1 - window) : 0, upto = window > 0 ? max(0, last_pos + 1 - window) : 0;
  const int32_t* table_row = block_table + (size_t)seq_rows[t0] * table_stride;
  const size_t page_stride = (size_t)n_kv_heads * HD * page_size;
  const float* k_head = k_cache + (size_t)kvh * HD * page_size;
  const float* v_head = v_cache + (size_t)kvh * HD * page_size;

  f32x4 qf[KG];
#pragma unroll
  for (int g = 0; g < KG; ++g)
    qf[g] = f32_operand(*reinterpret_cast<const f32x4*>(q + (size_t)row * q_stride + (size_t)head * HD + 16 * g + 4 * g4));

  // thread: K row tid / 4 + .., four dims; V^T row, four positions.  What no token of the block has
  // written or sees reads a place that one does.
  f32x4 kin[LOADS], vin[LOADS];
  auto fetch = [&](int p0) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int i = tid + 256 * j;
      const int p = min(p0 + i / (HD / 4), last_pos);
      kin[j] = *reinterpret_cast<const f32x4*>(k_head + (size_t)table_row[page_index(p, page_size)] * page_stride +
                                               (size_t)page_offset(p, page_size) * HD + 4 * (i % (HD / 4)));
      const int d = i / 16, pv = min(p0 + 4 * (i % 16), last_pos) & ~3;
      vin[j] = *reinterpret_cast<const f32x4*>(v_head + (size_t)table_row[page_index(pv, page_size)] * page_stride +
                                               (size_t)d * page_size + page_offset(pv, page_size));
    }
  };
  float M = -INFINITY, L = 0.0f;
  f32x4 O[DH];
#pragma unroll
  for (int d = 0; d < DH; ++d) O[d] = F32_ZERO;

  const int b_end = last_pos / ATT_BLOCK;
  fetch(from / ATT_BLOCK * ATT_BLOCK);
  for (int b = from / ATT_BLOCK; b <= b_end; ++b) {
    const int p0 = b * ATT_BLOCK;
    const bool whole = p0 >= upto && p0 + ATT_BLOCK - 1 <= first_pos;      // every token sees every position
    __syncthreads();
    bool odd = false;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int i = tid + 256 * j, c = i % (HD / 4), d = i / 16, c4 = i % 16;
      float* kd = ks + (i / (HD / 4)) * K_LD + 16 * (c / 4) + c % 4;
      float* vd = vs + d * V_LD + 16 * (c4 / 4) + c4 % 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kd[4 * e] = kin[j][e];
        float v = vin[j][e];
        if (!whole) {
          const int p = p0 + 4 * c4 + e;
          v = p >= from && p <= last_pos ? v : 0.0f;
          odd |= !__builtin_isfinite(v);
        }
        vd[4 * e] = v;
      }
    }
    // a value that is not finite, in a block that some tokens see a part of: no products with 0 there
    const bool spoiled = whole ? (__syncthreads(), false) : __syncthreads_or(odd);
    if (b < b_end) fetch(p0 + ATT_BLOCK);
    const bool seen = p0 <= pos && p0 + ATT_BLOCK - 1 >= lo;               // by this lane's token
    const bool works = wave_live && __any(seen);                           // the same for all waves of sixteen tokens

    f32x4 s[4];
    if (works) {
      f32x4 part[PT];
#pragma unroll
      for (int t = 0; t < PT; ++t) part[t] = F32_ZERO;
#pragma unroll
      for (int g = 0; g < KG; ++g) {
        f32x4 a[PT];
#pragma unroll
        for (int t = 0; t < PT; ++t) a[t] = *reinterpret_cast<const f32x4*>(&ks[(16 * PT * half + 16 * t + r16) * K_LD + 16 * g + 4 * g4]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < PT; ++t) F32_STEP(part[t], a[t], qf[g], i);
      }
#pragma unroll
      for (int t = 0; t < PT; ++t) {
        if (SHARED) scores[(2 * wave + t) * 64 + lane] = part[t];
        else s[t] = part[t];
      }
    }
    if (SHARED) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");        // the next block's loads stay under way
    if (!works) continue;
    if (SHARED) {
#pragma unroll
      for (int t = 0; t < 4; ++t) s[t] = scores[(4 * group + t) * 64 + lane];
    }
    float m_b, l_b;
    f32_weights(s, p0, lo, pos, scale, g4, m_b, l_b);
    f32x4 o[DH];
    if (!spoiled) {
      f32x4 pf[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) pf[t] = f32_operand(s[t]);
#pragma unroll
      for (int d = 0; d < DH; ++d) o[d] = F32_ZERO;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int dh = 0; dh < DH; dh += DS) {
          f32x4 a[DS];
#pragma unroll
          for (int d = 0; d < DS; ++d) a[d] = *reinterpret_cast<const f32x4*>(&vs[(16 * (d0 + dh + d) + r16) * V_LD + 16 * t + 4 * g4]);
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int d = 0; d < DS; ++d) F32_STEP(o[dh + d], a[d], pf[t], i);
        }
    } else {
#pragma unroll
      for (int d = 0; d < DH; ++d) o[d] = F32_ZERO;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int place = 16 * t + 4 * g + e;
            const float w = __shfl(s[t][e], r16 + 16 * g, AXON_WAVE);
            if (p0 + place < lo || p0 + place > pos) continue;
#pragma unroll
            for (int d = 0; d < DH; ++d)
#pragma unroll
              for (int r = 0; r < 4; ++r) o[d][r] = fmaf(w, vs[(16 * (d0 + d) + 4 * g4 + r) * V_LD + 16 * t + 4 * e + g], o[d][r]);
          }
    }
    const float mn = fmaxf(M, m_b), alpha = expf(M - mn), wgt = expf(m_b - mn);
    if (seen) {
      L = fmaf(l_b, wgt, L * alpha);
      M = mn;
#pragma unroll
      for (int d = 0; d < DH; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) O[d][r] = fmaf(o[d][r], wgt, O[d][r] * alpha);
    }
  }
  if (16 * group + r16 >= n) return;
  float* orow = out + ((size_t)row * n_heads + head) * HD;
#pragma unroll
  for (int d = 0; d < DH; ++d)
    *reinterpret_cast<f32x4*>(orow + 16 * (d0 + d) + 4 * g4) = f32x4{O[d][0] / L, O[d][1] / L, O[d][2] / L, O[d][3] / L};
}

// ============================================================================ decoding tokens
// One block of 64 positions for the heads of a group; NT: its tiles of 16 positions up to the token's own.
template <int HD, int NT>
__device__ __forceinline__ void f32_decode_block(const float* __restrict__ qrow, const float* __restrict__ k_head,
                                                 const float* __restrict__ v_head, const int32_t* __restrict__ table_row,
                                                 size_t page_stride, int page_size, int p0, int lo, int pos, float scale, int r16,
                                                 int g4, bool head_live, float* __restrict__ dst) {
  constexpr int KG = HD / 16, DT = HD / 16;
  f32x4 kf[NT][KG], vf[NT][DT], qf[KG];
  int k_page[NT], v_page[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    k_page[i] = table_row[page_index(min(p0 + 16 * i + r16, pos), page_size)];
    v_page[i] = table_row[page_index(min(p0 + 16 * i + 4 * g4, pos), page_size)];
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const float* kr = k_head + (size_t)k_page[i] * page_stride + (size_t)page_offset(min(p0 + 16 * i + r16, pos), page_size) * HD;
#pragma unroll
    for (int g = 0; g < KG; ++g) kf[i][g] = *reinterpret_cast<const f32x4*>(kr + 16 * g + 4 * g4);
  }
#pragma unroll
  for (int g = 0; g < KG; ++g) qf[g] = *reinterpret_cast<const f32x4*>(qrow + 16 * g + 4 * g4);
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const float* vr = v_head + (size_t)v_page[i] * page_stride + (page_offset(min(p0 + 16 * i + 4 * g4, pos), page_size) & ~3);
#pragma unroll
    for (int d = 0; d < DT; ++d) vf[i][d] = *reinterpret_cast<const f32x4*>(vr + (size_t)(16 * d + r16) * page_size);
  }

  f32x4 s[4] = {F32_ZERO, F32_ZERO, F32_ZERO, F32_ZERO};
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    const f32x4 qo = f32_operand(qf[g]);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const f32x4 a = f32_operand(kf[i][g]);
#pragma unroll
      for (int j = 0; j < 4; ++j) F32_STEP(s[i], a, qo, j);
    }
  }
  float m_b, l_b;
  f32_weights(s, p0, lo, pos, scale, g4, m_b, l_b);
  // the weight of a position outside the token's range is 0, and so must be what it is multiplied with
  if (p0 < lo || p0 + ATT_BLOCK - 1 > pos) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int p = p0 + 16 * i + 4 * g4 + e;
        const bool live = p >= lo && p <= pos;
#pragma unroll
        for (int d = 0; d < DT; ++d) vf[i][d][e] = live ? vf[i][d][e] : 0.0f;
      }
  }
  f32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = F32_ZERO;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const f32x4 pf = f32_operand(s[i]);
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const f32x4 a = f32_operand(vf[i][d]);
#pragma unroll
      for (int j = 0; j < 4; ++j) F32_STEP(o[d], a, pf, j);
    }
  }
  if (!head_live) return;
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    *reinterpret_cast<float2*>(dst + 16 * d + 4 * g4) = make_float2(o[d][0], o[d][1]);
    *reinterpret_cast<float2*>(dst + 16 * d + 4 * g4 + 2) = make_float2(o[d][2], o[d][3]);
  }
  if (g4 == 0) *reinterpret_cast<float2*>(dst + HD) = make_float2(m_b, l_b);
}

// The same work shared by the four waves of a block: each scores sixteen of the positions, the scores meet in LDS, every wave works
// out the weights from all of them and sums a quarter of the dims.  A wave alone had the pages' 64 KB to wait for, 256 products of 32
// cycles and some thousand lane exchanges one after the other.
template <int HD>
__device__ __forceinline__ void f32_decode_shared(const float* __restrict__ qrow, const float* __restrict__ k_head,
                                                  const float* __restrict__ v_head, const int32_t* __restrict__ table_row,
                                                  size_t page_stride, int page_size, int p0, int lo, int pos, float scale, int r16,
                                                  int g4, int wave, bool head_live, float* __restrict__ dst) {
  constexpr int KG = HD / 16, DH = HD / 64;            // chunks of 16 dims of a key; tiles of 16 dims a wave
  __shared__ __align__(16) f32x4 scores[4][64];
  const int nt = min(4, (pos - p0) / 16 + 1), d0 = wave * DH, lane = r16 + 16 * g4;
  f32x4 kf[KG], vf[4][DH], qf[KG];
  int v_page[4];
  const int kp = min(p0 + 16 * wave + r16, pos), k_page = table_row[page_index(kp, page_size)];
#pragma unroll
  for (int i = 0; i < 4; ++i) v_page[i] = table_row[page_index(min(p0 + 16 * i + 4 * g4, pos), page_size)];
#pragma unroll
  for (int g = 0; g < KG; ++g) qf[g] = *reinterpret_cast<const f32x4*>(qrow + 16 * g + 4 * g4);
  const float* kr = k_head + (size_t)k_page * page_stride + (size_t)page_offset(kp, page_size) * HD;
#pragma unroll
  for (int g = 0; g < KG; ++g) kf[g] = *reinterpret_cast<const f32x4*>(kr + 16 * g + 4 * g4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {                        // (tiles behind the token's own: its last positions again, not used)
    const float* vr = v_head + (size_t)v_page[i] * page_stride + (page_offset(min(p0 + 16 * i + 4 * g4, pos), page_size) & ~3);
#pragma unroll
    for (int d = 0; d < DH; ++d) vf[i][d] = *reinterpret_cast<const f32x4*>(vr + (size_t)(16 * (d0 + d) + r16) * page_size);
  }
  __builtin_amdgcn_sched_barrier(0);
  f32x4 mine = F32_ZERO;
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    const f32x4 qo = f32_operand(qf[g]), a = f32_operand(kf[g]);
#pragma unroll
    for (int j = 0; j < 4; ++j) F32_STEP(mine, a, qo, j);
  }
  scores[wave][lane] = mine;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  f32x4 s[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) s[t] = scores[t][lane];
  float m_b, l_b;
  f32_weights(s, p0, lo, pos, scale, g4, m_b, l_b);
  // the weight of a position outside the token's range is 0, and so must be what it is multiplied with
  if (p0 < lo || p0 + ATT_BLOCK - 1 > pos) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int p = p0 + 16 * i + 4 * g4 + e;
        const bool live = p >= lo && p <= pos;
#pragma unroll
        for (int d = 0; d < DH; ++d) vf[i][d][e] = live ? vf[i][d][e] : 0.0f;
      }
  }
  f32x4 o[DH];
#pragma unroll
  for (int d = 0; d < DH; ++d) o[d] = F32_ZERO;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i >= nt) break;
    const f32x4 pf = f32_operand(s[i]);
#pragma unroll
    for (int d = 0; d < DH; ++d) {
      const f32x4 a = f32_operand(vf[i][d]);
#pragma unroll
      for (int j = 0; j < 4; ++j) F32_STEP(o[d], a, pf, j);
    }
  }
  if (!head_live) return;
#pragma unroll
  for (int d = 0; d < DH; ++d) {
    *reinterpret_cast<float2*>(dst + 16 * (d0 + d) + 4 * g4) = make_float2(o[d][0], o[d][1]);
    *reinterpret_cast<float2*>(dst + 16 * (d0 + d) + 4 * g4 + 2) = make_float2(o[d][2], o[d][3]);
  }
  if (wave == 0 && g4 == 0) *reinterpret_cast<float2*>(dst + HD) = make_float2(m_b, l_b);
}

// One block of 64 positions of a (token, kv head), with the query heads of the group (up to
// 16) as the columns; K and V^T go from the pages straight into registers, all 64 KB asked for at
// once, and (o_b, m_b, l_b) of every head are left in `partial` for the fold (work list and layout as in
// attention_mfma.hip).  BW blocks of positions a block of threads: four of a wave each, or one, which at head size 128 four waves
// share (us with the fold, a wave alone / so: 5 tokens of 16 heads over 2 at 800 positions 15.0 / 12.4, 8 at 2,048 18.3 / 14.5, 9 of 28 over 4
// at 4,000 44.6 / 38.2, 64 at 1,000 58 / 53; 16 of 16 over 16 at 500 37.8 / 33.9, at 5,000 260 / 244; of 64, half as much to wait for: 32 over 32 at 1,500 156 / 181, 16 over 16 at 500 18.7 / 21.3).
// Bound by the wait for the pages: 8 tokens of 16 heads over
// 2 at 777 positions 64 -> 19 us with the fold, at 2,048 144 -> 17.
template <int HD, int BW>
__global__ void __launch_bounds__(BW == 4 || HD == 128 ? 256 : 64, 1)
attention_f32_decode_kernel(const float* __restrict__ q, int q_stride, const float* __restrict__ k_cache,
                            const float* __restrict__ v_cache, const int32_t* __restrict__ block_table, int table_stride,
                            const int32_t* __restrict__ positions, const int32_t* __restrict__ seq_rows,
                            const int32_t* __restrict__ token_index, int n_tokens, const int32_t* __restrict__ work,
                            float* __restrict__ partial, int max_chunks, int n_heads, int n_kv_heads, int page_size,
                            int window, float scale) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g4 = lane >> 4;
  const int sub = BW == 4 ? wave : blockIdx.x & 3, unit = BW == 4 ? blockIdx.x : blockIdx.x >> 2;
  const int item = work[unit / n_kv_heads];
  if (item < 0) return;
  const int slot = item / CMB_MAX_CHUNKS, chunk = item % CMB_MAX_CHUNKS;
  if (slot >= n_tokens || chunk >= max_chunks) return;
  const int t = token_index ? token_index[slot] : slot, kvh = unit % n_kv_heads, group = n_heads / n_kv_heads;
  const int pos = positions[t], lo = window > 0 ? max(0, pos + 1 - window) : 0;
  const int p0 = lo / DC_CHUNK * DC_CHUNK + chunk * DC_CHUNK + sub * ATT_BLOCK;
  if (p0 > pos || p0 + ATT_BLOCK - 1 < lo) return;
  const int32_t* table_row = block_table + (size_t)seq_rows[t] * table_stride;
  const size_t page_stride = (size_t)n_kv_heads * HD * page_size;
  const float* k_head = k_cache + (size_t)kvh * HD * page_size;
  const float* v_head = v_cache + (size_t)kvh * HD * page_size;

  float* dst = partial + (((size_t)slot * n_heads + kvh * group + min(r16, group - 1)) * (max_chunks * (DC_CHUNK / ATT_BLOCK)) +
                          chunk * (DC_CHUNK / ATT_BLOCK) + sub) * (HD + 2);
  const float* qrow = q + (size_t)t * q_stride + (size_t)(kvh * group + min(r16, group - 1)) * HD;
  if constexpr (BW == 1 && HD == 128) {
    if (pos - p0 < 16) {                               // one tile: nothing to share (1 token of 16 heads over 2 at 12 positions, us, shared / so: 7.7 / 7.0)
      if (wave == 0)
        f32_decode_block<HD, 1>(qrow, k_head, v_head, table_row, page_stride, page_size, p0, lo, pos, scale, r16, g4, r16 < group, dst);
      return;
    }
    f32_decode_shared<HD>(qrow, k_head, v_head, table_row, page_stride, page_size, p0, lo, pos, scale, r16, g4, wave, r16 < group, dst);
  } else {
    // A context's last block often holds a few positions: 32 heads over 32, 200 tokens at 10 positions 103 us with all four
    // tiles, 40 with one; 1 token of 16 heads over 2 14 / 9.
    if (pos - p0 < 16)
      f32_decode_block<HD, 1>(qrow, k_head, v_head, table_row, page_stride, page_size, p0, lo, pos, scale, r16, g4, r16 < group, dst);
    else if (pos - p0 < 32)
      f32_decode_block<HD, 2>(qrow, k_head, v_head, table_row, page_stride, page_size, p0, lo, pos, scale, r16, g4, r16 < group, dst);
    else
      f32_decode_block<HD, 4>(qrow, k_head, v_head, table_row, page_stride, page_size, p0, lo, pos, scale, r16, g4, r16 < group, dst);
  }
}

// The fold of a token's blocks in ascending order, thread d dim d.  The factors depend on the maxima
// alone, so they are worked out for HD blocks at once and only the multiply-adds remain a chain.
template <int HD>
__global__ void __launch_bounds__(HD)
attention_f32_combine_kernel(const float* __restrict__ partial, const int32_t* __restrict__ positions,
                             const int32_t* __restrict__ token_index, float* __restrict__ out, int max_chunks, int n_heads,
                             int window) {
  __shared__ float m_of[HD], l_of[HD], alpha_of[HD], weight_of[HD];
  const int t = token_index ? token_index[blockIdx.x] : blockIdx.x, head = blockIdx.y, d = threadIdx.x;
  const int pos = positions[t], lo = window > 0 ? max(0, pos + 1 - window) : 0, first = lo / DC_CHUNK * DC_CHUNK;
  const int b0 = (lo - first) / ATT_BLOCK, b1 = (pos - first) / ATT_BLOCK;
  const float* src = partial + ((size_t)blockIdx.x * n_heads + head) * (max_chunks * (DC_CHUNK / ATT_BLOCK)) * (HD + 2);
  float M = -INFINITY, L = 0.0f, O = 0.0f;
  for (int g0 = b0; g0 <= b1; g0 += HD) {
    const int n = min(HD, b1 - g0 + 1);
    __syncthreads();
    if (d < n) {
      m_of[d] = src[(size_t)(g0 + d) * (HD + 2) + HD];
      l_of[d] = src[(size_t)(g0 + d) * (HD + 2) + HD + 1];
    }
    __syncthreads();
    float before = M;
    for (int i = 0; i < n; ++i) {
      if (i < d) before = fmaxf(before, m_of[i]);
      M = fmaxf(M, m_of[i]);
    }
    if (d < n) {
      const float mn = fmaxf(before, m_of[d]);
      alpha_of[d] = expf(before - mn);
      weight_of[d] = expf(m_of[d] - mn);
    }
    __syncthreads();
    int i = 0;
    for (; i + 15 < n; i += 16) {
      float o[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) o[j] = src[(size_t)(g0 + i + j) * (HD + 2) + d];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        L = fmaf(l_of[i + j], weight_of[i + j], L * alpha_of[i + j]);
        O = fmaf(o[j], weight_of[i + j], O * alpha_of[i + j]);
      }
    }
#pragma unroll 4
    for (; i < n; ++i) {
      L = fmaf(l_of[i], weight_of[i], L * alpha_of[i]);
      O = fmaf(src[(size_t)(g0 + i) * (HD + 2) + d], weight_of[i], O * alpha_of[i]);
    }
  }
  out[((size_t)t * n_heads + head) * HD + d] = O / L;
}

// What attention_f32 takes: the prompt kernel stages pages in fours of positions; the decoding kernel
// has the heads of a group side by side in 16 columns.
int attention_f32_ok(int head_dim, int page_size, int n_heads, int n_kv_heads) {
  return (head_dim == 64 || head_dim == 128) && page_size >= 4 && (page_size & (page_size - 1)) == 0 && n_kv_heads > 0 &&
         n_heads % n_kv_heads == 0 && n_heads / n_kv_heads <= 16;
}

int launch_attention_f32_prefill(const float* q, int q_stride, const float* k_cache, const float* v_cache,
                                 const int32_t* block_table, int table_stride, const int32_t* positions,
                                 const int32_t* seq_rows, float* out, const int32_t* tiles, int n_tiles, int n_heads,
                                 int n_kv_heads, int head_dim, int page_size, int window, float scale, hipStream_t stream) {
  // Two waves for sixteen tokens while the chip has a place for each of their blocks, or nearly: by the most blocks of 64 tokens there can be, a
  // CU's worth and a half at head size 128, where prompts' blocks are unequally long and the long ones go first; one at head size 64, where a block
  // has half the products for the same stages; one and a half of them where a window makes them equally long.  us, 64 tokens a block / 32, of so
  // many blocks of 64: head size 128, 900 tokens of 16 heads (240) 108 / 77, 1,500 (384) 208 / 172, of 28 (672) 265 / 282, 3,000 of 16 (752) 538 / 610,
  // 8,192 of 16 3,786 / 4,732; window 300, 3,000 of 4 (192) 54 / 51, 1,300 of 16 (384) 78 / 89; head size 64, 900 of 16 heads (240) 61 / 50, 500 of
  // 40 (320) 36 / 41, 2,048 of 16 133 / 153, window 300, 1,900 of 4 (120) 29 / 23, 2,300 (144) 29 / 32.
  const long blocks = 4L * n_tiles * n_heads;
  const bool shared = blocks <= (window > 0 ? (head_dim == 128 ? 256 : 128) : (head_dim == 128 ? 384 : 256));
#define LAUNCH(HD, SHARED)                                                                                           \
  {                                                                                                                  \
    constexpr int lds = (ATT_BLOCK * (HD + 4) + HD * (ATT_BLOCK + 4) + (SHARED ? 4 * 2 * 64 * 4 : 0)) * (int)sizeof(float); \
    static bool configured = lds <= 48 * 1024;                                                                       \
    if (!configured) {                                                                                               \
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_f32_prefill_kernel<HD, SHARED>),   \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, lds);                           \
      if (e != hipSuccess) {                                                                                         \
        axk_set_error("attention_prefill: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));           \
        return -2;                                                                                                   \
      }                                                                                                              \
      configured = true;                                                                                             \
    }                                                                                                                \
    AXK_INSTANCE(INST_ATTENTION_F32_PREFILL, HD);                                                                    \
    AXK_INSTANCE(INST_ATTENTION_F32_WAVES, HD, SHARED ? 2 : 1);                                                      \
    attention_f32_prefill_kernel<HD, SHARED><<<dim3(n_tiles, n_heads, SHARED ? 8 : 4), 256, lds, stream>>>(          \
        q, q_stride, k_cache, v_cache, block_table, table_stride, positions, seq_rows, out, tiles, n_heads,          \
        n_kv_heads, page_size, window, scale);                                                                       \
  }
  if (head_dim == 64) { if (shared) LAUNCH(64, true) else LAUNCH(64, false) }
  else { if (shared) LAUNCH(128, true) else LAUNCH(128, false) }
#undef LAUNCH
  AXK_LAUNCH_CHECK("attention_prefill");
  return 0;
}

int launch_attention_f32_decode(const float* q, int q_stride, const float* k_cache, const float* v_cache,
                                const int32_t* block_table, int table_stride, const int32_t* positions,
                                const int32_t* seq_rows, float* out, const int32_t* token_index, int n_tokens,
                                const int32_t* work, int n_work, float* partial, int max_chunks, int n_heads,
                                int n_kv_heads, int head_dim, int page_size, int window, float scale, hipStream_t stream) {
  // A wave a block spreads the loads evenly; where contexts end within their first chunk most of its blocks have nothing to
  // do, and four waves a block are launched faster: 16 heads over 2, 128 tokens at 40 positions 26 / 16 us, 28 over 4, 64 at
  // 30 25 / 16, 64 at 100 26 / 19, 32 over 32, 400 at 100 597 / 475; 28 over 4, 64 at 1,000 62 / 64, 9 at 4,000 48 / 51, 1 at 500 15 / 19.
  const bool single = n_work >= 2 * n_tokens || (long)n_work * n_kv_heads * 4 <= 256;
#define LAUNCH(HD, BW)                                                                                               \
  {                                                                                                                  \
    AXK_INSTANCE(INST_ATTENTION_F32_DECODE, HD, BW);                                                                 \
    attention_f32_decode_kernel<HD, BW><<<(unsigned)n_work * n_kv_heads * (4 / BW), BW == 4 || HD == 128 ? 256 : 64, 0, stream>>>(           \
        q, q_stride, k_cache, v_cache, block_table, table_stride, positions, seq_rows, token_index, n_tokens, work,  \
        partial, max_chunks, n_heads, n_kv_heads, page_size, window, scale);                                         \
    attention_f32_combine_kernel<HD><<<dim3(n_tokens, n_heads), HD, 0, stream>>>(partial, positions, token_index, out, \
                                                                                 max_chunks, n_heads, window);       \
  }
  if (head_dim == 64) { if (single) LAUNCH(64, 1) else LAUNCH(64, 4) }
  else { if (single) LAUNCH(128, 1) else LAUNCH(128, 4) }
#undef LAUNCH
  AXK_LAUNCH_CHECK("attention_decode");
  return 0;
}

#endif  // !AXON_BF16
