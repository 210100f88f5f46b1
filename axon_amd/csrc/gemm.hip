// Matrix products out = X [M, K] . W [N, K]^T with a bias / residual epilogue.
//
// The rule every variant keeps: the K-reduction of one output element is one order of additions in
// ascending k that does not depend on M, on the tile shape or on what else is in the batch
// (the reference states the rule for its own kernels: src/cuda/decode.cu:352-369,
// src/cuda/prefill.cu:6-16).  Rows only ride along.
//
// gemm_fma: any M, N, K and strides, 32-bit multiply-adds, a chain per output and 32 k, whose sums are
// added in ascending order (a third of the rounding of one chain over all k): the float32 build's
// product (true 32-bit), and the bfloat16 build's fallback for shapes the MFMA kernels refuse.
// The chains run on the 32-bit matrix cores: a 16x16x4 product of 32-bit operands gives, bit for bit,
// what four fmaf in ascending k give (measured over random operands, denormals among them), at
// twice the rate that the vector unit has without its packed instructions.
#include "api.h"
#include "buffer.h"
#include "common.h"
#include "instances.h"

#define FMA_PART 32    // k of one chain

#define FMA_STEP(acc, a, b, j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32((a)[j], (b)[j], acc, 0, 0, 0)

// Four k of a row from `k` on; what lies behind K reads other numbers of the row here (VEC: K is a multiple of four,
// one 16-byte load; a branch round it would have the compiler wait for every load under way) and is cleared
// when it is used.  Rows that do not exist read a row that does: their outputs are not stored.
template <bool VEC>
__device__ __forceinline__ void fma_load(const elem_t* __restrict__ row, int k, int K, float (&out)[4]) {
  if (VEC) {
    load4_guarded(row + min(k, K - 4), 4, true, out);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = to_float(row[min(k + e, K - 1)]);
  }
}
__device__ __forceinline__ void fma_clear(float (&v)[4], int k, int K) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = k + e < K ? v[e] : 0.0f;
}

__device__ inline void fma_store(float v, float up, bool glu, const void* bias, int bias_is_f32, void* out, size_t at, int n,
                                 int mode) {
  if (bias) v += load_vec(bias, bias_is_f32, n);
  if (glu) ((elem_t*)out)[at] = from_float(swiglu1(v, up));
  else if (mode_stores_elem(mode)) ((elem_t*)out)[at] = from_float(mode_value(v, mode));
  else if (mode == MODE_ADD_F32) ((float*)out)[at] += v;
  else ((float*)out)[at] = v;
}

// Many rows (in the float32 build those that launch_fma_tiles does not give to gemm_fma_flow_kernel): 64 x 64 outputs a block of 4 waves, each 2 x 2 tiles of 16 x 16 (gated: half of a wave's
// columns are gate rows of W, half the up rows of the same outputs).  K is walked a chain at a time through
// two stages of LDS; the stage's operands are read first, then the next stage is written and the one
// after it asked for, all beside this stage's products.  A lane of a product holds k = 4 i + q of
// its row (q = lane / 16), so a row's 16 k are staged in the order [q][i]: one 16-byte read is a
// lane's operand of four products.  Rows of the stage are 144 bytes apart: the 16 rows that a read
// takes at a time fall into 16 different slots of the 64 banks.
#define TILE_M 64
#define TILE_LD (FMA_PART + 4)
template <bool GLU, bool VEC>
__global__ void __launch_bounds__(256, 2)
gemm_fma_kernel(const elem_t* __restrict__ x, int x_stride, const elem_t* __restrict__ w, const void* __restrict__ bias,
                int bias_is_f32, void* __restrict__ out, int out_stride, int M, int N, int K, int mode) {
  constexpr int R = 2, BM = TILE_M, ROWS = 2 * BM; // rows of X and then of W in a stage
  constexpr int BN = GLU ? BM / 2 : BM;            // columns of the output
  constexpr int LOADS = ROWS * FMA_PART / 4 / 256; // groups of four k a thread brings
  constexpr int ACROSS = FMA_PART / 4, DOWN = 256 / ACROSS;   // neighbouring threads bring a row's stage
  __shared__ __align__(16) float stages[2 * ROWS * TILE_LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int r16 = lane & 15, q = lane >> 4;
  const int wm = (wave >> 1) * 16 * R, wn = (wave & 1) * 16 * R;

  float in[LOADS][4];
  const elem_t* from[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int row = tid / ACROSS + DOWN * j;
    if (DOWN * j < BM) {
      from[j] = x + (size_t)min(m0 + row, M - 1) * x_stride;
    } else {
      // gated: a wave's columns are R / 2 tiles of gate rows, then the up rows of the same outputs
      const int half = (row - BM) / (16 * R), place = (row - BM) % (16 * R);
      const bool up = GLU && place >= 8 * R;
      const int n = GLU ? n0 + half * 8 * R + place - (up ? 8 * R : 0) : n0 + row - BM;
      from[j] = w + (size_t)(min(n, N - 1) + (up ? N : 0)) * K;
    }
  }
  const int k_mine = 4 * (tid % ACROSS);
  auto fetch = [&](int k0) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) fma_load<VEC>(from[j], k0 + k_mine, K, in[j]);
  };
  auto stage = [&](int which, int k0) {
    float* base = stages + which * ROWS * TILE_LD;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      float* to = base + (tid / ACROSS + DOWN * j) * TILE_LD + 16 * (tid % ACROSS / 4) + (tid & 3);
      if (k0 + FMA_PART > K) fma_clear(in[j], k0 + k_mine, K);
#pragma unroll
      for (int e = 0; e < 4; ++e) to[4 * e] = in[j][e];
    }
  };

  f32x4 sum[R][R];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) sum[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  fetch(0);
  stage(0, 0);
  if (FMA_PART < K) fetch(FMA_PART);
  __syncthreads();
  for (int k0 = 0, which = 0; k0 < K; k0 += FMA_PART, which ^= 1) {
    const float* base = stages + which * ROWS * TILE_LD;
    f32x4 a[2][R], b[2][R];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int i = 0; i < R; ++i) {
        a[g][i] = *reinterpret_cast<const f32x4*>(&base[(wm + 16 * i + r16) * TILE_LD + 16 * g + 4 * q]);
        b[g][i] = *reinterpret_cast<const f32x4*>(&base[(BM + wn + 16 * i + r16) * TILE_LD + 16 * g + 4 * q]);
      }
    // the next stage's numbers, asked for a step ago, go into LDS beside this stage's products
    if (k0 + FMA_PART < K) stage(which ^ 1, k0 + FMA_PART);
    if (k0 + 2 * FMA_PART < K) fetch(k0 + 2 * FMA_PART);
    f32x4 acc[R][R];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int j = 0; j < R; ++j) {
            if (g == 0 && s == 0) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            FMA_STEP(acc[i][j], a[g][i], b[g][j], s);
          }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j) sum[i][j] += acc[i][j];
    __syncthreads();
  }

  constexpr int COLS = GLU ? R / 2 : R;
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < COLS; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * q + e;
        const int n = n0 + (GLU ? wn / 2 : wn) + 16 * j + r16;
        if (m < M && n < N)
          fma_store(sum[i][j][e], GLU ? sum[i][j + (GLU ? COLS : 0)][e] : 0.0f, GLU, bias, bias_is_f32, out,
                    (size_t)m * out_stride + n, n, mode);
      }
}

// Few rows (decoding): such a product only waits for W, so a block takes up to 16 columns and the
// chains of an output, which do not need each other, are shared out over its 8 waves: every wave
// streams its chains' W from memory straight into operands, leaves the chains' sums in LDS, and a thread
// an output adds them in ascending order.  MT tiles of 16 rows of X ride along with each W (a wave reads
// them from L2 beside W, which is what bounds it from some 32 rows on).  What a wave multiplies next, W and X, is
// asked for as soon as the registers are free, with no branch between, so that loads are under way through the
// products, the barrier and the sums; they are buffer loads, whose k is in scalar registers, and the two halves of a
// line (16 k) are asked for one behind the other (four loads apart they came from L2 twice: 2,048 x K 5,632 at 16 rows
// 27 us, 22 so).  One chain of a wave at a time, or two where both operands are one tile: more of them (4 and 8)
// only wait for each other (the same 22 us against 20; a gated 5,632 x 2,048 of 5 rows 26 against 23 us).
// 5 rows, us, before (X asked for chain by chain between branches, a round's loads behind the last one's sums) / now:
// 2,560 x K 2,048 15.7 / 8.2, 2,048 x 2,048 11.7 / 8.9, gated 5,632 x 2,048 33.6 / 21.3 (4.3 TB/s), 2,048 x 5,632 29.2 / 17.2,
// 32,000 x 2,048 69 / 53 (4.9 TB/s); 32 rows of 2,560 x 2,048 23.7 / 14.3; 64 rows of 2,048 x 5,632 65 / 57.
#define FEW_WAVES 8
#define FEW_BRIEF (AXON_BF16 ? 4 : 7)      // so many chains, of all that the waves could take, go chain by chain (launch_fma_few)
#if AXON_BF16
typedef __attribute__((ext_vector_type(2))) unsigned fma_quad;      // four numbers as they lie in memory
#else
typedef u32x4 fma_quad;
#endif
// Rows as a buffer (buffer.h): a row's place in it is in the lane's register and the buffer begins at the k that is asked for, so
// that a load needs no address of its own, and what lies behind the last row reads as zeros.
struct FmaRows {
  const elem_t* base;
  unsigned bytes;
  // From number k of the rows on; where there is no such number, of no bytes: nothing is read.
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t from(int k, bool any = true) const {
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + k), 0, any ? bytes - (unsigned)k * (unsigned)sizeof(elem_t) : 0u, 0x00027000);
  }
};
__device__ __forceinline__ FmaRows fma_rows(const elem_t* matrix, int m, int M, int stride, int K) {
  const BufferRows rows = buffer_rows(m, M, stride, K, sizeof(elem_t));
  return {matrix + rows.first, rows.bytes};
}
// Four k of the row that begins `at` elements behind the first, k = k0 + in_chain .. + 3 (in_chain: this lane's place in
// the chain that begins at k0).  Aligned operands read on into the next row behind K; others take the row's last number.
// (A row's place: rows of numbers that are loaded singly may be any distance apart.)
template <bool VEC>
struct FmaPlace {
  typedef unsigned type;
};
template <>
struct FmaPlace<false> {
  typedef size_t type;
};
template <bool VEC>
__device__ __forceinline__ fma_quad fma_ask(const FmaRows& rows, typename FmaPlace<VEC>::type at, int k0, int in_chain, int K) {
  if (VEC) {
    const int off = (int)((at + in_chain) * sizeof(elem_t));
#if AXON_BF16
    return __builtin_amdgcn_raw_buffer_load_b64(rows.from(k0, k0 < K), off, 0, 0);
#else
    return __builtin_amdgcn_raw_buffer_load_b128(rows.from(k0, k0 < K), off, 0, 0);
#endif
  }
  union { fma_quad q; elem_t e[4]; } c;
#pragma unroll
  for (int e = 0; e < 4; ++e) c.e[e] = rows.base[at + min(k0 + in_chain + e, K - 1)];
  return c.q;
}
// What lies behind K of four k from `k` on becomes zeros.
__device__ __forceinline__ void fma_clear(fma_quad& raw, int k, int K) {
  union { fma_quad q; elem_t e[4]; } c;
  c.q = raw;
#pragma unroll
  for (int e = 0; e < 4; ++e) c.e[e] = k + e < K ? c.e[e] : from_float(0.0f);
  raw = c.q;
}
__device__ __forceinline__ f32x4 fma_operand(const fma_quad& raw) {
  union { fma_quad q; elem_t e[4]; } c;
  c.q = raw;
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = to_float(c.e[e]);
  return f32_operand(v);
}

template <int MT, int NR, bool GLU, bool VEC, bool SHORT>
__global__ void __launch_bounds__(64 * FEW_WAVES, 4)
gemm_fma_few_rows_kernel(const elem_t* __restrict__ x, int x_stride, const elem_t* __restrict__ w,
                         const void* __restrict__ bias, int bias_is_f32, void* __restrict__ out, int out_stride, int M,
                         int N, int K, int mode, int columns) {
  constexpr int NT = GLU ? 2 : 1;
  constexpr int ROUND = SHORT || MT * NT >= 2 ? 1 : 2;
  constexpr int PARTS = FEW_WAVES * ROUND, OUTS = MT * 16 * NR, ALL = NT * OUTS;
  constexpr int BUFFERS = PARTS * ALL * 4 > 32768 ? 1 : 2;          // of chains: two where two blocks a CU leave room
  __shared__ __align__(16) float chains[BUFFERS * PARTS * ALL];       // [chain][gate, up][row][NR columns]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * columns, m0 = blockIdx.y * MT * 16;
  FmaRows w_rows[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) w_rows[t] = fma_rows(w + (size_t)t * N * K, n0, N, K, K);
  const FmaRows x_rows = fma_rows(x, m0, M, x_stride, K);
  typedef typename FmaPlace<VEC>::type place_t;
  const place_t w_at = (place_t)min(min(r16, columns - 1), N - 1 - n0) * (place_t)K;
  place_t x_at[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) x_at[i] = (place_t)min(16 * i + r16, M - 1 - m0) * (place_t)x_stride;
  const int n_parts = (K + FMA_PART - 1) / FMA_PART;
  constexpr int MINE = (ALL + 64 * FEW_WAVES - 1) / (64 * FEW_WAVES);
  float sum[MINE];
#pragma unroll
  for (int i = 0; i < MINE; ++i) sum[i] = 0.0f;

  fma_quad wq[ROUND][NT][2], xq[ROUND][MT][2];
  // whole: of a round whose chains all exist
  auto ask = [&](int p, int first, bool whole) {
    const int k0 = (first + p * FEW_WAVES + wave) * FMA_PART;
    if (!VEC && !whole && k0 >= K) return;   // no chain, the same for the whole wave
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int g = 0; g < 2; ++g) wq[p][t][g] = fma_ask<VEC>(w_rows[t], w_at, k0, 16 * g + 4 * q, K);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int g = 0; g < 2; ++g) xq[p][i][g] = fma_ask<VEC>(x_rows, x_at[i], k0, 16 * g + 4 * q, K);
  };
#pragma unroll
  for (int p = 0; p < ROUND; ++p) ask(p, 0, false);
  int buffer = 0;
  auto round = [&](int first, bool more, bool whole) {
    float* to = chains + buffer * PARTS * ALL;
#pragma unroll
    for (int p = 0; p < ROUND; ++p) {
      const int part = p * FEW_WAVES + wave, k0 = (first + part) * FMA_PART, k = k0 + 4 * q;
      if (!more && k0 >= K) continue;                      // no chain: in the last round alone
      if (k0 < K && k0 + FMA_PART > K) {                   // K ends in this chain: the same for the whole wave
#pragma unroll
        for (int g = 0; g < 2; ++g) {
#pragma unroll
          for (int t = 0; t < NT; ++t) fma_clear(wq[p][t][g], k + 16 * g, K);
#pragma unroll
          for (int i = 0; i < MT; ++i) fma_clear(xq[p][i][g], k + 16 * g, K);
        }
      }
      f32x4 a[NT][2], b[MT][2];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
#pragma unroll
        for (int t = 0; t < NT; ++t) a[t][g] = fma_operand(wq[p][t][g]);
#pragma unroll
        for (int i = 0; i < MT; ++i) b[i][g] = fma_operand(xq[p][i][g]);
      }
      if (more) ask(p, first + PARTS, whole);
      f32x4 acc[MT][NT];
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              if (g == 0 && s == 0) acc[i][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
              FMA_STEP(acc[i][t], a[t][g], b[i][g], s);
            }
      // columns 4 q .. 4 q + 3 of row 16 i + r16
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          if (4 * q < NR) *reinterpret_cast<f32x4*>(&to[(part * NT + t) * OUTS + (16 * i + r16) * NR + 4 * q]) = acc[i][t];
    }
    wait_lgkmcnt<0>();
    __builtin_amdgcn_s_barrier();          // (loads stay under way)
    asm volatile("" ::: "memory");
    const int count = min(PARTS, n_parts - first);
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
      const int o = tid + 64 * FEW_WAVES * i;
      if (o < ALL) {
        if (count == PARTS) {
#pragma unroll
          for (int p = 0; p < PARTS; ++p) sum[i] += to[p * ALL + o];
        } else {
          for (int p = 0; p < count; ++p) sum[i] += to[p * ALL + o];
        }
      }
    }
    if (BUFFERS == 1) {
      wait_lgkmcnt<0>();                     // the sums' reads have run before another wave writes the next round's there
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    if (BUFFERS == 2) buffer ^= 1;
  };
  int first = 0;
  if constexpr (VEC) {
    for (; first + PARTS < n_parts; first += PARTS) round(first, true, false);
  } else {                       // the check of every chain takes up to 7 % (a row of 300 x K 5,631)
    for (; first + 2 * PARTS <= n_parts; first += PARTS) round(first, true, true);
    if (first + PARTS < n_parts) {
      round(first, true, false);
      first += PARTS;
    }
  }
  round(first, false, false);

  float up[MINE];
  if (GLU) {                     // the up sums go to the threads that hold the gates'
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MINE; ++i)
      if (tid + 64 * FEW_WAVES * i < ALL) chains[tid + 64 * FEW_WAVES * i] = sum[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MINE; ++i) up[i] = chains[(tid + 64 * FEW_WAVES * i) % OUTS + (NT - 1) * OUTS];
  }
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    const int o = tid + 64 * FEW_WAVES * i, m = m0 + o / NR, c = o % NR, col = n0 + c;
    if (o < OUTS && c < columns && m < M && col < N)
      fma_store(sum[i], GLU ? up[i] : 0.0f, GLU, bias, bias_is_f32, out, (size_t)m * out_stride + col, col, mode);
  }
}

// The same with X asked for chain by chain, when it is multiplied, several chains of W before it; a wave without a chain asks for
// nothing and multiplies nothing (launch_fma_few says for which products).
//  * Numbers that have to be loaded singly (a K, rows or a base that are not aligned for four): four loads take the place of one, with
//    addresses of their own, and all of X ahead does not fit the registers.  us, all ahead / so: 20 rows of 1,000 x K 1,001
//    14.0 / 13.1, 40 of 2,048 x 2,047 40.4 / 37.0, gated 5,632 x 2,049 5 rows 59.3 / 58.6, 32 91.5 / 86.5, 64 140 / 122; 256 x 127 of
//    5 rows 3.2 / 2.7, of 64 6.7 / 4.4.
//  * Fewer chains than waves: 64 rows of 64 x K 96 4.5 / 3.3 us, of 256 x 128 4.6 / 3.4, of 4,096 x 192 5.7 / 5.0, gated 512 x 128
//    5.9 / 4.2; 5 rows 2.5 / 2.3, 2.5 / 2.4, 3.4 / 3.3 and 3.4 / 2.7.
template <int MT, int NR, bool GLU, bool VEC, bool SHORT>
__global__ void __launch_bounds__(64 * FEW_WAVES, 2)
gemm_fma_by_chain_kernel(const elem_t* __restrict__ x, int x_stride, const elem_t* __restrict__ w, const void* __restrict__ bias,
                         int bias_is_f32, void* __restrict__ out, int out_stride, int M, int N, int K, int mode, int columns) {
  constexpr int NT = GLU ? 2 : 1;
  constexpr int PW = SHORT || MT * NT >= 8 ? 1 : MT * NT >= 3 ? 2 : MT * NT == 2 ? 4 : 8;   // chains of a wave in a round
  constexpr int PARTS = FEW_WAVES * PW, OUTS = MT * 16 * NR;
  __shared__ __align__(16) float chains[PARTS * NT * OUTS];                        // [chain][gate, up][row][column]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * columns, m0 = blockIdx.y * MT * 16;
  const elem_t* w_row = w + (size_t)min(n0 + min(r16, columns - 1), N - 1) * K;
  const elem_t* x_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) x_row[i] = x + (size_t)min(m0 + 16 * i + r16, M - 1) * x_stride;
  const int n_parts = (K + FMA_PART - 1) / FMA_PART;
  constexpr int MINE = (OUTS + 64 * FEW_WAVES - 1) / (64 * FEW_WAVES);
  float sum[MINE], sum_up[MINE];
#pragma unroll
  for (int i = 0; i < MINE; ++i) sum[i] = sum_up[i] = 0.0f;

  for (int first = 0; first < n_parts; first += PARTS) {
    float wv[NT][PW][2][4];
#pragma unroll
    for (int p = 0; p < PW; ++p)
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          fma_load<VEC>(w_row + (size_t)t * N * K, (first + wave * PW + p) * FMA_PART + 16 * g + 4 * q, K, wv[t][p][g]);
#pragma unroll
    for (int p = 0; p < PW; ++p) {
      const int part = wave * PW + p, k0 = (first + part) * FMA_PART;
      if (k0 >= K) break;                            // the same for the whole wave
      f32x4 a[NT][2];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          if (k0 + FMA_PART > K) fma_clear(wv[t][p][g], k0 + 16 * g + 4 * q, K);
          a[t][g] = f32_operand(wv[t][p][g]);
        }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        f32x4 b[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          float xv[4];
          fma_load<VEC>(x_row[i], k0 + 16 * g + 4 * q, K, xv);
          if (k0 + FMA_PART > K) fma_clear(xv, k0 + 16 * g + 4 * q, K);
          b[g] = f32_operand(xv);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int s = 0; s < 4; ++s) FMA_STEP(acc, a[t][g], b[g], s);
          // columns 4 q .. 4 q + 3 of row 16 i + r16
          if (4 * q < NR) *reinterpret_cast<f32x4*>(&chains[(part * NT + t) * OUTS + (16 * i + r16) * NR + 4 * q]) = acc;
        }
      }
    }
    __syncthreads();
    const int count = min(PARTS, n_parts - first);
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
      const int o = tid + 64 * FEW_WAVES * i;
      if (o < OUTS) {
#pragma unroll 8
        for (int p = 0; p < count; ++p) {
          sum[i] += chains[p * NT * OUTS + o];
          if (GLU) sum_up[i] += chains[(p * NT + NT - 1) * OUTS + o];
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    const int o = tid + 64 * FEW_WAVES * i, m = m0 + o / NR, c = o % NR, col = n0 + c;
    if (o < OUTS && c < columns && m < M && col < N)
      fma_store(sum[i], sum_up[i], GLU, bias, bias_is_f32, out, (size_t)m * out_stride + col, col, mode);
  }
}

#if !AXON_BF16
// gemm_fma_kernel's tiles and chains for rows of 32-bit numbers that are aligned: rows go to LDS as they lie in memory, by direct loads,
// FLOW_STAGES stages ahead, and the numbers that a product wants of them (k = 4 s + q of row lane % 16) are read two tiles
// at a time, two reads behind each of the first products of the step before.  So nothing is written to LDS, converted or cleared by the
// vector unit, a wave waits for nothing that was not asked for half a step ago, and a chain's sums are added beside
// the next chain's products.  A row of a stage is eight slots of 16 bytes, permuted by slot ^ (row / 2 % 8): the four k of 16
// rows that a read takes fall on the 64 banks.
// What bounds it: with four blocks a CU 83 % of what the products alone take (139 TFLOP/s at the clock that they leave); with one or two
// blocks a CU also how they divide the rows, so a block has 32 to 96 of them (flow_rows).
// 777 rows, us, through registers / here: 2,560 x K 2,048 121 / 114, 2,048 x 2,060 89 / 76, 2,048 x 5,632 234 / 198, gated 5,632 x
// 2,048 338 / 329, 32,000 x 2,048 960 / 942; 512 rows of 2,048 x 5,632 (a block a CU) 142 / 116, 2,048 rows 414 / 393.  With a read a
// number (128 LDS instructions a block and step) 409 for the last, three stages (three blocks a CU) 412.
#define FLOW_STAGES 4
#define FLOW_STAGE(rows) (((rows) + TILE_M) * FMA_PART * 4)
#define FLOW_LEAST_K 192      // (launch_fma_tiles)
typedef const __attribute__((address_space(1))) void* fma_global_t;
typedef __attribute__((address_space(3))) void* fma_lds_t;
typedef __attribute__((ext_vector_type(2))) float f32x2;
// A product's operand of TILES tiles: a lane's number of each, read two tiles at a time, 2 KB (16 rows of a stage) apart, and the
// last of an odd number alone.
template <int TILES>
struct FmaOperand {
  static constexpr int PAIRS = (TILES + 1) / 2;
  f32x2 two[TILES > 1 ? TILES / 2 : 1];
  float one;
  __device__ __forceinline__ float number(int i) const { return TILES % 2 && i == TILES - 1 ? one : two[i / 2][i % 2]; }
  // read `pair` of the PAIRS
  template <int I = PAIRS - 1>
  __device__ __forceinline__ void read(unsigned lds_address, int pair) {
    if (pair == I) {
      if constexpr (TILES % 2 && I == PAIRS - 1) asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(one) : "v"(lds_address), "n"(I * 4096));
      else asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(two[I]) : "v"(lds_address), "n"(I * 16), "n"(I * 16 + 8));
    } else if constexpr (I > 0) {
      read<I - 1>(lds_address, pair);
    }
  }
  __device__ __forceinline__ void use() {
#pragma unroll
    for (int i = 0; i < TILES / 2; ++i) asm volatile("" : "+v"(two[i]));
    if constexpr (TILES % 2) asm volatile("" : "+v"(one));
  }
};
template <int V>
struct FmaNumber {
  static constexpr int value = V;
};
// WAVES_M x (4 / WAVES_M) waves, each TM x TN tiles of 16 x 16: 16 WAVES_M TM rows by 64 rows of W a block.
template <bool GLU, int WAVES_M, int TM, int TN>
__global__ void __launch_bounds__(256, TM * TN <= 6 ? 2 : 1)
gemm_fma_flow_kernel(const float* __restrict__ x, int x_stride, const float* __restrict__ w, const void* __restrict__ bias,
                     int bias_is_f32, void* __restrict__ out, int out_stride, int M, int N, int K, int mode) {
  constexpr int BM = 16 * WAVES_M * TM, BN = GLU ? TILE_M / 2 : TILE_M, STAGE = FLOW_STAGE(BM), PRODUCTS = 8 * TM * TN;
  constexpr int XL = (BM / 8 + 3) / 4, LOADS = XL + 2;           // load instructions of a wave and stage: of X, with W's two
  constexpr int PAIRS = FmaOperand<TM>::PAIRS, READS = 8 * (PAIRS + 1), EACH = (2 * READS + PRODUCTS - 1) / PRODUCTS;
  static_assert(4 / WAVES_M * TN * 16 == TILE_M && (!GLU || TN == 2) && LOADS * FLOW_STAGES < 64, "64 rows of W a block");
  extern __shared__ __align__(128) unsigned char flow[];          // [stage]: X [BM][32], W [64][32]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int r16 = lane & 15, q = lane >> 4;
  const int wm = WAVES_M == 2 ? (wave >> 1) * 16 * TM : 0, wn = (WAVES_M == 2 ? wave & 1 : wave) * 16 * TN;

  // A load fills 8 rows of a stage, lane l slot l % 8 of row l / 8, which holds k chunk slot ^ (row / 2 % 8): loads 0 .. XL - 1 rows
  // 8 (4 j + wave) and on of X (where there are none: some twice), the last two the same of W (gated: in a wave's 32 rows 16 gate
  // rows, then the up rows of the same outputs)
  const int lrow = lane >> 3;
  const bool up = GLU && (wave & 2);
  const FmaRows x_rows = fma_rows(x, m0, M, x_stride, K);
  const FmaRows w_rows = fma_rows(w + (up ? (size_t)N * K : 0), n0, N, K, K);
  auto group = [&](int j) { return j < XL ? min(4 * j + wave, BM / 8 - 1) : 4 * (j - XL) + wave; };
  unsigned at[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int row = 8 * group(j) + lrow, chunk = (lane & 7) ^ ((4 * group(j) + (lane >> 4)) & 7);
    const int col = GLU ? 16 * (j - XL) + 8 * (wave & 1) + lrow : row;
    at[j] = (j < XL ? (unsigned)min(row, M - 1 - m0) * (unsigned)x_stride : (unsigned)min(col, N - 1 - n0) * (unsigned)K) * 4 + 16 * chunk;
  }
  auto ask = [&](int t, int j) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds((j < XL ? x_rows : w_rows).from(t * FMA_PART),
                                             (fma_lds_t)(flow + t % FLOW_STAGES * STAGE + (j < XL ? 0 : BM * 128) + group(j) * 1024), 16,
                                             (int)at[j], 0, 0, 0);
  };
  const unsigned lds0 = (unsigned)(size_t)(fma_lds_t)flow;
  unsigned x_at[8], w_at[8];               // of product s of a chain: of X's first tile, of W's
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    x_at[s] = lds0 + (wm + r16) * 128 + ((s ^ (r16 >> 1)) << 4) + 4 * q;
    w_at[s] = x_at[s] + BM * 128 + (wn - wm) * 128;
  }
  FmaOperand<TM> a[2][8];                  // of a wave's tiles
  FmaOperand<TN> b[2][8];
  // read p of those of a stage: X's and W's numbers of product p / (PAIRS + 1)
  auto read = [&](auto set_of, unsigned stage, int p) {
    constexpr int set = decltype(set_of)::value;
    const int s = p / (PAIRS + 1), of = p % (PAIRS + 1);
    if (of < PAIRS) a[set][s].read(x_at[s] + stage, of);
    else b[set][s].read(w_at[s] + stage, 0);
  };
  auto arrived = [&](auto set_of) {
    constexpr int set = decltype(set_of)::value;
    wait_lgkmcnt<0>();
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      a[set][s].use();
      b[set][s].use();
    }
  };
  f32x4 sum[TM][TN], acc[2][TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[i][j] = acc[1][i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const int n_steps = (K + FMA_PART - 1) / FMA_PART;
  static_assert(FLOW_LEAST_K > FLOW_STAGES * FMA_PART, "as many steps as stages");
#pragma unroll
  for (int t = 0; t < FLOW_STAGES; ++t)
#pragma unroll
    for (int j = 0; j < LOADS; ++j) ask(t, j);
  wait_vmcnt<LOADS*(FLOW_STAGES - 1)>();
  __builtin_amdgcn_s_barrier();            // stage 0 is in LDS for every wave
#pragma unroll
  for (int p = 0; p < READS; ++p) read(FmaNumber<0>(), 0u, p);
  arrived(FmaNumber<0>());
  // Step t, whose numbers are in registers: its stage is free behind the barrier.  asks: for stage t + FLOW_STAGES.
  auto step = [&](int t, auto set_of, auto asks_of) {
    constexpr int set = decltype(set_of)::value, other = set ^ 1;
    constexpr bool asks = decltype(asks_of)::value != 0;
    if constexpr (asks) {
      wait_vmcnt<LOADS*(FLOW_STAGES - 2)>();
    } else {
      const int left = n_steps - t;        // of the stages behind the next, left - 2 may still be under way
      if (FLOW_STAGES >= 4 && left >= 4) wait_vmcnt<2 * LOADS>();
      else if (left >= 3) wait_vmcnt<LOADS>();
      else wait_vmcnt<0>();
    }
    __builtin_amdgcn_s_barrier();          // stage t + 1 is in LDS for every wave; nobody reads stage t any more
    const unsigned next = (unsigned)((t + 1) % FLOW_STAGES * STAGE);
#pragma unroll
    for (int p = 0; p < PRODUCTS; ++p) {
      const int s = p / (TM * TN), i = p / TN % TM, j = p % TN;
      if (s == 0) acc[set][i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      acc[set][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[set][s].number(i), b[set][s].number(j), acc[set][i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = p * EACH; r < (p + 1) * EACH; ++r)      // as soon as they go: spread over more products they take 1 to 5 % longer
        if (r < READS) read(FmaNumber<other>(), next, r);
      constexpr int HALF = PRODUCTS / 2;
      if (p >= HALF && p < HALF + TM * TN) sum[(p - HALF) / TN][p % TN] += acc[other][(p - HALF) / TN][p % TN];      // the chain before
      if (asks && (PRODUCTS - 1 - p) % 3 == 0 && (PRODUCTS - 1 - p) / 3 < LOADS) ask(t + FLOW_STAGES, LOADS - 1 - (PRODUCTS - 1 - p) / 3);
      __builtin_amdgcn_sched_barrier(0);
    }
    arrived(FmaNumber<other>());           // (behind the last step: whatever lies there, not used)
  };
  const int whole = K / FMA_PART;          // the last step of a K that is no multiple of 32 has fewer products
  int t = 0;
  for (; t + 1 + FLOW_STAGES < n_steps; t += 2) {
    step(t, FmaNumber<0>(), FmaNumber<1>());
    step(t + 1, FmaNumber<1>(), FmaNumber<1>());
  }
  if (t + FLOW_STAGES < n_steps) {         // one more asks
    step(t, FmaNumber<0>(), FmaNumber<1>());
    step(t + 1, FmaNumber<1>(), FmaNumber<0>());
    t += 2;
  }
  for (; t + 1 < whole; t += 2) {
    step(t, FmaNumber<0>(), FmaNumber<0>());
    step(t + 1, FmaNumber<1>(), FmaNumber<0>());
  }
  auto last = [&](auto set_of) {           // the products of the k that are left
    constexpr int set = decltype(set_of)::value;
    const int count = (K - whole * FMA_PART) / 4;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        sum[i][j] += acc[set ^ 1][i][j];
        acc[set][i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (s < count) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[set][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[set][s].number(i), b[set][s].number(j), acc[set][i][j], 0, 0, 0);
      }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) sum[i][j] += acc[set][i][j];
  };
  if (t < whole) {                         // t is even: one whole step, and what may be left
    step(t, FmaNumber<0>(), FmaNumber<0>());
    last(FmaNumber<1>());
  } else {
    last(FmaNumber<0>());
  }

  constexpr int COLS = GLU ? TN / 2 : TN;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < COLS; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * q + e;
        const int n = n0 + (GLU ? wn / 2 : wn) + 16 * j + r16;
        if (m < M && n < N)
          fma_store(sum[i][j][e], GLU ? sum[i][j + (GLU ? COLS : 0)][e] : 0.0f, GLU, bias, bias_is_f32, out,
                    (size_t)m * out_stride + n, n, mode);
      }
}
#endif

template <int MT, bool GLU, bool VEC>
static void launch_fma_few(const elem_t* x, int x_stride, const elem_t* w, const void* bias, int bias_is_f32, void* out,
                           int out_stride, int m, int n, int k, int mode, hipStream_t stream) {
  // As many blocks as give every CU the same number of them, with at most 16 columns each, and so many that X counts less than W
  // (5 rows of 2,560 columns of K 2,048 in 256 blocks of 10: 7.6 us, in 160 of 16 8.1; of gated 5,632 in 512 of 11: 20.1, in 352 of 16
  // 23.9).
  // X that is loaded singly counts more than a last round: 16 columns from four blocks a CU on (16 rows of 16,390 x 1,001 in blocks
  // of 13: 51.7, of 16 48.9), and whole or half tiles chain by chain.
  const int rows = ceil_div(m, 16 * MT), tiles = ceil_div(n, 16) * rows, each = ceil_div(tiles, 256);
  const int spread = max(MT == 1 ? 4 : 8, min(16, ceil_div(n * rows, 256 * each)));
  // Which kernel.  Numbers loaded singly: one tile of rows and one of W, in a K of more than a chain a wave, are asked for ahead like
  // others (us, against chain by chain: 5 rows of 1,000 x K 1,001 7.5 / 9.5, of 300 x 5,631 31 / 40, of 2,048 x 515 6.0 / 8.4; 16 of
  // 2,048 x 769 9.7 / 10.3, of 16,390 x 515 27.5 / 33.7).  Aligned: fewer chains than waves go chain by chain,
  // and 64 rows of as many (us, ahead / so: 512 x K 256 4.5 / 4.3, 2,048 x 256 5.0 / 4.9; gated, and of fewer rows, ahead is the faster: 5 rows of
  // 2,048 x 256 3.0 / 3.2, of gated 5,632 x 256 a fifth).  In the bfloat16 build, whose numbers are half as long, up to half the waves
  // (ahead / so: 5 rows of 512 x 192 2.7 / 2.8, 40 of 2,048 x 224 4.4 / 4.8, 40 of 512 x 256 4.1 / 4.6).
  constexpr bool AHEAD = VEC || (MT == 1 && !GLU);
  const bool brief = k <= FEW_WAVES * FMA_PART;
#define FEW(KERNEL, SHORT, COLUMNS)                                                                                         \
  {                                                                                                                         \
    const int columns = COLUMNS;                                                                                            \
    const dim3 blocks(ceil_div(n, columns), rows);                                                                          \
    if (columns <= 8) KERNEL<MT, 8, GLU, VEC, SHORT><<<blocks, 64 * FEW_WAVES, 0, stream>>>(FEW_ARGS, columns);             \
    else KERNEL<MT, 16, GLU, VEC, SHORT><<<blocks, 64 * FEW_WAVES, 0, stream>>>(FEW_ARGS, columns);                         \
  }
#define BY_CHAIN(SHORT, COLUMNS)                              \
  {                                                           \
    AXK_INSTANCE(INST_GEMM_FMA_BY_CHAIN, 16 * MT, GLU, VEC);  \
    FEW(gemm_fma_by_chain_kernel, SHORT, COLUMNS)             \
  }
#define FEW_ARGS x, x_stride, w, bias, bias_is_f32, out, out_stride, m, n, k, mode
  if constexpr (VEC) {
    if (k <= FEW_BRIEF * FMA_PART || (!AXON_BF16 && brief && MT == 4 && !GLU)) BY_CHAIN(true, max(8, spread))
    else if (brief) FEW(gemm_fma_few_rows_kernel, true, spread)
    else FEW(gemm_fma_few_rows_kernel, false, spread)
  } else {
    if (brief) BY_CHAIN(true, tiles < 256 ? 8 : 16)
    else if constexpr (AHEAD) FEW(gemm_fma_few_rows_kernel, false, each >= 4 ? 16 : spread)
    else BY_CHAIN(false, tiles < 256 ? 8 : 16)
  }
#undef FEW_ARGS
#undef BY_CHAIN
#undef FEW
}

#if !AXON_BF16
// Rows a block of gemm_fma_flow_kernel: what takes least by how many blocks the fullest CU then has: of one `alone`, of more
// `each` for every one and `odd` where one stays without its neighbour (us for K 2,048, measured with 2,048, 2,560 and 8,192
// columns and gated 5,632 at 129 to 2,048 rows, all within 5 % of it; of 32 rows the first three blocks take 5 more).  64 rows of all / so, K 2,048: 2,048
// columns, 129 and 200 rows 47 / 30, 300 48 / 40, 626 76 / 56, 1,500 118 / 105; 2,560 columns, 430 rows 76 / 56, 777 117 / 84, 1,024
// 117 / 101; gated 5,632, 129 rows 117 / 86, 900 405 / 367, 1,500 620 / 570.  Blocks of 112 and of 128 rows, one a CU, are the best of none.
// With K the other heights' times grow faster than those of 64 rows, gated 96 excepted, by one in 80,000 k (each height at 14 shapes and K 256
// to 14,336: so chosen 0.916 of the time with 64 rows for all, 1.005 of the best height's, none over 2 % longer than with 64; without that up to 22 %:
// 900 rows of 4,096 of K 11,008 759 / 865 with 80, gated 512 of 5,632 1,158 / 1,305 with 32).
static int flow_rows(int columns, int m, int k, bool glu) {
  int best = 0;
  double least = 0.0;
  const double dear = 1.0 + (k > 1024 ? (k - 1024) / 80000.0 : 0.0);
  auto is = [&](int rows, double alone, double each, double odd) {
    const long blocks = ((long)columns * ceil_div(m, rows) + 255) / 256;
    double cost = blocks == 1 ? alone : blocks * each + (blocks % 2 ? odd : 0.0) + (rows == 32 && blocks <= 3 ? 5.0 : 0.0);
    if (rows != 64 && !(glu && rows == 96)) cost *= dear;
    if (best == 0 || cost < least) {
      best = rows;
      least = cost;
    }
  };
  is(64, 47.0, 36.7, 5.0);
  is(32, 30.0, 19.7, 0.0);
  is(96, 62.0, 51.8, 8.0);
  if (!glu) {
    is(48, 39.0, 29.4, 2.0);
    is(80, 55.0, 45.3, 7.0);
  }
  return best;
}

template <bool GLU, int WAVES_M, int TM, int TN>
static int launch_flow(unsigned columns, const float* x, int x_stride, const float* w, const void* bias, int bias_is_f32, void* out,
                       int out_stride, int m, int n, int k, int mode, hipStream_t stream) {
  constexpr int rows = 16 * WAVES_M * TM, lds = FLOW_STAGES * FLOW_STAGE(rows);
  constexpr auto kernel = &gemm_fma_flow_kernel<GLU, WAVES_M, TM, TN>;
  static bool configured = lds <= 64 * 1024;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      axk_set_error("gemm_fma: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  AXK_INSTANCE(INST_GEMM_FMA_FLOW_ROWS, rows, GLU);
  kernel<<<dim3(columns, ceil_div(m, rows)), 256, lds, stream>>>(x, x_stride, w, bias, bias_is_f32, out, out_stride, m, n, k, mode);
  return 0;
}
#endif

template <bool GLU, bool VEC>
static int launch_fma_tiles(dim3 tiles, const elem_t* x, int x_stride, const elem_t* w, const void* bias, int bias_is_f32, void* out,
                             int out_stride, int m, int n, int k, int mode, hipStream_t stream) {
#if !AXON_BF16
  // Short K: the stages that are filled before the first product count more than what they save, and where there are more
  // than two blocks a CU these cover each other's waits.  us, through registers / by direct loads: up to 512 blocks, 400 rows of 1,000
  // columns of K 64 4.8 / 5.4, 128 6.6 / 6.9, 192 8.4 / 8.3, 256 10.0 / 9.6; more, 777 rows of 4,096 of K 96 12.6 / 15.9, 256 24.0 / 25.5,
  // 512 42.3 / 42.8, 640 51.4 / 51.0; of 32,000 of K 256 136 / 146, 640 309 / 314, as long from 1,024 on.
  if constexpr (VEC) {
    if (k >= ((long)tiles.x * tiles.y <= 512 ? FLOW_LEAST_K : 640)) {
      AXK_INSTANCE(INST_GEMM_FMA_FLOW, GLU);
#define FLOW(WAVES_M, TM, TN) return launch_flow<GLU, WAVES_M, TM, TN>(tiles.x, x, x_stride, w, bias, bias_is_f32, out, out_stride, m, n, k, mode, stream)
      const int rows = flow_rows(tiles.x, m, k, GLU);
      if (rows == 32) FLOW(2, 1, 2);
      if (rows == 96) FLOW(2, 3, 2);
      if constexpr (!GLU) {
        if (rows == 48) FLOW(1, 3, 1);
        if (rows == 80) FLOW(1, 5, 1);
      }
      FLOW(2, 2, 2);
#undef FLOW
    }
  }
#endif
  gemm_fma_kernel<GLU, VEC><<<tiles, 256, 0, stream>>>(x, x_stride, w, bias, bias_is_f32, out, out_stride, m, n, k, mode);
  return 0;
}

// Whether 33 to 128 rows of aligned 32-bit numbers go to the tiles though these are fewer than the CUs: where a wave a chain
// would give a CU two blocks, tiles of 32 rows are the faster.  us, K 2,048: one block a CU, 2,048 columns of 64 rows 20.5 / 28.7, of 128
// 22.7 / 29.3; two, 2,560 of 65 33.6 / 28.8, of 128 39 / 29, 8,192 of 33 32.5 / 29.6, of 64 40.5 / 29.6, gated 5,632 of 64 53 / 46; four, 16,000 of
// K 1,024 of 64 42 / 27.
template <bool VEC>
static bool tiles_of_few_rows(int m, int n, int k) {
  return !AXON_BF16 && VEC && k >= 512 && (long)ceil_div(n, 16) * ceil_div(m, 64) > 256;
}

static int launch_fma(const elem_t* x, int x_stride, const elem_t* w, const void* bias, int bias_is_f32, void* out,
                      int out_stride, int m, int n, int k, int mode, hipStream_t stream) {
  const size_t vbytes = 4 * sizeof(elem_t);
  // (rows a block reads as a buffer lie within 4 GB)
  const bool vec_w = (k % 4 == 0) && ((uintptr_t)w % vbytes == 0) && k < (1 << 23);
  const bool vec_x = (k % 4 == 0) && (x_stride % 4 == 0) && ((uintptr_t)x % vbytes == 0) && x_stride < (1 << 23);
#define FMA_ARGS x, x_stride, w, bias, bias_is_f32, out, out_stride, m, n, k, mode, stream
// Up to 32 rows a product waits for W; from 33 to 128 so it does where the tiles would be fewer than the CUs.  us, a wave a
// chain / tiles: 128 rows of 2,048 columns of K 5,632 (64 tiles) 58 / 114, 64 of 8,192 of K 2,048 (128) 42 / 45, 65 of them (256) 67 / 46, of gated
// 5,632 (352) 78 / 75, 33 and 64 of 32,000 (500) 119 / 78 and 153 / 81.
#define FMA_LAUNCH(GLU, VEC)                                                                  \
  const dim3 tiles(ceil_div(n, GLU ? TILE_M / 2 : TILE_M), ceil_div(m, TILE_M));              \
  if (m <= 16) {                                                                              \
    AXK_INSTANCE(INST_GEMM_FMA, 16, GLU);                                                     \
    launch_fma_few<1, GLU, VEC>(FMA_ARGS);                                                    \
  } else if (m <= 32) {                                                                       \
    AXK_INSTANCE(INST_GEMM_FMA, 32, GLU);                                                     \
    launch_fma_few<2, GLU, VEC>(FMA_ARGS);                                                    \
  } else if (m <= 128 && (long)tiles.x * tiles.y < 256 && !tiles_of_few_rows<VEC>(m, n, k)) { \
    AXK_INSTANCE(INST_GEMM_FMA, 64, GLU);                                                     \
    launch_fma_few<4, GLU, VEC>(FMA_ARGS);                                                    \
  } else {                                                                                    \
    AXK_INSTANCE(INST_GEMM_FMA, 128, GLU);                                                    \
    if (const int rc = launch_fma_tiles<GLU, VEC>(tiles, FMA_ARGS)) return rc;                \
  }
  const bool glu = mode == MODE_SWIGLU;
  if (vec_x && vec_w) {
    if (glu) { FMA_LAUNCH(true, true) } else { FMA_LAUNCH(false, true) }
  } else {
    if (glu) { FMA_LAUNCH(true, false) } else { FMA_LAUNCH(false, false) }
  }
#undef FMA_ARGS
#undef FMA_LAUNCH
  AXK_LAUNCH_CHECK("gemm_fma");
  return 0;
}

#if AXON_BF16
int launch_gemm_mfma(const bf16_t* x, int x_stride, const bf16_t* w, const void* bias, int bias_is_f32, void* out,
                     int out_stride, int m, int n, int k, int mode, hipStream_t stream, const GemmNormFold* then_norm,
                     void* workspace, size_t workspace_bytes);
int gemm_pack_ok(int rows, int k, int gated);
int launch_pack_matrix(const bf16_t* src, bf16_t* dst, int rows, int k, hipStream_t stream);
size_t gemm_workspace_bytes(int m, int n, int k, int mode);
int gemm_segments(int tiles32, int k);
int gemm_then_norm_ok(int m, int n, int k);
int gemm_qkv_rope_ok(int m, int n, int k, int head_dim, int rotary_dim);
int launch_gemm_qkv_rope(const bf16_t* x, int x_stride, const bf16_t* w, const void* bias, int bias_is_f32, bf16_t* out,
                         int out_stride, int m, int n, int k, const float* table, const int32_t* positions,
                         const int32_t* seq_rows, const int32_t* block_table, int table_stride, bf16_t* k_cache,
                         bf16_t* v_cache, int n_heads, int n_kv_heads, int head_dim, int page_size, void* workspace,
                         size_t workspace_bytes, hipStream_t stream);
int gemm_normed_ok(int m, int k);
int launch_gemm_normed_glu(const float* rows, int rows_stride, const bf16_t* gain, float eps, const bf16_t* w, bf16_t* out,
                           int out_stride, int m, int n, int k, hipStream_t stream);
int launch_gemm_normed_qkv_rope(const float* rows, int rows_stride, const bf16_t* gain, float eps,
                                const bf16_t* w, const void* bias, int bias_is_f32, bf16_t* out, int out_stride, int m, int n,
                                int k, const float* table, const int32_t* positions, const int32_t* seq_rows,
                                const int32_t* block_table, int table_stride, bf16_t* k_cache, bf16_t* v_cache, int n_heads,
                                int n_kv_heads, int head_dim, int page_size, hipStream_t stream);
#endif

static int gemm_checked(const void* x, int x_stride, const void* w, int w_packed, const void* bias, int bias_is_f32,
                        void* out, int out_stride, int m, int n, int k, int mode, const GemmNormFold* fold,
                        void* workspace, long workspace_bytes, void* stream) {
  AXK_REQUIRE(m >= 0 && n > 0 && k > 0, "gemm: bad sizes M=%d N=%d K=%d", m, n, k);
  AXK_REQUIRE(x_stride >= k && out_stride >= n, "gemm: strides x=%d (K=%d) out=%d (N=%d) too small", x_stride, k,
              out_stride, n);
  AXK_REQUIRE(mode >= 0 && mode <= MODE_RELU_SQUARED, "gemm: unknown mode %d", mode);
  AXK_REQUIRE(mode != MODE_SWIGLU || bias == nullptr, "gemm: the gated epilogue takes no bias");
  AXK_REQUIRE(ceil_div(m, 16) <= 65535, "gemm: M=%d is more rows than one launch takes", m);
  if (m == 0) return 0;
  if (w_packed) {
#if AXON_BF16
    return launch_gemm_mfma((const bf16_t*)x, x_stride, (const bf16_t*)w, bias, bias_is_f32, out, out_stride, m, n, k, mode,
                            (hipStream_t)stream, fold, workspace, workspace_bytes > 0 ? (size_t)workspace_bytes : 0);
#else
    axk_set_error("gemm: packed matrices exist only in the bfloat16 build");
    return -1;
#endif
  }
  AXK_REQUIRE(fold == nullptr, "gemm: a norm follows only products with a packed matrix");
  return launch_fma((const elem_t*)x, x_stride, (const elem_t*)w, bias, bias_is_f32, out, out_stride, m, n, k, mode,
                    (hipStream_t)stream);
}

extern "C" long axk_gemm_workspace(int m, int n, int k, int mode) {
#if AXON_BF16
  return m > 0 && n > 0 && k > 0 ? (long)gemm_workspace_bytes(m, n, k, mode) : 0;
#else
  return 0;
#endif
}

extern "C" int axk_gemm(const void* x, int x_stride, const void* w, int w_packed, const void* bias, int bias_is_f32,
                        void* out, int out_stride, int m, int n, int k, int mode, void* workspace, long workspace_bytes,
                        void* stream) {
  return gemm_checked(x, x_stride, w, w_packed, bias, bias_is_f32, out, out_stride, m, n, k, mode, nullptr, workspace,
                      workspace_bytes, stream);
}

extern "C" int axk_pack_ok(int rows, int k, int gated) {
#if AXON_BF16
  return gemm_pack_ok(rows, k, gated);
#else
  return 0;   // the 32-bit build multiplies row-major matrices
#endif
}

extern "C" long axk_packed_elems(int rows, int k) { return (long)((rows + 15) / 16 * 16) * k; }

extern "C" int axk_pack_matrix(const void* src, void* dst, int rows, int k, void* stream) {
#if AXON_BF16
  AXK_REQUIRE(gemm_pack_ok(rows, k, 0), "pack_matrix: [%d, %d] cannot be packed", rows, k);
  AXK_REQUIRE(((uintptr_t)src & 15) == 0 && ((uintptr_t)dst & 15) == 0, "pack_matrix: operands must be 16-byte aligned");
  return launch_pack_matrix((const bf16_t*)src, (bf16_t*)dst, rows, k, (hipStream_t)stream);
#else
  axk_set_error("pack_matrix: only in the bfloat16 build");
  return -1;
#endif
}

// Segments K is cut into for a packed [n, k] matrix (gated: n is the width of the output, the
// matrix holds 2 n rows): the order of addition of every product with it.  1 where nothing is packed.
extern "C" int axk_gemm_segments(int n, int k, int gated) {
#if AXON_BF16
  if (n <= 0 || k <= 0 || !gemm_pack_ok(gated ? 2 * n : n, k, gated)) return 1;
  return gemm_segments(gated ? n / 16 : (n + 31) / 32, k);
#else
  return 1;
#endif
}

extern "C" int axk_gemm_then_norm_ok(int m, int n, int k) {
#if AXON_BF16
  return m > 0 && n > 0 && k > 0 && gemm_then_norm_ok(m, n, k);
#else
  return 0;   // the 32-bit build keeps the norm a pass of its own
#endif
}

extern "C" int axk_gemm_then_norm(const void* x, int x_stride, const void* w, const void* bias, int bias_is_f32,
                                  float* out, int out_stride, int m, int n, int k, const void* norm_gain,
                                  int norm_gain_is_f32, float norm_eps, void* norm_values, void* workspace,
                                  long workspace_bytes, void* stream) {
  AXK_REQUIRE(axk_gemm_then_norm_ok(m, n, k), "gemm: M=%d N=%d K=%d does not run with K split: the norm stays apart", m,
              n, k);
  AXK_REQUIRE(norm_gain && norm_values, "gemm: the norm behind the product needs its gain and its output");
  AXK_REQUIRE(out_stride % 4 == 0 && ((uintptr_t)out & 15) == 0 && ((uintptr_t)norm_values & 7) == 0,
              "gemm: the rows to add into must be 16-byte aligned (stride %d) and the norm's output 8-byte aligned",
              out_stride);
  const GemmNormFold fold = {norm_gain, norm_gain_is_f32, norm_values, norm_eps};
  return gemm_checked(x, x_stride, w, 1, bias, bias_is_f32, out, out_stride, m, n, k, MODE_ADD_F32, &fold, workspace,
                      workspace_bytes, stream);
}

extern "C" int axk_gemm_qkv_rope_ok(int m, int n, int k, int head_dim, int rotary_dim) {
#if AXON_BF16
  return n > 0 && k > 0 && head_dim > 0 && gemm_qkv_rope_ok(m, n, k, head_dim, rotary_dim);
#else
  return 0;   // the 32-bit build keeps the product, the rotation and the store apart
#endif
}

extern "C" int axk_gemm_qkv_rope(const void* x, int x_stride, const void* w, const void* bias, int bias_is_f32,
                                 void* qkv, int qkv_stride, int m, int k, const float* table, const int32_t* positions, const int32_t* seq_rows,
                                 const int32_t* block_table, int table_stride, void* k_cache, void* v_cache,
                                 int n_heads, int n_kv_heads, int head_dim, int page_size, int write_kv, void* workspace,
                                 long workspace_bytes, void* stream) {
#if AXON_BF16
  AXK_REQUIRE(n_heads > 0 && n_kv_heads > 0 && page_size > 0 && head_dim > 0, "gemm_qkv_rope: heads %d/%d of %d, page %d",
              n_heads, n_kv_heads, head_dim, page_size);
  const int n = (n_heads + (write_kv ? 2 * n_kv_heads : 0)) * head_dim;
  AXK_REQUIRE(axk_gemm_qkv_rope_ok(m, n, k, head_dim, head_dim), "gemm_qkv_rope: M=%d N=%d K=%d head_dim=%d are not taken",
              m, n, k, head_dim);
  AXK_REQUIRE(x_stride >= k && x_stride % 8 == 0 && qkv_stride >= n_heads * head_dim && qkv_stride % 4 == 0 &&
                  ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0 && ((uintptr_t)qkv & 7) == 0 &&
                  ((uintptr_t)table & 15) == 0,
              "gemm_qkv_rope: strides x=%d qkv=%d or the alignment of an operand are not taken", x_stride, qkv_stride);
  AXK_REQUIRE(table && positions && (!write_kv || (seq_rows && block_table && k_cache && v_cache)),
              "gemm_qkv_rope: a table, the positions or the cache is missing");
  return launch_gemm_qkv_rope((const bf16_t*)x, x_stride, (const bf16_t*)w, bias, bias_is_f32, (bf16_t*)qkv, qkv_stride,
                              m, n, k, table, positions, seq_rows, block_table, table_stride,
                              (bf16_t*)k_cache, (bf16_t*)v_cache, n_heads, n_kv_heads, head_dim, page_size, workspace,
                              workspace_bytes > 0 ? (size_t)workspace_bytes : 0, (hipStream_t)stream);
#else
  axk_set_error("gemm_qkv_rope: only in the bfloat16 build");
  return -1;
#endif
}

// ---------------------------------------------------------------------------- the norm inside the product
// Few rows (a decoding step): the gated product and the [q; k; v] product read the float32 rows
// themselves and apply the RMS norm on the way (the norm kernel's arithmetic, the same bits), so
// the norm is no launch of its own.  `ok` depends on the sizes alone.
extern "C" int axk_gemm_normed_ok(int m, int n, int k, int gated) {
#if AXON_BF16
  if (m <= 0 || n <= 0 || k <= 0 || !gemm_pack_ok(gated ? 2 * n : n, k, gated)) return 0;
  return gemm_normed_ok(m, k);
#else
  return 0;   // the 32-bit build keeps the norm a pass of its own
#endif
}

extern "C" int axk_gemm_normed_glu(const float* rows, int rows_stride, const void* gain, int gain_is_f32, float eps,
                                   const void* w, void* out, int out_stride, int m, int n, int k, void* stream) {
#if AXON_BF16
  AXK_REQUIRE(axk_gemm_normed_ok(m, n, k, 1), "gemm_normed_glu: M=%d N=%d K=%d are not taken", m, n, k);
  AXK_REQUIRE(!gain_is_f32, "gemm_normed_glu: the gain must be bfloat16");
  AXK_REQUIRE(rows && gain && w && out, "gemm_normed_glu: an operand is missing");
  AXK_REQUIRE(rows_stride >= k && rows_stride % 4 == 0 && out_stride >= n && ((uintptr_t)rows & 15) == 0 &&
                  ((uintptr_t)gain & 15) == 0 && ((uintptr_t)w & 15) == 0,
              "gemm_normed_glu: strides rows=%d out=%d or the alignment of an operand are not taken", rows_stride, out_stride);
  return launch_gemm_normed_glu(rows, rows_stride, (const bf16_t*)gain, eps, (const bf16_t*)w, (bf16_t*)out, out_stride, m, n,
                                k, (hipStream_t)stream);
#else
  axk_set_error("gemm_normed_glu: only in the bfloat16 build");
  return -1;
#endif
}

extern "C" int axk_gemm_normed_qkv_rope(const float* rows, int rows_stride, const void* gain, int gain_is_f32, float eps,
                                        const void* w, const void* bias, int bias_is_f32, void* qkv, int qkv_stride, int m,
                                        int k, const float* table, const int32_t* positions, const int32_t* seq_rows,
                                        const int32_t* block_table, int table_stride, void* k_cache, void* v_cache,
                                        int n_heads, int n_kv_heads, int head_dim, int page_size, int write_kv, void* stream) {
#if AXON_BF16
  AXK_REQUIRE(n_heads > 0 && n_kv_heads > 0 && page_size > 0 && head_dim > 0,
              "gemm_normed_qkv_rope: heads %d/%d of %d, page %d", n_heads, n_kv_heads, head_dim, page_size);
  const int n = (n_heads + (write_kv ? 2 * n_kv_heads : 0)) * head_dim;
  AXK_REQUIRE(axk_gemm_normed_ok(m, n, k, 0) && axk_gemm_qkv_rope_ok(m, n, k, head_dim, head_dim),
              "gemm_normed_qkv_rope: M=%d N=%d K=%d head_dim=%d are not taken", m, n, k, head_dim);
  AXK_REQUIRE(rows && gain && w && qkv, "gemm_normed_qkv_rope: an operand is missing");
  AXK_REQUIRE(!gain_is_f32, "gemm_normed_qkv_rope: the gain must be bfloat16");
  AXK_REQUIRE(rows_stride >= k && rows_stride % 4 == 0 && qkv_stride >= n_heads * head_dim && qkv_stride % 4 == 0 &&
                  ((uintptr_t)rows & 15) == 0 && ((uintptr_t)gain & 15) == 0 && ((uintptr_t)w & 15) == 0 &&
                  ((uintptr_t)qkv & 7) == 0 && ((uintptr_t)table & 15) == 0,
              "gemm_normed_qkv_rope: strides rows=%d qkv=%d or the alignment of an operand are not taken", rows_stride,
              qkv_stride);
  AXK_REQUIRE(table && positions && (!write_kv || (seq_rows && block_table && k_cache && v_cache)),
              "gemm_normed_qkv_rope: a table, the positions or the cache is missing");
  return launch_gemm_normed_qkv_rope(rows, rows_stride, (const bf16_t*)gain, eps, (const bf16_t*)w, bias, bias_is_f32,
                                     (bf16_t*)qkv, qkv_stride, m, n, k, table, positions, seq_rows, block_table, table_stride,
                                     (bf16_t*)k_cache, (bf16_t*)v_cache, n_heads, n_kv_heads, head_dim, page_size,
                                     (hipStream_t)stream);
#else
  axk_set_error("gemm_normed_qkv_rope: only in the bfloat16 build");
  return -1;
#endif
}
