// Grouped products: many small matrices, each applied to its own rows or its own columns.
//
//   out[orow(r), g ogs + n] = epilogue( sum_k X[xrow(r), g xgs + k] W[g][n][k] + bias[g][n] )
//
// Two ways of saying which rows meet which matrix:
//   * block-diagonal (tiles == null): every row r < M goes through every group g < G, group g
//     reading its own slice of the row's columns (a recurrent layer's gates per block of channels,
//     a per-head projection of an attention layer);
//   * routed (tiles given, on the device): the rows are listed per group in tiles of up to 16
//     (group, first row, count); xrow / orow name the row of X a listed row reads and the row of
//     out it writes (a mixture of experts: rows are (token, chosen expert) pairs in expert order).
//     The grid is launched for the most tiles there can be; blocks beyond *n_tiles leave at once.
//
// Epilogues: bias; a gated linear unit with clamps (W holds 2 N rows a group, gate rows then up
// rows: g = min(gate, limit), u = clamp(up, -limit, limit), out = g sigmoid(alpha g) (u + shift); an
// infinite limit, alpha 1 and shift 0 give silu(gate) up); a multiplication by sigmoid(gate[orow, g ogs + n]),
// or by sigmoid(gate[orow, g]), one number a group; a factor a row on X (row_scale[orow], float32: the sums are
// multiplied by it before bias and unit, as if the row of X had been); out in float32 or in the compute dtype.
//
// The K-reduction of one output is one chain in ascending k that depends on K and the build alone
// (32-bit FMA, or 16x16x32 MFMAs where the bfloat16 build can use them: K a multiple of 32 and
// 16-byte aligned rows), never on which other rows share the tile.
#include <type_traits>

#include "api.h"
#include "common.h"
#include "instances.h"

namespace {

struct GroupedArgs {
  const void* x; int x_is_f32; long x_row_stride; long x_group_stride; const int32_t* x_rows;
  const elem_t* w; const void* bias; int bias_is_f32;
  void* out; int out_is_f32; long out_row_stride; long out_group_stride; const int32_t* out_rows;
  const float* gate; long gate_row_stride; int gate_per_group;
  const float* row_scale;
  int glu; float glu_limit; float glu_alpha; float glu_shift;
  const int32_t* tiles; const int32_t* n_tiles;
  int M, N, K, G;
  bool vec_out;                         // four neighbouring outputs are one aligned store
  bool by_tile;                         // a list of 64-row tiles is gone through tile by tile (axk_grouped_gemm_by_tile)
};

#define GG_ROWS 16
#define GG_COLS 64
#define GG_BK 32

__device__ inline float gg_load_x(const GroupedArgs& a, long at) {
  return a.x_is_f32 ? ((const float*)a.x)[at] : to_float(((const elem_t*)a.x)[at]);
}

__device__ inline float clamped_glu(float gate, float up, float limit, float alpha, float shift) {
  const float g = fminf(gate, limit);
  const float u = fminf(fmaxf(up, -limit), limit);
  return (g * (1.0f / (1.0f + expf(-(alpha * g))))) * (u + shift);
}

__device__ inline float gg_value(const GroupedArgs& a, int g, int orow, int n, float v, float up) {
  if (a.row_scale) {                    // the row of X counts row_scale[orow] times: the product is linear in it
    const float w = a.row_scale[orow];
    v *= w;
    up *= w;
  }
  if (a.bias) {
    const int per = a.glu ? 2 * a.N : a.N;
    v += load_vec(a.bias, a.bias_is_f32, g * per + n);
    if (a.glu) up += load_vec(a.bias, a.bias_is_f32, g * per + a.N + n);
  }
  if (a.glu) v = clamped_glu(v, up, a.glu_limit, a.glu_alpha, a.glu_shift);
  if (a.gate) v = v * (1.0f / (1.0f + expf(-a.gate[(long)orow * a.gate_row_stride + (a.gate_per_group ? g : (long)g * a.out_group_stride + n)])));
  return v;
}

__device__ inline void gg_store(const GroupedArgs& a, int g, int orow, int n, float v, float up) {
  v = gg_value(a, g, orow, n, v, up);
  const long at = (long)orow * a.out_row_stride + (long)g * a.out_group_stride + n;
  if (a.out_is_f32) ((float*)a.out)[at] = v;
  else ((elem_t*)a.out)[at] = from_float(v);
}

// which rows and which group this block works on; false: nothing
__device__ inline bool gg_tile(const GroupedArgs& a, int& g, int& first, int& count) {
  if (a.tiles) {
    if ((int)blockIdx.x >= *a.n_tiles) return false;
    g = a.tiles[3 * blockIdx.x];
    first = a.tiles[3 * blockIdx.x + 1];
    count = a.tiles[3 * blockIdx.x + 2];
  } else {
    g = blockIdx.z;
    first = blockIdx.x * GG_ROWS;
    count = min(GG_ROWS, a.M - first);
  }
  return count > 0;
}

// 16 rows x 64 columns at a time in a block of 256 threads: thread (ty, tx) owns rows 4 ty .. 4 ty + 3 of
// column tx.  A listed tile of more than 16 rows (a list made for the tiles of 64) is walked 16 rows at a time.
template <bool GLU>
__global__ void __launch_bounds__(256) grouped_gemm_fma_kernel(GroupedArgs a) {
  __shared__ float xs[GG_ROWS][GG_BK + 1];
  __shared__ float ws[GG_COLS][GG_BK + 1];
  __shared__ float us[GLU ? GG_COLS : 1][GG_BK + 1];
  __shared__ int xrow[GG_ROWS], orow[GG_ROWS];
  int g, tile_first, tile_count;
  if (!gg_tile(a, g, tile_first, tile_count)) return;
  const int tid = threadIdx.x, tx = tid & 63, ty = tid >> 6;
  const int n0 = blockIdx.y * GG_COLS;
  const int w_rows = GLU ? 2 * a.N : a.N;
  const elem_t* wg = a.w + (long)g * w_rows * a.K;
  for (int done = 0; done < tile_count; done += GG_ROWS) {
    const int first = tile_first + done, count = min(GG_ROWS, tile_count - done);
    __syncthreads();
    if (tid < GG_ROWS) {
      const int r = first + min(tid, count - 1);
      xrow[tid] = a.x_rows ? a.x_rows[r] : r;
      orow[tid] = a.out_rows ? a.out_rows[r] : r;
    }
    __syncthreads();
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f}, acc_up[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k0 = 0; k0 < a.K; k0 += GG_BK) {
      for (int i = tid; i < GG_ROWS * GG_BK; i += 256) {
        const int r = i / GG_BK, kk = i % GG_BK;
        xs[r][kk] = (r < count && k0 + kk < a.K)
                        ? gg_load_x(a, (long)xrow[r] * a.x_row_stride + (long)g * a.x_group_stride + k0 + kk) : 0.0f;
      }
      for (int i = tid; i < GG_COLS * GG_BK; i += 256) {
        const int c = i / GG_BK, kk = i % GG_BK;
        const bool ok = n0 + c < a.N && k0 + kk < a.K;
        ws[c][kk] = ok ? to_float(wg[(long)(n0 + c) * a.K + k0 + kk]) : 0.0f;
        if (GLU) us[c][kk] = ok ? to_float(wg[(long)(a.N + n0 + c) * a.K + k0 + kk]) : 0.0f;
      }
      __syncthreads();
#pragma unroll
      for (int kk = 0; kk < GG_BK; ++kk) {
        const float b = ws[tx][kk];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(xs[ty * 4 + i][kk], b, acc[i]);
        if (GLU) {
          const float bu = us[tx][kk];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc_up[i] = fmaf(xs[ty * 4 + i][kk], bu, acc_up[i]);
        }
      }
      __syncthreads();
    }
    const int n = n0 + tx;
    if (n < a.N) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = ty * 4 + i;
        if (r < count) gg_store(a, g, orow[r], n, acc[i], acc_up[i]);
      }
    }
  }
}

#if AXON_BF16
typedef __attribute__((ext_vector_type(8))) __bf16 gg_bf16x8;
typedef __attribute__((ext_vector_type(4))) float gg_f32x4;

__device__ inline gg_bf16x8 gg_frag(uint4 v) { return __builtin_bit_cast(gg_bf16x8, v); }

// Columns n .. n + 3 of a row (what a lane holds of a product).
__device__ inline void gg_store4(const GroupedArgs& a, int g, int orow, int n, const gg_f32x4& v, const gg_f32x4& up) {
  if (!a.vec_out || n + 4 > a.N) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (n + c < a.N) gg_store(a, g, orow, n + c, v[c], up[c]);
    return;
  }
  float r[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) r[c] = gg_value(a, g, orow, n + c, v[c], up[c]);
  const long at = (long)orow * a.out_row_stride + (long)g * a.out_group_stride + n;
  if (a.out_is_f32) *reinterpret_cast<float4*>((float*)a.out + at) = make_float4(r[0], r[1], r[2], r[3]);
  else *reinterpret_cast<uint2*>((bf16_t*)a.out + at) = make_uint2(pack2_bf16(r[0], r[1]), pack2_bf16(r[2], r[3]));
}

// 16 rows x 64 columns a block of four waves, a wave 16 columns: W rows as the MFMA's first
// operand, X rows as its second, both straight from memory (lane l holds row l % 16, the eight k
// from 8 (l / 16)); lane l ends with row l % 16 of the columns 4 (l / 16) .. + 3.  Such a product waits for W
// alone, and an output is one chain over k, so a wave keeps RING steps of 32 k under way: each is asked
// for again as soon as it is multiplied.  Rows and columns that do not exist read ones that do.  The 32 pairs
// of 8 tokens over 32 experts of [1,408, 2,048] and [2,048, 704]: 42 and 19 us, launches included (120 and 45 with four steps
// asked for at a time and waited for together).
template <bool GLU, bool XF32, int RING>
__global__ void __launch_bounds__(256) grouped_gemm_mfma_kernel(GroupedArgs a) {
  int g, first, count;
  if (!gg_tile(a, g, first, count)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = blockIdx.y * GG_COLS + wave * 16;
  if (n0 >= a.N) return;
  const int r = lane & 15, kq = (lane >> 4) * 8;
  const int rr = first + min(r, count - 1);
  const int xr = a.x_rows ? a.x_rows[rr] : rr;
  const int orow = a.out_rows ? a.out_rows[rr] : rr;
  const long x_at = (long)xr * a.x_row_stride + (long)g * a.x_group_stride + kq;
  const int w_rows = GLU ? 2 * a.N : a.N;
  const bf16_t* wrow = a.w + ((long)g * w_rows + min(n0 + r, a.N - 1)) * a.K + kq;
  const bf16_t* urow = wrow + (long)a.N * a.K;
  gg_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, acc_up = {0.0f, 0.0f, 0.0f, 0.0f};
  uint4 xf[RING][XF32 ? 2 : 1], wf[RING], uf[GLU ? RING : 1];
  auto ask = [&](int s, int k) {
    if (XF32) {
      xf[s][0] = *reinterpret_cast<const uint4*>((const float*)a.x + x_at + k);
      xf[s][XF32 ? 1 : 0] = *reinterpret_cast<const uint4*>((const float*)a.x + x_at + k + 4);
    } else {
      xf[s][0] = *reinterpret_cast<const uint4*>((const bf16_t*)a.x + x_at + k);
    }
    wf[s] = *reinterpret_cast<const uint4*>(wrow + k);
    if (GLU) uf[GLU ? s : 0] = *reinterpret_cast<const uint4*>(urow + k);
  };
  auto multiply = [&](int s) {
    uint4 x = xf[s][0];
    if (XF32) {
      const float4 lo = __builtin_bit_cast(float4, xf[s][0]), hi = __builtin_bit_cast(float4, xf[s][XF32 ? 1 : 0]);
      x = make_uint4(pack2_bf16(lo.x, lo.y), pack2_bf16(lo.z, lo.w), pack2_bf16(hi.x, hi.y), pack2_bf16(hi.z, hi.w));
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gg_frag(wf[s]), gg_frag(x), acc, 0, 0, 0);
    if (GLU) acc_up = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gg_frag(uf[GLU ? s : 0]), gg_frag(x), acc_up, 0, 0, 0);
  };
  // (a step behind the last asks for the last again: a branch would have every load under way waited for)
#pragma unroll
  for (int s = 0; s < RING; ++s) ask(s, min(32 * s, a.K - 32));
  int k0 = 0;
  for (; k0 + 32 * RING <= a.K; k0 += 32 * RING) {
#pragma unroll
    for (int s = 0; s < RING; ++s) {
      multiply(s);
      ask(s, min(k0 + 32 * (RING + s), a.K - 32));
    }
  }
#pragma unroll
  for (int s = 0; s < RING; ++s)
    if (k0 + 32 * s < a.K) multiply(s);
  if (r >= count) return;
  gg_store4(a, g, orow, n0 + (lane >> 4) * 4, acc, acc_up);
}

// Many rows a group (a long prompt's pairs of an expert, the tokens of a prompt through a block of
// channels): 64 rows x 128 or 256 rows of W a block, through two stages of 64 k of LDS that are filled by direct loads
// (X in float32: through registers, where it is rounded).  Four waves, each all or half of the 64 rows x 64 rows of W
// (up to 4 x 4 products a step of 32 k); with the gated epilogue a wave's 64 rows of W are 32 gate rows and the 32
// up rows of the same columns.  The next stage is on its way while this one is multiplied, and the two halves
// of a stage are read one ahead of the products.  Rows of a stage are 128 bytes, their 16-byte slots permuted by
// slot ^ (row / 2 % 8): the 16 rows a read takes at a time fall into 16 different slots of the 64 banks.  The chain of an
// output is the one of the kernel above (16x16x32 products in ascending k), so which of the two runs changes no
// bit.  2,048 tokens, 4 of 32 experts of [1,408, 2,048] and [2,048, 704]: 81 and 57 us (163 and 113 with stages of 32 k
// through registers, by columns).
#define GT_ROWS 64
#define GT_BK 64
#define GT_STAGE(wrows) ((GT_ROWS + (wrows)) * GT_BK * 2)
typedef const __attribute__((address_space(1))) void* gg_global_t;
typedef __attribute__((address_space(3))) void* gg_lds_t;
template <bool GLU, bool XF32, int WROWS>
__global__ void __launch_bounds__(256, 2) grouped_gemm_tile_kernel(GroupedArgs a) {
  static_assert(WROWS == 128 || (WROWS == 256 && GLU), "a wave's 64 rows of W, for half or for all of the rows of X");
  constexpr int STAGE = GT_STAGE(WROWS), XT = WROWS / 64, WL = WROWS / 32;   // tiles of 16 rows a wave, load instructions of W a wave
  extern __shared__ __align__(256) unsigned char stages[];        // [2]: X [64][64], W [WROWS][64]
  constexpr int COLS = GLU ? WROWS / 2 : WROWS;
  // Blocks go to the eight XCDs in turn: each XCD gets a run of neighbours of the list [group, columns, rows]
  // (routed: [columns, tile]), so that the tiles of a group that read the same rows of W do so through one L2; or, by_tile, of the list
  // [tile, columns]: an XCD has a tile with all of its columns, so that its rows of X and of the output stay there.
  const int col_tiles = (a.N + COLS - 1) / COLS, row_tiles = a.tiles ? *a.n_tiles : (a.M + GT_ROWS - 1) / GT_ROWS;
  const long total = (long)row_tiles * col_tiles * (a.tiles ? 1 : a.G), share = (total + 7) / 8;
  const long item = (long)(blockIdx.x % 8) * share + blockIdx.x / 8;
  if ((long)(blockIdx.x / 8) >= share || item >= total) return;
  const bool by_tile = !GLU && a.by_tile;
  const int row_tile = (int)(by_tile ? item / col_tiles : item % row_tiles);
  const int n0 = (int)(by_tile ? item % col_tiles : item / row_tiles % col_tiles) * COLS;
  int g, first, count;
  if (a.tiles) {
    g = a.tiles[3 * row_tile]; first = a.tiles[3 * row_tile + 1]; count = a.tiles[3 * row_tile + 2];
  } else {
    g = (int)(item / row_tiles / col_tiles); first = row_tile * GT_ROWS; count = min(GT_ROWS, a.M - first);
  }
  if (count <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w_rows = GLU ? 2 * a.N : a.N;
  const bf16_t* wg = a.w + (long)g * w_rows * a.K;
  // a load instruction fills 8 rows: lane l row l / 8, slot l % 8.  A wave brings WROWS / 4 rows of W and 16 of X.
  const int lrow = lane >> 3, lslot = lane & 7;
  const int w_wave = WROWS == 256 ? wave : wave & 1, x_wave = WROWS == 256 ? 0 : 32 * (wave >> 1);   // what it multiplies
  long w_at[WL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int row = 8 * WL * wave + 8 * i + lrow;                                // of the stage's W
    const int col = GLU ? n0 + 32 * (row >> 6) + (row & 31) : n0 + row;
    w_at[i] = (long)(min(col, a.N - 1) + (GLU && (row & 32) ? a.N : 0)) * a.K + 8 * (lslot ^ (4 * (i & 1) + (lane >> 4)));
  }
  long x_at[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = first + min(16 * wave + 8 * i + lrow, count - 1);
    x_at[i] = (long)(a.x_rows ? a.x_rows[r] : r) * a.x_row_stride + (long)g * a.x_group_stride + 8 * (lslot ^ (4 * (i & 1) + (lane >> 4)));
  }
  // the last 32 k of a K that is no multiple of 64: the slots behind them bring the ones before again (not used)
  auto tail = [&](int k0, int i) {
    const int chunk = lslot ^ (4 * (i & 1) + (lane >> 4));
    return k0 + GT_BK > a.K && chunk >= 4 ? k0 - 32 : k0;
  };
  uint4 held[XF32 ? 4 : 1];
  auto ask = [&](int k0, int which) {
    unsigned char* st = stages + which * STAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (XF32) {
        const float* src = (const float*)a.x + x_at[i] + tail(k0, i);
        held[XF32 ? 2 * i : 0] = *reinterpret_cast<const uint4*>(src);
        held[XF32 ? 2 * i + 1 : 0] = *reinterpret_cast<const uint4*>(src + 4);
      } else {
        __builtin_amdgcn_global_load_lds((gg_global_t)((const bf16_t*)a.x + x_at[i] + tail(k0, i)),
                                         (gg_lds_t)(st + (16 * wave + 8 * i) * 128), 16, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < WL; ++i)
      __builtin_amdgcn_global_load_lds((gg_global_t)(wg + w_at[i] + tail(k0, i)),
                                       (gg_lds_t)(st + (GT_ROWS + 8 * WL * wave + 8 * i) * 128), 16, 0, 0);
  };
  auto place_x = [&](int which) {                  // float32 rows, rounded, where a direct load would have put them
    if (!XF32) return;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float4 lo = __builtin_bit_cast(float4, held[XF32 ? 2 * i : 0]), hi = __builtin_bit_cast(float4, held[XF32 ? 2 * i + 1 : 0]);
      *reinterpret_cast<uint4*>(stages + which * STAGE + (16 * wave + 8 * i) * 128 + 16 * lane) =
          make_uint4(pack2_bf16(lo.x, lo.y), pack2_bf16(lo.z, lo.w), pack2_bf16(hi.x, hi.y), pack2_bf16(hi.z, hi.w));
    }
  };
  gg_f32x4 acc[XT][4];
#pragma unroll
  for (int i = 0; i < XT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = gg_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int fr = lane & 15, q = lane >> 4;
  const unsigned lds0 = (unsigned)(size_t)(gg_lds_t)stages;
  const unsigned at = lds0 + fr * 128 + ((q ^ (fr >> 1)) << 4);
  const unsigned x_read = at + x_wave * 128, w_read = at + (GT_ROWS + 64 * w_wave) * 128;
  const int n_steps = (a.K + GT_BK - 1) / GT_BK;
  ask(0, 0);
  for (int t = 0; t < n_steps; ++t) {
    place_x(t & 1);
    wait_vmcnt<0>();
    __syncthreads();                               // this stage is there, and the other one's readers are done
    if (t + 1 < n_steps) ask((t + 1) * GT_BK, (t + 1) & 1);
    const unsigned xr = x_read + (t & 1) * STAGE, wr = w_read + (t & 1) * STAGE;
    u32x4 xf[2][XT], wf[2][4];
    read_frags<XT, 2048>(xf[0], xr);
    read_frags<4, 2048>(wf[0], wr);
    read_frags<XT, 2048>(xf[1], xr ^ 64);          // (no branch between a read and its wait: the halves a short K lacks are read too)
    read_frags<4, 2048>(wf[1], wr ^ 64);
    wait_lgkmcnt<XT + 4>();
    use_frags<XT>(xf[0]);
    use_frags<4>(wf[0]);
#pragma unroll
    for (int i = 0; i < XT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gg_bf16x8, wf[0][j]), __builtin_bit_cast(gg_bf16x8, xf[0][i]),
                                                            acc[i][j], 0, 0, 0);
    wait_lgkmcnt<0>();
    use_frags<XT>(xf[1]);
    use_frags<4>(wf[1]);
    if (t * GT_BK + 32 < a.K) {
#pragma unroll
      for (int i = 0; i < XT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gg_bf16x8, wf[1][j]), __builtin_bit_cast(gg_bf16x8, xf[1][i]),
                                                              acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < XT; ++i) {
    const int r = x_wave + 16 * i + fr;
    if (r >= count) continue;
    const int orow = a.out_rows ? a.out_rows[first + r] : first + r;
#pragma unroll
    for (int j = 0; j < (GLU ? 2 : 4); ++j)
      gg_store4(a, g, orow, n0 + (GLU ? 32 : 64) * w_wave + 16 * j + 4 * q, acc[i][j], acc[i][GLU ? j + 2 : j]);
  }
}

// The gated product of more rows still: 128 rows x 256 rows of W a block of eight waves, each 64 x 64 (a wave's 64 rows of W are 32 gate rows
// and the up rows of the same columns).  Stages of 64 k as above, three of them (144 KB, a block a CU): a step's fragments are in
// registers when it begins, the next step's are read behind its first products, and a stage's loads go out between the products of the
// stage two before it.  The chains are the same.  Lists of tiles of 128 rows, K a multiple of 64, X in the compute dtype.
// Waves whose 64 rows a tile lacks only bring operands.  Bound by LDS, which is filled and read for 1,400 cycles a stage of 1,024 cycles of
// products, and by what the last round leaves idle: 256 blocks take 36 us at K 2,048 (0.97 PFLOP/s).  us, tiles of 64 rows / here: 4 of 32
// experts of [1,408, 2,048], 2,048 tokens 82 / 71 (104 / 84 in a step, which reads W from HBM), 4,096 151 / 133; 6 of 64 of [2,816,
// 4,096], 2,048 tokens 480 / 420, 256 288 / 265; 2 of 16 of [5,632, 4,096], 2,048 tokens 328 / 269.  Products that are not gated lose with
// short K (4 of 32 of [2,048, 704] 56 / 70: nobody multiplies while a block stores).
#define GW_ROWS 128
#define GW_COLS 256                                    // rows of W
#define GW_STAGES 3
#define GW_STAGE ((GW_ROWS + GW_COLS) * GT_BK * 2)
__global__ void __launch_bounds__(512, 1) grouped_gemm_wide_kernel(GroupedArgs a) {
  constexpr int COLS = GW_COLS / 2, LOADS = (GW_ROWS + GW_COLS) / 64;       // load instructions of a wave and stage
  extern __shared__ __align__(256) unsigned char stages[];        // [3]: X [128][64], W [256][64]
  const int col_tiles = (a.N + COLS - 1) / COLS, row_tiles = *a.n_tiles;
  const long total = (long)row_tiles * col_tiles, share = (total + 7) / 8, item = (long)(blockIdx.x % 8) * share + blockIdx.x / 8;
  if ((long)(blockIdx.x / 8) >= share || item >= total) return;       // (the order of blocks: as above)
  const int row_tile = (int)(item % row_tiles), n0 = (int)(item / row_tiles) * COLS;
  const int g = a.tiles[3 * row_tile], first = a.tiles[3 * row_tile + 1], count = a.tiles[3 * row_tile + 2];
  if (count <= 0) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 2, wn = wave & 3;
  const bf16_t* wg = a.w + (long)g * 2 * a.N * a.K;
  // a load instruction fills 8 rows: lane l row l / 8, slot l % 8; a wave's i-th the rows 8 (8 i + wave) and on, of X and then of W
  const int lrow = lane >> 3, chunk = (lane & 7) ^ (4 * (wave & 1) + (lane >> 4));
  const bf16_t* from[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    if (i < GW_ROWS / 64) {
      const int r = first + min(8 * (8 * i + wave) + lrow, count - 1);
      from[i] = (const bf16_t*)a.x + (long)(a.x_rows ? a.x_rows[r] : r) * a.x_row_stride + (long)g * a.x_group_stride + 8 * chunk;
    } else {
      const int row = 8 * (8 * (i - GW_ROWS / 64) + wave) + lrow;
      from[i] = wg + (long)(min(n0 + 32 * (row >> 6) + (row & 31), a.N - 1) + (row & 32 ? a.N : 0)) * a.K + 8 * chunk;
    }
  }
  auto ask = [&](int t, int i) {
    __builtin_amdgcn_global_load_lds((gg_global_t)(from[i] + t * GT_BK), (gg_lds_t)(stages + t % GW_STAGES * GW_STAGE + (8 * i + wave) * 1024), 16, 0, 0);
  };
  const int n_stages = a.K / GT_BK;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) ask(0, i);
  if (n_stages > 1) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) ask(1, i);
    wait_vmcnt<LOADS>();
  } else {
    wait_vmcnt<0>();
  }
  __builtin_amdgcn_s_barrier();                        // stage 0 is there for every wave
  if (64 * wm >= count) {                              // nothing to multiply: its share of the loads, and the barriers
    for (int t = 0; t + 1 < n_stages; ++t) {
      if (t + 2 < n_stages) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) ask(t + 2, i);
        wait_vmcnt<LOADS>();
      } else {
        wait_vmcnt<0>();
      }
      __builtin_amdgcn_s_barrier();
    }
    return;
  }
  gg_f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = gg_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int fr = lane & 15, q = lane >> 4;
  const unsigned lds0 = (unsigned)(size_t)(gg_lds_t)stages;
  const unsigned at = lds0 + fr * 128 + ((q ^ (fr >> 1)) << 4);
  const unsigned x_read = at + wm * 64 * 128, w_read = at + (GW_ROWS + 64 * wn) * 128;
  u32x4 xf[2][4], wf[2][4];
  read_frags<4, 2048>(xf[0], x_read);
  read_frags<4, 2048>(wf[0], w_read);
  wait_lgkmcnt<0>();
  use_frags<4>(xf[0]);
  use_frags<4>(wf[0]);
  // A stage's two steps.  NEXT: there is one behind it; ASKS: and one behind that, whose place nobody reads any more.
  auto stage = [&](int t, auto next_of, auto asks_of) {
    constexpr bool NEXT = decltype(next_of)::value, ASKS = decltype(asks_of)::value;
    const unsigned here = t % GW_STAGES * GW_STAGE, behind = (t + 1) % GW_STAGES * GW_STAGE;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (half == 1 && NEXT) {
        if (ASKS) wait_vmcnt<LOADS>();
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_barrier();                  // the next stage is there for every wave; nobody reads the one before this one
      }
      const unsigned xr = half ? x_read + behind : (x_read ^ 64) + here, wr = half ? w_read + behind : (w_read ^ 64) + here;
#pragma unroll
      for (int p = 0; p < 16; ++p) {
        const int i = p / 4, j = p % 4;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gg_bf16x8, wf[half][j]), __builtin_bit_cast(gg_bf16x8, xf[half][i]),
                                                            acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (half == 0 || NEXT) {
          if (p < 4) lds_read16_step<2048, 4>(xf[half ^ 1][p % 4], xr, p);
          else if (p < 8) lds_read16_step<2048, 4>(wf[half ^ 1][p % 4], wr, p - 4);
        }
        if (ASKS && half == 0 && p % 2 == 1 && p / 2 < LOADS) ask(t + 2, p / 2);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (half == 0 || NEXT) {
        wait_lgkmcnt<0>();
        use_frags<4>(xf[half ^ 1]);
        use_frags<4>(wf[half ^ 1]);
      }
    }
  };
  int t = 0;
  for (; t + 2 < n_stages; ++t) stage(t, std::true_type(), std::true_type());
  if (t + 1 < n_stages) stage(t++, std::true_type(), std::false_type());
  stage(t, std::false_type(), std::false_type());
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 64 * wm + 16 * i + fr;
    if (r >= count) continue;
    const int orow = a.out_rows ? a.out_rows[first + r] : first + r;
#pragma unroll
    for (int j = 0; j < 2; ++j) gg_store4(a, g, orow, n0 + 32 * wn + 16 * j + 4 * q, acc[i][j], acc[i][j + 2]);
  }
}

int launch_wide(const GroupedArgs& a, dim3 grid, hipStream_t s) {
  constexpr int lds = GW_STAGES * GW_STAGE;
  static_assert(lds <= 160 * 1024, "the stages do not fit the LDS of a CU");
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&grouped_gemm_wide_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      axk_set_error("grouped_gemm: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  AXK_INSTANCE(INST_GROUPED_GEMM, 5, 1);
  grouped_gemm_wide_kernel<<<grid, 512, lds, s>>>(a);
  return 0;
}

template <bool GLU, bool XF32, int WROWS>
int launch_tile(const GroupedArgs& a, dim3 grid, hipStream_t s) {
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&grouped_gemm_tile_kernel<GLU, XF32, WROWS>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 2 * GT_STAGE(WROWS));
    if (e != hipSuccess) {
      axk_set_error("grouped_gemm: cannot reserve %d bytes of LDS: %s", 2 * GT_STAGE(WROWS), hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  AXK_INSTANCE(INST_GROUPED_GEMM, WROWS == 256 ? 2 : 3, GLU);
  grouped_gemm_tile_kernel<GLU, XF32, WROWS><<<grid, 256, 2 * GT_STAGE(WROWS), s>>>(a);
  return 0;
}
#endif

}  // namespace

extern "C" int axk_grouped_gemm_uses_mfma(int k, int x_is_f32, long x_row_stride, long x_group_stride) {
#if AXON_BF16
  const int per16 = x_is_f32 ? 4 : 8;     // elements of X in 16 bytes
  return k % 32 == 0 && x_row_stride % per16 == 0 && x_group_stride % per16 == 0;
#else
  return 0;
#endif
}

// Whether a list of 64-row tiles is gone through tile by tile: not gated, where a group's W is no more than three of an XCD's L2 of 4 MB.
// A tile that meets all of a larger W reads it from further away, again for each tile.  us, by columns / by tile: 4 of 32 experts
// [2,048, 704] (2.9 MB) of 2,048 tokens 63.8 / 57.3, of 4,096 115 / 108, 8 of 64 [2,048, 256] (1 MB) 73.5 / 66.6, 2 of 8 [2,048, 1,408]
// (5.8 MB) 51.0 / 42.0, 6 of 64 166 / 164, 4 of 16 [1,024, 1,024] 43.5 / 34.3; 2 of 16 [4,096, 1,408] (11.5 MB) 106 / 104, [4,096, 2,816]
// (23 MB) 188 / 207, of 4,096 tokens 325 / 388, of 512 91 / 86, 2 of 8 [4,096, 14,336] (117 MB) 797 / 1,090.  Gated, whose W is twice as large for its columns:
// 4 of 32 [1,408, 2,048] 78 / 80, 2 of 16 [2,816, 4,096] 171 / 202.
extern "C" int axk_grouped_gemm_by_tile(int n, int k, int glu) {
  return !glu && (size_t)n * k * sizeof(elem_t) <= (12u << 20);
}

// Whether a gated routed product takes a list of tiles of 128 rows: where those of 64 are more than a round of two blocks a CU (an
// expert's last tile half full).  us, 64 / 128 rows: 4 of 32 experts of [1,408, 2,048] of 1,024 tokens (480 blocks) 45 / 62, of
// 2,048 (864) 82 / 71; 6 of 64 of [2,816, 4,096] of 256 (616) 288 / 265; 2 of 16 of [5,632, 4,096] of 256 (352) 150 / 160, of 512 (528) 203 / 168;
// 2 of 8 of [2,048, 1,024] of 1,024 (288) 21 / 23, of 2,048 (544) 42 / 37; 8 of 64 of [512, 512] of 2,048 (576) 33.5 / 32.7.
extern "C" int axk_grouped_gemm_wide(int pairs, int groups, int n, int k) {
#if AXON_BF16
  return k % GT_BK == 0 && (long)(pairs / 64 + groups / 2) * ceil_div(n, 128) > 512;
#else
  return 0;
#endif
}

extern "C" int axk_grouped_gemm(const void* x, int x_is_f32, long x_row_stride, long x_group_stride, const int32_t* x_rows,
                                const void* w, const void* bias, int bias_is_f32, void* out, int out_is_f32,
                                long out_row_stride, long out_group_stride, const int32_t* out_rows, const float* gate,
                                long gate_row_stride, int gate_per_group, const float* row_scale, int glu, float glu_limit,
                                float glu_alpha, float glu_shift, const int32_t* tiles,
                                const int32_t* n_tiles, int max_tiles, int tile_rows, int m, int n, int k, int groups,
                                void* stream) {
  AXK_REQUIRE(m >= 0 && n > 0 && k > 0 && groups > 0, "grouped_gemm: bad sizes M=%d N=%d K=%d groups=%d", m, n, k, groups);
  AXK_REQUIRE((tiles == nullptr) == (n_tiles == nullptr) && (tiles == nullptr || max_tiles >= 0),
              "grouped_gemm: a list of tiles comes with its length and the most tiles there can be");
  AXK_REQUIRE(tiles != nullptr || (x_rows == nullptr && out_rows == nullptr),
              "grouped_gemm: rows are named only beside a list of tiles");
  AXK_REQUIRE(tile_rows == 16 || tile_rows == 64 || (tile_rows == 128 && tiles != nullptr), "grouped_gemm: tiles of %d rows (16, 64 or 128)", tile_rows);
  const int row_tiles = tiles ? max_tiles : ceil_div(m, GG_ROWS);
  if (row_tiles == 0) return 0;
  AXK_REQUIRE(groups <= 65535 && ceil_div(n, GG_COLS) <= 65535, "grouped_gemm: %d groups of %d columns are too many", groups, n);
  GroupedArgs a{x, x_is_f32, x_row_stride, x_group_stride, x_rows, (const elem_t*)w, bias, bias_is_f32, out, out_is_f32,
                out_row_stride, out_group_stride, out_rows, gate, gate_row_stride, gate_per_group, row_scale, glu, glu_limit, glu_alpha,
                glu_shift, tiles, n_tiles,
                m, n, k, groups,
                out_row_stride % 4 == 0 && out_group_stride % 4 == 0 && (uintptr_t)out % (out_is_f32 ? 16 : 8) == 0,
                tiles != nullptr && axk_grouped_gemm_by_tile(n, k, glu)};
  dim3 grid(row_tiles, ceil_div(n, GG_COLS), tiles ? 1 : groups);
  hipStream_t s = (hipStream_t)stream;
#if AXON_BF16
  const bool mfma = axk_grouped_gemm_uses_mfma(k, x_is_f32, x_row_stride, x_group_stride) && ((uintptr_t)x & 15) == 0 &&
                    ((uintptr_t)w & 15) == 0;
  if (mfma && tile_rows == 128) {
    AXK_REQUIRE(glu && !x_is_f32 && k % GT_BK == 0,
                "grouped_gemm: tiles of 128 rows are for gated products of a K of a multiple of 64, not float32 X (K=%d)", k);
    const long blocks = (long)max_tiles * ceil_div(n, GW_COLS / 2);
    AXK_REQUIRE(blocks < (1l << 31) - 8, "grouped_gemm: %ld blocks are more than one launch takes", blocks);
    const dim3 big((unsigned)((blocks + 7) / 8 * 8));
    if (const int rc = launch_wide(a, big, s)) return rc;
    AXK_LAUNCH_CHECK("grouped_gemm");
    return 0;
  }
  AXK_REQUIRE(tile_rows != 128, "grouped_gemm: tiles of 128 rows are the matrix cores' (K a multiple of 64, operands aligned for 16 bytes)");
  // many rows a group: tiles of 64 rows through LDS (a list of tiles says by its tile size which it was made for)
  if (mfma && (tiles ? tile_rows == 64 : m >= 256)) {
    // 128 rows of W a block, three blocks a CU, unless the gated product has two rounds of blocks of 256: those read
    // X half as often, which pays where K is long.  us, 256 rows of W a block against 128: 10 blocks of channels [512, 256] at
    // 256 rows 14.7 / 9.4, at 2,048 38 / 26; 16 heads [512, 128] at 2,048 41 / 27; 4 of 32 experts of 2,048 tokens
    // [2,048, 704] (by columns) 69 / 63, gated [1,408, 2,048] 81 / 85, of 1,024 tokens (576 blocks) 46 / 57, of 512 (384) 44 / 41, of
    // 256 41 / 33; 2 of 8 of 128 tokens gated [1,024, 1,024] 20 / 16; 8 of 64 of 2,048 gated [512, 2,048] 74 / 67.
    const long row_blocks = (long)(tiles ? max_tiles : ceil_div(m, GT_ROWS)) * (tiles ? 1 : groups);
    const bool wide = glu && row_blocks * ceil_div(n, 128) >= 512;
    const long blocks = row_blocks * ceil_div(n, glu && !wide ? 64 : 128);
    AXK_REQUIRE(blocks < (1l << 31) - 8, "grouped_gemm: %ld blocks are more than one launch takes", blocks);
    const dim3 big((unsigned)((blocks + 7) / 8 * 8));
    int rc;
#define TILE(GLU, WROWS) (x_is_f32 ? launch_tile<GLU, true, WROWS>(a, big, s) : launch_tile<GLU, false, WROWS>(a, big, s))
    if (wide) rc = TILE(true, 256);
    else rc = glu ? TILE(true, 128) : TILE(false, 128);
#undef TILE
    if (rc) return rc;
    AXK_LAUNCH_CHECK("grouped_gemm");
    return 0;
  }
  if (mfma) {
    // A K of up to 256 in a ring of four, beside whose registers more waves have room and which asks for little beyond it:
    // 4 groups of [64, 32] at 130 rows 4.7 us with eight, 3.9 with four, 16 of [512, 96] at 255 21 / 13, 8 of 64
    // experts of 128 tokens [2,048, 256] 46 / 37, 16 of [512, 128] at 8 rows 4.5 / 4.7; but 8 of 128 of 4 [1,536, 2,048] 76 / 103.
#define FEW(GLU, RING)                                                                          \
  if (x_is_f32) grouped_gemm_mfma_kernel<GLU, true, RING><<<grid, 256, 0, s>>>(a);              \
  else grouped_gemm_mfma_kernel<GLU, false, RING><<<grid, 256, 0, s>>>(a);
    if (glu) {
      if (k <= 256) { AXK_INSTANCE(INST_GROUPED_GEMM, 4, 1); FEW(true, 4) }
      else { AXK_INSTANCE(INST_GROUPED_GEMM, 1, 1); FEW(true, 8) }
    } else {
      if (k <= 256) { AXK_INSTANCE(INST_GROUPED_GEMM, 4, 0); FEW(false, 4) }
      else { AXK_INSTANCE(INST_GROUPED_GEMM, 1, 0); FEW(false, 8) }
    }
#undef FEW
    AXK_LAUNCH_CHECK("grouped_gemm");
    return 0;
  }
#endif
  if (glu) { AXK_INSTANCE(INST_GROUPED_GEMM, 0, 1); grouped_gemm_fma_kernel<true><<<grid, 256, 0, s>>>(a); }
  else { AXK_INSTANCE(INST_GROUPED_GEMM, 0, 0); grouped_gemm_fma_kernel<false><<<grid, 256, 0, s>>>(a); }
  AXK_LAUNCH_CHECK("grouped_gemm");
  return 0;
}
