// Routing for a mixture of experts: the `top` largest of a token's router logits, their softmax,
// and the (token, chosen expert) pairs listed expert by expert in tiles of up to 16 rows, which
// the grouped product takes as its work list.  Everything stays on the device: the launches of a
// step depend on the number of tokens alone.
#include <type_traits>

#include "api.h"
#include "common.h"

namespace {

// One thread per token.  The largest logit first; of equal logits the lower expert.  Weights:
// exp(z - z_first) over the sum of these, added in the order chosen.
__global__ void route_topk_kernel(const float* __restrict__ logits, int n_tokens, int n_experts, int top,
                                  int32_t* __restrict__ experts, float* __restrict__ weights) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tokens) return;
  const float* z = logits + (long)t * n_experts;
  int32_t* chosen = experts + (long)t * top;
  float* w = weights + (long)t * top;
  float first = 0.0f, sum = 0.0f;
  for (int k = 0; k < top; ++k) {
    int best = -1;
    float best_z = 0.0f;
    for (int e = 0; e < n_experts; ++e) {
      bool taken = false;
      for (int j = 0; j < k; ++j) taken |= chosen[j] == e;
      if (taken) continue;
      const float v = z[e];
      if (best < 0 || v > best_z) { best = e; best_z = v; }
    }
    chosen[k] = best;
    if (k == 0) first = best_z;
    const float p = expf(best_z - first);
    w[k] = p;
    sum += p;
  }
  for (int k = 0; k < top; ++k) w[k] = w[k] / sum;
}

// The same choice by a wave per token (up to 1,024 experts: lane l holds the logits of experts l, l + 64, ...):
// `top` times the largest logit not yet taken, by a butterfly over (logit, lower expert first).
__global__ void route_topk_wave_kernel(const float* __restrict__ logits, int n_tokens, int n_experts, int top,
                                       int32_t* __restrict__ experts, float* __restrict__ weights) {
  const int t = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64, lane = threadIdx.x & 63;
  if (t >= n_tokens) return;
  float z[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = lane + 64 * i < n_experts ? logits[(long)t * n_experts + lane + 64 * i] : -INFINITY;
  unsigned taken = 0;
  float first = 0.0f, sum = 0.0f, mine = 0.0f;        // lane k keeps the k-th weight
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int e = lane + 64 * i;
      if (e < n_experts && !(taken >> i & 1) && (at == 0x7fffffff || z[i] > best)) { best = z[i]; at = e; }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float other = __shfl_xor(best, off, 64);
      const int other_at = __shfl_xor(at, off, 64);
      if (other_at != 0x7fffffff && (at == 0x7fffffff || other > best || (other == best && other_at < at))) { best = other; at = other_at; }
    }
    if ((at & 63) == lane) taken |= 1u << (at >> 6);
    if (k == 0) first = best;
    const float p = expf(best - first);
    sum += p;
    if (lane == k % 64) { mine = p; experts[(long)t * top + k] = at; }
  }
  if (lane < top) weights[(long)t * top + lane] = mine / sum;
}

// Scores of every expert: s_e = sigmoid(z_e), which do not compete, or (SOFTMAX) the softmax over all of them; the choice is made by s_e + correction_e (if given),
// the weights come from s_e alone.  The experts form `groups` equal groups of neighbours; a group's
// score is the sum of its two largest choice scores (of its one, if it has one expert), only experts
// of the `keep` best groups can be chosen (of equal groups the lower), and among those the `top`
// largest choice scores win (of equal ones the lower expert).  weights_k = s_k / (sum of the chosen s,
// added in the order chosen, + 1e-20) * scale, or without `normalize` the score itself times scale.  Rows of
// logits are logits_stride apart (further columns may hold other products of the same input).  A wave per token: lane l holds experts l, l + 64, ...
// (up to 1,024) and, for the groups' scores, walks group l (up to 64 groups).
template <bool SOFTMAX>
__global__ void route_scored_wave_kernel(const float* __restrict__ logits, long logits_stride, const float* __restrict__ correction,
                                         int n_tokens, int n_experts, int top, int groups, int keep, float scale, int normalize,
                                         int32_t* __restrict__ experts, float* __restrict__ weights) {
  const int t = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64, lane = threadIdx.x & 63;
  if (t >= n_tokens) return;
  const float* z = logits + (long)t * logits_stride;
  const int size = n_experts / groups;
  float z_most = 0.0f, z_share = 1.0f;
  if (SOFTMAX) {
    z_most = -INFINITY;
    for (int e = lane; e < n_experts; e += 64) z_most = fmaxf(z_most, z[e]);
    z_most = wave_max(z_most);
    float total = 0.0f;
    for (int e = lane; e < n_experts; e += 64) total += expf(z[e] - z_most);
    z_share = 1.0f / wave_sum(total);
  }
  auto score = [&](int e) { return SOFTMAX ? expf(z[e] - z_most) * z_share : 1.0f / (1.0f + expf(-z[e])); };
  unsigned long long kept = ~0ull;
  if (groups > 1) {
    float first = -INFINITY, second = -INFINITY;
    if (lane < groups)
      for (int e = lane * size; e < (lane + 1) * size; ++e) {
        const float c = score(e) + (correction ? correction[e] : 0.0f);
        if (c > first) { second = first; first = c; }
        else if (c > second) second = c;
      }
    const float mine = size > 1 ? first + second : first;
    int ahead = 0;                                   // groups that rank before this lane's
    for (int g = 0; g < groups; ++g) {
      const float other = __shfl(mine, g, 64);
      ahead += (other > mine || (other == mine && g < lane)) ? 1 : 0;
    }
    kept = __ballot(lane < groups && ahead < keep);
  }
  float choice[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int e = lane + 64 * i;
    choice[i] = -INFINITY;
    if (e < n_experts && (kept >> (e / size) & 1)) choice[i] = score(e) + (correction ? correction[e] : 0.0f);
  }
  unsigned taken = 0;
  float sum = 0.0f, mine = 0.0f;                     // lane k keeps the k-th score
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int e = lane + 64 * i;
      if (e < n_experts && (kept >> (e / size) & 1) && !(taken >> i & 1) && (at == 0x7fffffff || choice[i] > best)) { best = choice[i]; at = e; }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float other = __shfl_xor(best, off, 64);
      const int other_at = __shfl_xor(at, off, 64);
      if (other_at != 0x7fffffff && (at == 0x7fffffff || other > best || (other == best && other_at < at))) { best = other; at = other_at; }
    }
    if ((at & 63) == lane) taken |= 1u << (at >> 6);
    const float s = score(at);
    sum += s;
    if (lane == k % 64) { mine = s; experts[(long)t * top + k] = at; }
  }
  if (lane < top) weights[(long)t * top + lane] = normalize ? (mine / (sum + 1e-20f)) * scale : mine * scale;
}

// One block.  pairs p = t top + k in expert order -> sorted [n_pairs], with the token of each
// (sorted_tokens); tiles [.][3] = (expert, first place in sorted, count <= tile_rows), *n_tiles of them; if given,
// the same rows in tiles of wide_rows too (wide_tiles, *n_wide of them).
// Which place a pair gets inside its expert's stretch is not fixed (atomic counters); no result
// depends on it: every row of a product is a chain of its own.  Pairs whose expert is n_experts or more (an
// identity, which has no matrices) are not listed.
// Bound by its waits: the first KEPT pairs a thread are read at once and keep the place that counting them gave, so that they
// are neither read nor counted again; the experts' stretches and tiles are summed up by all threads, in as many steps as there are experts
// for; and the lists are put in order in LDS where they fit (`staged`), since two scattered words a pair are as many lines.  us, two counts a
// pair, one thread for the stretches and scattered words / here: 2,048 tokens, 4 of 32 13.2 / 8.2, 6 of 64 21.9 / 8.3, 8 of 64 (too many to be
// staged) 26.8 / 16.5.  Few pairs want no more places than they are (8 tokens, 2 of 8, 2.4 / 3.8 with sixteen of them and six steps each of three
// sums / 2.3 here; 4 of 32 4.3 / 3.8 / 2.5): one, four or sixteen a thread.
#define SORT_THREADS 1024
#define SORT_KEPT 16
template <int KEPT>
__global__ void __launch_bounds__(SORT_THREADS)
route_sort_kernel(const int32_t* __restrict__ experts, int n_pairs, int n_experts, int top, int32_t* __restrict__ sorted,
                  int32_t* __restrict__ sorted_tokens, int32_t* __restrict__ tiles, int32_t* __restrict__ n_tiles,
                  int32_t* __restrict__ place_of, int32_t* __restrict__ first_of, int tile_rows, int32_t* __restrict__ wide_tiles,
                  int32_t* __restrict__ n_wide, int wide_rows, bool staged) {
  extern __shared__ int counts[];              // [n_experts] counts, [n_experts] where a stretch begins, [n_experts] next free places, staged: [n_pairs]
  __shared__ int waves[3][SORT_THREADS / AXON_WAVE], all;
  int *first = counts + n_experts, *next = first + n_experts;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int expert[KEPT], rank[KEPT];
#pragma unroll
  for (int i = 0; i < KEPT; ++i) expert[i] = tid + SORT_THREADS * i < n_pairs ? experts[tid + SORT_THREADS * i] : n_experts;
  for (int e = tid; e < n_experts; e += SORT_THREADS) counts[e] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < KEPT; ++i)
    if (expert[i] < n_experts) rank[i] = atomicAdd(&counts[expert[i]], 1);
  __syncthreads();
  const bool more = n_pairs > SORT_THREADS * KEPT;
  if (more) {
    for (int e = tid; e < n_experts; e += SORT_THREADS) next[e] = counts[e];
    __syncthreads();
    for (int p = tid + SORT_THREADS * KEPT; p < n_pairs; p += SORT_THREADS)
      if (experts[p] < n_experts) atomicAdd(&counts[experts[p]], 1);
    __syncthreads();
  }
  // a thread's neighbouring experts; pairs, tiles and wide tiles before them
  const int each = (n_experts + SORT_THREADS - 1) / SORT_THREADS, e0 = min(tid * each, n_experts), e1 = min(e0 + each, n_experts);
  int sums[3] = {0, 0, 0}, before[3];
  for (int e = e0; e < e1; ++e) {
    sums[0] += counts[e];
    sums[1] += (counts[e] + tile_rows - 1) / tile_rows;
    sums[2] += (counts[e] + wide_rows - 1) / wide_rows;
  }
  int upto[3] = {sums[0], sums[1], sums[2]};
  for (int off = 1; off < 64 && off < n_experts; off <<= 1) {      // (of fewer experts the lanes behind them are not asked)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int other = __shfl_up(upto[k], off, 64);
      upto[k] += lane >= off ? other : 0;
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) before[k] = upto[k] - sums[k];
  if (n_experts > 64) {                        // (else the first wave has them all)
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (lane == 63) waves[k][wave] = upto[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k)
      for (int w = 0; w < wave; ++w) before[k] += waves[k][w];
  }
  for (int e = e0; e < e1; ++e) {
    const int n = counts[e];
    first[e] = before[0];
    if (more) next[e] += before[0];
    if (first_of) first_of[e] = before[0];
    for (int i = 0; i < n; i += tile_rows, ++before[1]) {
      tiles[3 * before[1]] = e; tiles[3 * before[1] + 1] = before[0] + i; tiles[3 * before[1] + 2] = min(tile_rows, n - i);
    }
    if (wide_tiles)
      for (int i = 0; i < n; i += wide_rows, ++before[2]) {
        wide_tiles[3 * before[2]] = e; wide_tiles[3 * before[2] + 1] = before[0] + i; wide_tiles[3 * before[2] + 2] = min(wide_rows, n - i);
      }
    before[0] += n;
  }
  if (tid == (n_experts > 64 ? SORT_THREADS : n_experts) - 1) {       // (its experts are the last, or it has none)
    *n_tiles = before[1];
    if (wide_tiles) *n_wide = before[2];
    if (first_of) first_of[n_experts] = before[0];
    all = before[0];
  }
  __syncthreads();
  const int listed = all;
  int* order = next + n_experts;
  auto put = [&](int p, int place) {
    if (staged) {
      order[place] = p;
    } else {
      sorted[place] = p;
      sorted_tokens[place] = p / top;
    }
    if (place_of) place_of[p] = place;
  };
#pragma unroll
  for (int i = 0; i < KEPT; ++i)
    if (expert[i] < n_experts) put(tid + SORT_THREADS * i, first[expert[i]] + rank[i]);
  for (int p = tid + SORT_THREADS * KEPT; p < n_pairs; p += SORT_THREADS)
    if (experts[p] < n_experts) put(p, atomicAdd(&next[experts[p]], 1));
  if (!staged) return;
  __syncthreads();
  for (int i = tid; i < listed; i += SORT_THREADS) {
    const int p = order[i];
    sorted[i] = p;
    sorted_tokens[i] = p / top;
  }
}

// y[t, :] (+)= sum_k weights[t, k] rows[row of pair t top + k, :], k ascending; a pair's row is the pair
// itself, or place_of[pair]; without weights the rows are added as they are.  extra (or null): a further
// row a token, added last, times sigmoid(extra_gate[t extra_gate_stride]) if a gate is given.  input (or null): a pair
// whose expert (experts[pair]) is n_experts or more is an identity, its row is input[t, :].
// G neighbouring columns a thread (4 where width and addresses allow), the rows of four, two and then one pair asked for together:
// one after another, each waited for where its row lies and then for the row.
// Four pairs and a further row of 2,048 columns, us, so / here: 2,126 tokens 31.3 / 19.4, 2,048 21.9 / 14.6, 8 4.7 / 4.6.
template <int G>
__global__ void __launch_bounds__(256)
route_combine_kernel(const float* __restrict__ rows, const float* __restrict__ weights, float* __restrict__ y,
                     int top, int width, int accumulate, const int32_t* __restrict__ place_of,
                     const float* __restrict__ extra, const float* __restrict__ extra_gate, long extra_gate_stride,
                     const int32_t* __restrict__ experts, int n_experts, const elem_t* __restrict__ input,
                     long input_stride) {
  const int t = blockIdx.y;
  const int c = G * (blockIdx.x * blockDim.x + threadIdx.x);
  if (c >= width) return;
  auto load = [&](const float* from, float (&v)[G]) {
    if constexpr (G == 4) {
      const float4 q = *reinterpret_cast<const float4*>(from);
      v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
      v[0] = from[0];
    }
  };
  float acc[G], more[G];
  if (accumulate) load(y + (long)t * width + c, acc);
  if (extra) load(extra + (long)t * width + c, more);
  if (!accumulate) {
#pragma unroll
    for (int e = 0; e < G; ++e) acc[e] = 0.0f;
  }
  const float gate = extra && extra_gate ? extra_gate[(long)t * extra_gate_stride] : 0.0f;
  auto add = [&](int first, auto how_many) {
    constexpr int PAIRS = decltype(how_many)::value;
    const long pair = (long)t * top + first;
    float row[PAIRS][G], weight[PAIRS];
    long at[PAIRS];
    bool own[PAIRS];                   // the pair's row is the token's input
#pragma unroll
    for (int j = 0; j < PAIRS; ++j) {
      own[j] = input && experts[pair + j] >= n_experts;
      at[j] = place_of ? (long)place_of[pair + j] : pair + j;
      weight[j] = weights ? weights[pair + j] : 1.0f;
    }
#pragma unroll
    for (int j = 0; j < PAIRS; ++j) {
      if (own[j]) {
#pragma unroll
        for (int e = 0; e < G; ++e) row[j][e] = to_float(input[(long)t * input_stride + c + e]);
      } else {
        load(rows + at[j] * width + c, row[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < PAIRS; ++j)
#pragma unroll
      for (int e = 0; e < G; ++e) acc[e] = weights ? fmaf(weight[j], row[j][e], acc[e]) : acc[e] + row[j][e];
  };
  int k = 0;
  for (; k + 4 <= top; k += 4) add(k, std::integral_constant<int, 4>());
  if (k + 2 <= top) {
    add(k, std::integral_constant<int, 2>());
    k += 2;
  }
  if (k < top) add(k, std::integral_constant<int, 1>());
  if (extra) {
    const float share = 1.0f / (1.0f + expf(-gate));
#pragma unroll
    for (int e = 0; e < G; ++e) acc[e] = extra_gate ? fmaf(share, more[e], acc[e]) : acc[e] + more[e];
  }
  float* to = y + (long)t * width + c;
  if constexpr (G == 4) *reinterpret_cast<float4*>(to) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  else to[0] = acc[0];
}

// out[r, :] = x[rows[r], :] (rows of the compute dtype).
__global__ void gather_rows_kernel(const elem_t* __restrict__ x, long x_stride, const int32_t* __restrict__ rows,
                                   elem_t* __restrict__ out, int width) {
  const elem_t* src = x + (long)rows[blockIdx.x] * x_stride;
  elem_t* dst = out + (long)blockIdx.x * width;
  for (int i = threadIdx.x; i < width; i += blockDim.x) dst[i] = src[i];
}

}  // namespace

extern "C" int axk_route_topk(const float* logits, int n_tokens, int n_experts, int top, int32_t* experts, float* weights,
                              void* stream) {
  AXK_REQUIRE(n_tokens >= 0 && n_experts > 0 && top > 0 && top <= n_experts, "route_topk: %d tokens, %d of %d experts",
              n_tokens, top, n_experts);
  if (n_tokens == 0) return 0;
  if (n_experts <= 1024 && top <= 64) {
    route_topk_wave_kernel<<<ceil_div(n_tokens, 4), 256, 0, (hipStream_t)stream>>>(logits, n_tokens, n_experts, top, experts, weights);
    AXK_LAUNCH_CHECK("route_topk");
    return 0;
  }
  route_topk_kernel<<<ceil_div(n_tokens, 64), 64, 0, (hipStream_t)stream>>>(logits, n_tokens, n_experts, top, experts, weights);
  AXK_LAUNCH_CHECK("route_topk");
  return 0;
}

extern "C" int axk_route_scored(const float* logits, long logits_stride, const float* correction, int n_tokens, int n_experts,
                                int top, int groups, int keep, float scale, int normalize, int softmax, int32_t* experts, float* weights,
                                void* stream) {
  AXK_REQUIRE(logits_stride >= n_experts, "route_scored: rows of %ld logits for %d experts", logits_stride, n_experts);
  AXK_REQUIRE(n_tokens >= 0 && n_experts > 0 && n_experts <= 1024 && top > 0 && top <= 64,
              "route_scored: %d tokens, %d of %d experts (at most 64 of 1024)", n_tokens, top, n_experts);
  AXK_REQUIRE(groups >= 1 && groups <= 64 && n_experts % groups == 0 && keep >= 1 && keep <= groups &&
              (long)keep * (n_experts / groups) >= top,
              "route_scored: %d of %d groups of %d experts for %d a token", keep, groups, n_experts / (groups > 0 ? groups : 1), top);
  if (n_tokens == 0) return 0;
  auto kernel = softmax ? route_scored_wave_kernel<true> : route_scored_wave_kernel<false>;
  kernel<<<ceil_div(n_tokens, 4), 256, 0, (hipStream_t)stream>>>(logits, logits_stride, correction, n_tokens, n_experts, top, groups,
                                                                 keep, scale, normalize, experts, weights);
  AXK_LAUNCH_CHECK("route_scored");
  return 0;
}

extern "C" int axk_route_max_tiles(int n_pairs, int n_experts, int tile_rows) {
  return ceil_div(n_pairs, tile_rows > 0 ? tile_rows : 16) + n_experts;
}

extern "C" int axk_gather_rows(const void* x, long x_stride, const int32_t* rows, void* out, int n_rows, int width, void* stream) {
  AXK_REQUIRE(n_rows >= 0 && width > 0 && x_stride >= width, "gather_rows: %d rows of %d (stride %ld)", n_rows, width, x_stride);
  if (n_rows == 0) return 0;
  gather_rows_kernel<<<n_rows, 256, 0, (hipStream_t)stream>>>((const elem_t*)x, x_stride, rows, (elem_t*)out, width);
  AXK_LAUNCH_CHECK("gather_rows");
  return 0;
}

extern "C" int axk_route_sort(const int32_t* experts, int n_pairs, int n_experts, int top, int32_t* sorted,
                              int32_t* sorted_tokens, int32_t* tiles, int32_t* n_tiles, int32_t* place_of, int32_t* first_of,
                              int tile_rows, int32_t* wide_tiles, int32_t* n_wide, int wide_rows, void* stream) {
  AXK_REQUIRE(n_pairs >= 0 && n_experts > 0 && top > 0 && n_experts <= 4096 && tile_rows > 0,
              "route_sort: %d pairs, %d experts, tiles of %d", n_pairs, n_experts, tile_rows);
  AXK_REQUIRE((wide_tiles == nullptr) == (n_wide == nullptr) && (wide_tiles == nullptr || wide_rows > 0),
              "route_sort: a second list of tiles (of %d) comes with its length", wide_rows);
  const long lists = 3l * n_experts * (long)sizeof(int), order = (long)n_pairs * (long)sizeof(int);
  const bool staged = n_pairs > SORT_THREADS && lists + order <= 60 * 1024;       // (a launch gets 64 KB unasked)
  auto kernel = n_pairs <= SORT_THREADS ? route_sort_kernel<1> : n_pairs <= 4 * SORT_THREADS ? route_sort_kernel<4> : route_sort_kernel<SORT_KEPT>;
  kernel<<<1, SORT_THREADS, lists + (staged ? order : 0), (hipStream_t)stream>>>(
      experts, n_pairs, n_experts, top, sorted, sorted_tokens, tiles, n_tiles, place_of, first_of, tile_rows, wide_tiles, n_wide,
      wide_tiles ? wide_rows : tile_rows, staged);
  AXK_LAUNCH_CHECK("route_sort");
  return 0;
}

extern "C" int axk_route_combine(const float* rows, const float* weights, float* y, int n_tokens, int top, int width,
                                 int accumulate, const int32_t* place_of, const float* extra, const float* extra_gate,
                                 long extra_gate_stride, const int32_t* experts, int n_experts, const void* input, long input_stride,
                                 void* stream) {
  AXK_REQUIRE(n_tokens >= 0 && top > 0 && width > 0 && n_tokens <= 65535, "route_combine: T=%d top=%d width=%d", n_tokens, top,
              width);
  AXK_REQUIRE(input == nullptr || (experts != nullptr && input_stride >= width), "route_combine: identities need the chosen experts and rows of %d", width);
  if (n_tokens == 0) return 0;
  const bool vec = width % 4 == 0 && (((uintptr_t)rows | (uintptr_t)y | (uintptr_t)extra) & 15) == 0;
  auto kernel = vec ? route_combine_kernel<4> : route_combine_kernel<1>;
  // (few tokens: blocks of a wave, so that a token's columns are on several CUs)
  const int threads = vec && n_tokens < 256 ? 64 : 256;
  kernel<<<dim3(ceil_div(width, (vec ? 4 : 1) * threads), n_tokens), threads, 0, (hipStream_t)stream>>>(
      rows, weights, y, top, width, accumulate, place_of, extra, extra_gate, extra_gate_stride, experts, n_experts,
      (const elem_t*)input, input_stride);
  AXK_LAUNCH_CHECK("route_combine");
  return 0;
}
