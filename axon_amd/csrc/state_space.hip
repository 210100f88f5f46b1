// A selective state-space mixer in its recurrent form (the "state-space duality" layer of Mamba-2-like
// models): per request and head a state S [N, P] of 32-bit floats, carried from token to token,
//   dt_t = softplus(raw_t + dt_bias),  a_t = exp(-exp(A_log) dt_t),
//   S_t = a_t S_(t-1) + dt_t B_t x_t^T,  y_t = S_t^T C_t + D x_t,
// behind a short causal convolution with silu over the channels [x | B | C], and followed by a gate and
// an RMS norm in equal parts.  Head h reads B and C of group h / (heads / groups).
//
// A request's state row holds two copies of (heads N P floats of S, head by head [N][P], then
// [taps - 1][channels] of the convolution's last inputs, oldest first); zeros for a new request, which
// is also what the convolution reads before the first token.  The state behind position p lives in copy
// p & 1: a step whose first position is s reads copy (s - 1) & 1 and writes the copy of its last
// position, so a step of one token never writes what it read and gives the same state and output if it
// is run again (a decoding step is run once before it is captured into a graph).  The tokens of a
// request are contiguous in a step and a request is in a step once, so two tokens belong to one request
// iff their state slots (seq_rows) are equal.  Everything here is 32-bit in both builds but the
// convolution's weights as stored and the normed output.
#include <math.h>

#include "api.h"
#include "common.h"
#include "instances.h"

namespace {

__device__ inline float ss_silu(float z) { return z / (1.0f + expf(-z)); }
__device__ inline float ss_softplus(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

// u[t, c] = act(bias[c] + sum_k w[c, k] in(t - (taps - 1 - k))) for the channels c of x (float32 rows
// x_stride apart): the last column of w is the current token's; inputs before the step come from the state.
// Threads behind the channels work out the heads' step sizes: terms[t, h] = (dt, a) from raw[t, h].
__global__ void state_conv_kernel(const float* __restrict__ x, long x_stride, const elem_t* __restrict__ w,
                                  const void* __restrict__ bias, int bias_is_f32, int silu, const float* __restrict__ state,
                                  long state_stride, long copy_elems, long tail_at, const int32_t* __restrict__ positions,
                                  const int32_t* __restrict__ seq_rows, float* __restrict__ u, int channels, int taps,
                                  const float* __restrict__ raw, long raw_stride, const void* __restrict__ dt_bias,
                                  int dt_bias_is_f32, const void* __restrict__ a_log, int a_log_is_f32,
                                  float* __restrict__ terms, int heads) {
  const int t = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) {
    const int h = c - channels;
    if (h < heads) {
      const float dt = ss_softplus(raw[(long)t * raw_stride + h] + load_vec(dt_bias, dt_bias_is_f32, h));
      terms[((long)t * heads + h) * 2] = dt;
      terms[((long)t * heads + h) * 2 + 1] = expf(-(expf(load_vec(a_log, a_log_is_f32, h)) * dt));
    }
    return;
  }
  const int slot = seq_rows[t];
  // how many earlier tokens of this step belong to the same request (up to taps - 1 matter)
  int inside = 0;
  while (inside < taps - 1 && t - inside - 1 >= 0 && seq_rows[t - inside - 1] == slot) ++inside;
  // the copy behind the position before the request's first of this step
  const int before = (positions[t] - inside + 1) & 1;
  const float* kept = state + (long)slot * state_stride + (long)before * copy_elems + tail_at;      // [taps - 1][channels]
  float acc = 0.0f;
  for (int k = 0; k < taps; ++k) {
    const int back = taps - 1 - k;            // the input `back` tokens before this one
    float v;
    if (back <= inside) v = x[(long)(t - back) * x_stride + c];
    else v = kept[(long)(taps - 1 - (back - inside)) * channels + c];        // the (back - inside)-th last kept input
    acc = fmaf(to_float(w[(long)c * taps + k]), v, acc);
  }
  if (bias) acc += load_vec(bias, bias_is_f32, c);
  u[(long)t * channels + c] = silu ? ss_silu(acc) : acc;
}

// The same for steps of many tokens: a thread has four channels of SS_CONV_RUN tokens, whose inputs it asks for together, each
// once, where a thread a (token, channel) asked for `taps` of them one behind another, each a wait.  Behind a request's start the
// inputs before it come from the state.  The sums of a channel go the same way.
// 2,560 channels of four taps, 32 heads, us, a thread a (token, channel) / here: 192 tokens 5.7 / 6.7, 256 7.3 / 6.8, 512 11.1 / 8.4, 1,024
// 18.8 / 10.4, 2,125 35.3 / 16.0 (in three requests 35.8 / 18.4).
#define SS_CONV_RUN 8
template <int TAPS>
__global__ void __launch_bounds__(128)
state_conv_runs_kernel(const float* __restrict__ x, long x_stride, const elem_t* __restrict__ w, const void* __restrict__ bias,
                       int bias_is_f32, int silu, const float* __restrict__ state, long state_stride, long copy_elems, long tail_at,
                       const int32_t* __restrict__ positions, const int32_t* __restrict__ seq_rows, float* __restrict__ u, int n_tokens,
                       int channels, const float* __restrict__ raw, long raw_stride, const void* __restrict__ dt_bias,
                       int dt_bias_is_f32, const void* __restrict__ a_log, int a_log_is_f32, float* __restrict__ terms, int heads) {
  constexpr int BEFORE = TAPS - 1;
  const int t0 = blockIdx.y * SS_CONV_RUN, quad = blockIdx.x * 128 + threadIdx.x, c = 4 * quad, tokens = min(SS_CONV_RUN, n_tokens - t0);
  if (c >= channels) {
    const int h = quad - channels / 4;
    if (h >= heads) return;
    const float shift = load_vec(dt_bias, dt_bias_is_f32, h), rate = expf(load_vec(a_log, a_log_is_f32, h));
    float in[SS_CONV_RUN];
#pragma unroll
    for (int i = 0; i < SS_CONV_RUN; ++i) in[i] = raw[(long)(t0 + min(i, tokens - 1)) * raw_stride + h];
#pragma unroll
    for (int i = 0; i < SS_CONV_RUN; ++i)
      if (i < tokens) {
        const float dt = ss_softplus(in[i] + shift);
        *reinterpret_cast<float2*>(terms + ((long)(t0 + i) * heads + h) * 2) = make_float2(dt, expf(-(rate * dt)));
      }
    return;
  }
  // the inputs of the tokens t0 - BEFORE .. t0 + SS_CONV_RUN - 1 (the step's first and last again beyond it)
  float4 in[BEFORE + SS_CONV_RUN];
  int slot[BEFORE + SS_CONV_RUN];
#pragma unroll
  for (int i = 0; i < BEFORE + SS_CONV_RUN; ++i) {
    const int t = min(max(t0 + i - BEFORE, 0), n_tokens - 1);
    in[i] = *reinterpret_cast<const float4*>(x + (long)t * x_stride + c);
    slot[i] = t0 + i - BEFORE >= 0 ? seq_rows[t] : -1;
  }
  float taps[4][TAPS], b[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int k = 0; k < TAPS; ++k) taps[e][k] = to_float(w[(long)(c + e) * TAPS + k]);
    b[e] = bias ? load_vec(bias, bias_is_f32, c + e) : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < SS_CONV_RUN; ++i) {
    if (i >= tokens) return;
    int inside = 0;                    // earlier tokens of this step of the same request, up to BEFORE: the same for the block
    bool on = true;
#pragma unroll
    for (int back = 1; back <= BEFORE; ++back) {
      on = on && slot[i + BEFORE - back] == slot[i + BEFORE];
      inside += on ? 1 : 0;
    }
    const float* kept = nullptr;
    if (inside < BEFORE)
      kept = state + (long)slot[i + BEFORE] * state_stride + (long)((positions[t0 + i] - inside + 1) & 1) * copy_elems + tail_at + c;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < TAPS; ++k) {
      const int back = TAPS - 1 - k;
      float v[4];
      if (back <= inside) {
        const float4 q = in[i + BEFORE - back];
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = kept[(long)(BEFORE - (back - inside)) * channels + e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(taps[e][k], v[e], acc[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (bias) acc[e] += b[e];
      acc[e] = silu ? ss_silu(acc[e]) : acc[e];
    }
    *reinterpret_cast<float4*>(u + (long)(t0 + i) * channels + c) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  }
}

// The sum over the sixteen lanes of a row, in every lane of the row, by lane permutations of the adder (pairs,
// quads, halves of the row, the row): a fixed order.
__device__ inline float ss_row_sum(float v) {
#define SS_DPP(val, ctrl) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, val), ctrl, 0xf, 0xf, false))
  v += SS_DPP(v, 0xb1);     // quad_perm [1, 0, 3, 2]
  v += SS_DPP(v, 0x4e);     // quad_perm [2, 3, 0, 1]
  v += SS_DPP(v, 0x141);    // row_half_mirror
  v += SS_DPP(v, 0x140);    // row_mirror
#undef SS_DPP
  return v;
}

// The same sums of four values, in the four quads of a row each: lanes 4 q .. 4 q + 3 end with the sum of value q.  The same
// additions (the two numbers of a step change places), ten of the last eight steps' sixteen instructions fewer, and what follows is
// done once for four values.  The quads that an addition leaves alone are a bit each (bank_mask): as an instruction, since the
// compiler makes two of it, and behind two cycles that a lane permutation wants after its operand is written.
__device__ inline float ss_row_sums_of_four(float a, float b, float c, float d) {
#define SS_DPP(val, ctrl) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, val), ctrl, 0xf, 0xf, false))
  a += SS_DPP(a, 0xb1); b += SS_DPP(b, 0xb1); c += SS_DPP(c, 0xb1); d += SS_DPP(d, 0xb1);     // quad_perm [1, 0, 3, 2]
  a += SS_DPP(a, 0x4e); b += SS_DPP(b, 0x4e); c += SS_DPP(c, 0x4e); d += SS_DPP(d, 0x4e);     // quad_perm [2, 3, 0, 1]
#undef SS_DPP
  float ab, cd, all;                   // halves of a row: of a (and c) in quads 0 and 2, of b (and d) in 1 and 3; then the rows
  asm("s_nop 1\n\t"
      "v_add_f32_dpp %1, %3, %3 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %2, %5, %5 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %1, %4, %4 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %2, %6, %6 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
      "s_nop 0\n\t"
      "v_add_f32_dpp %0, %1, %1 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %0, %2, %2 row_ror:8 row_mask:0xf bank_mask:0xc"
      : "=&v"(all), "=&v"(ab), "=&v"(cd)
      : "v"(a), "v"(b), "v"(c), "v"(d));
  return all;
}

// From the lanes of an even row of sixteen to those of the row behind it; zero in the even rows.
__device__ inline float ss_hand_on(float v) {
  const auto s = __builtin_amdgcn_permlane16_swap(0u, __float_as_uint(v), false, false);     // odd rows of the one, even rows of the other
  const unsigned behind = s[0];
  return __uint_as_float(behind);
}

// A value dim's N rows of the state lie in thirty-two lanes, two halves of sixteen, each with its ROWS rows a lane: lane l of
// half f holds l + 16 (f ROWS + i).  A sum over n is sixteen partial chains l, l + 16, l + 32, ... in ascending n, folded in
// a fixed order: the first half begins each chain, hands it on, and the second half ends it.  OWN: rows a chain has.
template <int OWN>
struct SsRows {
  static constexpr int ROWS = OWN >= 2 ? OWN / 2 : 1;
  static __device__ inline int row(int lane, int i) { return (lane & 15) + 16 * (lane / 16 * ROWS + i); }
  // the chain goes on over this lane's rows (one row a chain: it has none in the second half)
  static __device__ inline float chain(float part, int half, const float (&S)[ROWS], const float (&C)[ROWS]) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const float on = fmaf(S[i], C[i], part);
      part = OWN == 1 && half ? part : on;
    }
    return part;
  }
};

// A request's kept inputs of the convolution behind `count` tokens of this step: of (what was kept, this step's inputs) the
// last taps - 1; place i takes what lies `count` places later (where both copies are one: read before it is written,
// ascending).  By all threads of a block.
__device__ inline void ss_keep_inputs(const float* from, float* to, long tail_at, const float* __restrict__ conv_in,
                                      long conv_in_stride, int first, int count, int channels, int taps) {
  float* kept = to + tail_at;
  const float* kept_from = from + tail_at;
  for (int c = threadIdx.x; c < channels; c += blockDim.x)
    for (int i = 0; i < taps - 1; ++i) {
      const int at = i + count;
      kept[(long)i * channels + c] = at < taps - 1 ? kept_from[(long)at * channels + c]
                                                   : conv_in[(long)(first + at - (taps - 1)) * conv_in_stride + c];
    }
}

// A decoding step.  grid (tokens, heads, blocks of 8 value dims), every token a request of its own in slot seq_rows[t]; a
// block is 256 threads: thirty-two lanes side by side share a value dim p and hold that column of the state (N up to
// 16 OWN rows) as SsRows says.  u [T, channels] = [x: heads P | B: groups N | C: groups N] behind the convolution;
// terms [T, heads, 2] = (dt, a).  y [T, heads P] float32.  The block (head 0, dims 0) also brings the convolution's
// kept inputs up to date from conv_in (the convolution's inputs, float32 rows conv_in_stride apart).  A token's sums do
// not depend on how the request was cut into steps.
#define SS_DIMS 8          // value dims a block
#define SS_LANES 32
#define SS_WALKERS (SS_DIMS * SS_LANES)
template <int OWN>
__global__ void __launch_bounds__(SS_WALKERS)
state_space_step_kernel(const float* __restrict__ u, const float* __restrict__ terms, const void* __restrict__ d_skip,
                        int d_is_f32, float* __restrict__ state, long state_stride, long copy_elems, long tail_at,
                        const int32_t* __restrict__ positions, const int32_t* __restrict__ seq_rows,
                        const float* __restrict__ conv_in, long conv_in_stride, float* __restrict__ y, int heads, int groups,
                        int P, int N, int channels, int taps) {
  typedef SsRows<OWN> Rows;
  constexpr int ROWS = Rows::ROWS;
  const int t = blockIdx.x, h = blockIdx.y, g = h / (heads / groups), slot = seq_rows[t];
  const int lane = threadIdx.x % SS_LANES, half = lane / 16, p = blockIdx.z * SS_DIMS + threadIdx.x / SS_LANES;
  const bool has_p = p < P;
  const int start = positions[t];
  const float* from = state + (long)slot * state_stride + (long)((start + 1) & 1) * copy_elems;
  float* to = state + (long)slot * state_stride + (long)(start & 1) * copy_elems;
  const int inner = heads * P;
  const long s_at = (long)h * N * P, x_col = (long)h * P + (has_p ? p : 0);
  const float* row = u + (long)t * channels;
  const float* B = row + inner + (long)g * N;
  const float* C = B + (long)groups * N;
  const float x = row[x_col], dt = terms[((long)t * heads + h) * 2], a = terms[((long)t * heads + h) * 2 + 1];
  const float dskip = load_vec(d_skip, d_is_f32, h);
  float S[ROWS], Bs[ROWS], Cs[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int n = Rows::row(lane, i), at = min(n, N - 1);      // rows beyond N: zeros in S, what they meet does not count
    S[i] = has_p && n < N ? from[s_at + (long)n * P + p] : 0.0f;
    Bs[i] = B[at];
    Cs[i] = C[at];
  }
  const float dx = dt * x;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) S[i] = Rows::row(lane, i) < N ? fmaf(a, S[i], dx * Bs[i]) : 0.0f;
  const float begun = ss_hand_on(Rows::chain(0.0f, half, S, Cs));
  const float part = ss_row_sum(Rows::chain(begun, half, S, Cs));
  if (lane == 16 && has_p) y[(long)t * inner + x_col] = fmaf(dskip, x, part);
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int n = Rows::row(lane, i);
    if (has_p && n < N) to[s_at + (long)n * P + p] = S[i];
  }
  if (blockIdx.y == 0 && blockIdx.z == 0) ss_keep_inputs(from, to, tail_at, conv_in, conv_in_stride, t, 1, channels, taps);
}

// The walk of stretches of tokens (a request's tokens of the step, or segments of them): the arithmetic and
// the order of the kernel above, its operands through LDS.  The second half of a value dim's lanes is SS_BEHIND tokens behind
// the first: in a turn the first begins the chains of token j while the second ends those of token j - 2, so that both halves
// work in every turn and two neighbouring turns' chains do not wait for each other.
// SS_CHUNK turns' B and C rows, the block's values of x, and (dt, a), each half's of its own token, go to LDS by direct
// loads, a dword a lane, during the first half of the chunk before (one barrier a chunk).  A lane's rows of B and C lie
// there side by side, so that it reads four at a time, conflict-free, the operands of two turns while the two before them
// are worked on.  A lane of the second half keeps the output of the chunk's turn that has its number; one store a chunk,
// while the next chunk is worked on.
// What bounds it: a wave's own instructions and their latency, one token after the other (some 130 ns a turn).  32 heads of 64
// dims, 128 rows, 2 groups, us, with sixteen lanes a value dim and a dword load a row of B and C a token / here: stretches of
// 311, 611 and 1,203 tokens 308 / 196, one chain of 1,024 257 / 137, of 64 26 / 16, two of 1,024 270 / 155, five of 300 166 / 110,
// 32 of a token 44 / 41; 256 rows and 16 heads, 1,024 tokens 390 / 179; a decoding step of 32 tokens 44 / 36 (the kernel
// above).  Slower: one token behind (202 for the three stretches), two chunks ahead instead of one.  Thirty-two chains of half the
// length take 183, but are other sums.
#define SS_CHUNK 16
#define SS_BEHIND 2
template <int OWN>
struct SsChunk {
  static constexpr int QUADS = SsRows<OWN>::ROWS >= 4 ? SsRows<OWN>::ROWS / 4 : 1;        // reads of four of a lane's rows
  static constexpr int PLACES = SS_LANES * QUADS * 4;           // floats a turn's B (or C) takes (fewer than four rows: places unused)
  static constexpr int WAVES = SS_WALKERS / AXON_WAVE, PIECES = PLACES / 64;
  static constexpr int PER = 2 * PIECES / WAVES;                // loads of a wave and turn
  static constexpr int X_AT = SS_CHUNK * 2 * PLACES, TERMS_AT = X_AT + 2 * SS_DIMS * SS_CHUNK, FLOATS = TERMS_AT + 4 * SS_CHUNK;
};

template <int V>
struct SsNumber {
  static constexpr int value = V;
};

template <int OWN>
struct SsStaged {
  u32x4 B[2][SsChunk<OWN>::QUADS], C[2][SsChunk<OWN>::QUADS];
  u32x4 x[1], terms[1];
};

template <int OWN, bool FULL, bool SEGMENTS>
__global__ void __launch_bounds__(SS_WALKERS)
state_space_walk_kernel(const float* __restrict__ u, const float* __restrict__ terms, const void* __restrict__ d_skip,
                        int d_is_f32, float* __restrict__ state, long state_stride, long copy_elems, long tail_at,
                        const int32_t* __restrict__ spans, const int32_t* __restrict__ positions,
                        const float* __restrict__ conv_in, long conv_in_stride, float* __restrict__ y, int heads, int groups,
                        int P, int N, int channels, int taps, const int32_t* __restrict__ segs, float* __restrict__ ends,
                        float* __restrict__ cum) {
  typedef SsChunk<OWN> Chunk;
  typedef SsRows<OWN> Rows;
  constexpr int ROWS = Rows::ROWS, PLACES = Chunk::PLACES, QUADS = Chunk::QUADS, PER = Chunk::PER, WAVES = Chunk::WAVES;
  constexpr int PIECES = Chunk::PIECES, SUB = SS_BEHIND;
  static_assert(WAVES == 4 && 2 * SS_DIMS * SS_CHUNK == WAVES * AXON_WAVE && 4 * SS_CHUNK == AXON_WAVE && PIECES % 2 == 0,
                "who asks for what of a chunk");
  static_assert(SUB == 2 && SS_CHUNK % (2 * SUB) == 0, "a turn's pair goes by the chunk's turn");
  __shared__ __align__(16) float lds[2][Chunk::FLOATS];
  const int* stretch = SEGMENTS ? segs + 4 * blockIdx.x : spans + 3 * blockIdx.x;
  const int slot = stretch[0], first = stretch[1], count = stretch[2];
  const bool from_state = SEGMENTS ? stretch[3] != 0 : true;
  const int h = blockIdx.y, g = h / (heads / groups);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int of_dim = threadIdx.x % SS_LANES, half = of_dim / 16, ns = of_dim & 15;
  const int p = blockIdx.z * SS_DIMS + threadIdx.x / SS_LANES;
  const bool has_p = p < P;
  const int start = positions[first];
  const float* from = state + (long)slot * state_stride + (long)((start + 1) & 1) * copy_elems;
  float* to = state + (long)slot * state_stride + (long)((start + count - 1) & 1) * copy_elems;
  const int inner = heads * P;
  const long s_at = (long)h * N * P, x_col = (long)h * P + (has_p ? p : 0);
  const long b_col = inner + (long)g * N;
  float S[ROWS], second[ROWS];         // the second half has no token in the first turns: its rows' beginning comes after them
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int n = Rows::row(of_dim, i);
    second[i] = from_state && has_p && n < N ? from[s_at + (long)n * P + p] : 0.0f;
    S[i] = half ? 0.0f : second[i];
  }
  const float dskip = load_vec(d_skip, d_is_f32, h);
  const int turns = count + SS_BEHIND;

  // What this lane asks for of a turn: load j of the wave is piece j WAVES + wave of (B's pieces, C's pieces), the c-th 64
  // of the places (quad, lane of the row set, place): the set's lane's row 4 quad + place.  Odd pieces are the second half's,
  // and odd waves ask for odd pieces: their token is an earlier one.
  typedef const __attribute__((address_space(1))) void* from_t;
  typedef __attribute__((address_space(3))) void* to_t;
  unsigned col[PER];                   // in bytes from the row's B
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int piece = j * WAVES + wave, c = piece % PIECES;
    const int at = c * 64 + lane, n = Rows::row(at / 4 % SS_LANES, min(at / (4 * SS_LANES) * 4 + at % 4, ROWS - 1));
    col[j] = (unsigned)((piece < PIECES ? 0 : groups * N) + min(n, N - 1)) * 4u;        // places beyond the state: any row
  }
  // a half's token of a turn (before the first token and behind the last: that one, not used)
  auto token = [&](int turn, int behind) { return max(min(turn - behind * SS_BEHIND, count - 1), 0); };
  // COUNT turns of the chunk that begins with the stretch's turn t0, from its turn k on
  const unsigned row_bytes = (unsigned)channels * 4u;
  const char* rows = (const char*)(u + (long)first * channels + b_col);
  auto ask = [&](int buffer, int t0, int k, auto how_many) {
    constexpr int COUNT = decltype(how_many)::value;
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
      const char* row = rows + (unsigned long)(unsigned)token(t0 + k + i, wave & 1) * row_bytes;
#pragma unroll
      for (int j = 0; j < PER; ++j)
        __builtin_amdgcn_global_load_lds((from_t)(row + col[j]), (to_t)(&lds[buffer][0] + (k + i) * 2 * PLACES + (j * WAVES + wave) * 64), 4, 0, 0);
    }
  };
  // the rest of a chunk: x [half][value dim of the block][turn] (a wave 64 of them), (dt, a) [half][turn] (one wave)
  auto ask_rest = [&](int buffer, int t0) {
    const int pp = blockIdx.z * SS_DIMS + (wave & 1) * (AXON_WAVE / SS_CHUNK) + lane / SS_CHUNK;
    const long tx = first + token(t0 + lane % SS_CHUNK, wave >> 1), tt = first + token(t0 + (lane >> 1) % SS_CHUNK, lane / 32);
    __builtin_amdgcn_global_load_lds((from_t)(u + tx * channels + (long)h * P + min(pp, P - 1)),
                                     (to_t)(&lds[buffer][0] + Chunk::X_AT + wave * AXON_WAVE), 4, 0, 0);
    if (wave == 0)
      __builtin_amdgcn_global_load_lds((from_t)(terms + (tt * heads + h) * 2 + (lane & 1)), (to_t)(&lds[buffer][0] + Chunk::TERMS_AT), 4, 0, 0);
  };
  ask_rest(0, 0);
#pragma unroll
  for (int k = 0; k < SS_CHUNK; ++k)
    if (k < turns) ask(0, 0, k, SsNumber<1>());

  const unsigned lds0 = (unsigned)(size_t)(to_t)&lds[0][0];
  const unsigned bc_at = lds0 + of_dim * 16, terms_at = lds0 + (Chunk::TERMS_AT + half * 2 * SS_CHUNK) * 4;
  const unsigned x_at = lds0 + (Chunk::X_AT + (half * SS_DIMS + threadIdx.x / SS_LANES) * SS_CHUNK) * 4;
  float decay = 1.0f;                  // of a segment: the product of its tokens' a so far (the first half's)
  // lane ns of a half has the chunk's turn 4 (ns % 4) + ns / 4: its sum and its x (of the second half's token)
  const int own_turn = 4 * (ns & 3) + ns / 4;
  float kept_sum = 0.0f, kept_x = 0.0f, kept_decay = 1.0f;      // (kept_decay: of turn ns, the first half's token's)
  float parts[2 * SUB] = {};           // of four turns, before their lanes are added up
  float begun[SUB] = {};               // what the second half was handed

  // the operands of the chunk's turns k0 + pair SUB ..: `pair` is known when compiled
  auto read = [&](SsStaged<OWN>& o, unsigned at, int k0, int pair) {
    const unsigned rows = bc_at + at + k0 * (2 * PLACES * 4);
#pragma unroll
    for (int k = 0; k < SUB; ++k)
#pragma unroll
      for (int q = 0; q < QUADS; ++q) {
        lds_read16_step<16 * SS_LANES, 4 * SUB * QUADS>(o.B[k][q], rows, (pair * SUB + k) * 2 * QUADS + q);
        lds_read16_step<16 * SS_LANES, 4 * SUB * QUADS>(o.C[k][q], rows, (pair * SUB + k) * 2 * QUADS + QUADS + q);
      }
    lds_read16_step<16, 2>(o.terms[0], terms_at + at + k0 * 8, pair);
    lds_read16<0>(o.x[0], x_at + at + k0 * 4);
    __builtin_amdgcn_sched_barrier(0);          // all of them ahead of the work that they are to be hidden behind
  };
  auto arrived = [&](SsStaged<OWN>& o) {
    wait_lgkmcnt<0>();
#pragma unroll
    for (int k = 0; k < SUB; ++k) {
      use_frags<QUADS>(o.B[k]);
      use_frags<QUADS>(o.C[k]);
    }
    use_frags<1>(o.terms);
    use_frags<1>(o.x);
  };
  // the work of SUB turns from the chunk's turn k0 + pair SUB on (left: the chunk's turns in which the first half has a token,
  // from where on its rows stay as they are; WHOLE: it has one in all; begins: the chunk's turn 0 is the stretch's)
  auto work = [&](const SsStaged<OWN>& o, int k0, int pair, int left, bool begins, auto whole) {
    constexpr bool WHOLE = decltype(whole)::value != 0;
    [[maybe_unused]] const int own = ns - k0;          // (of segments)
#pragma unroll
    for (int k = 0; k < SUB; ++k) {
      const int at = pair * SUB + k;
      if (WHOLE || k0 + at < left + SS_BEHIND) {
        const float dt = __uint_as_float(o.terms[0][k * 2]), a = __uint_as_float(o.terms[0][k * 2 + 1]);
        const float x = __uint_as_float(o.x[0][at]);
        const float dx = dt * x;
        float C[ROWS];
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
          const float B = __uint_as_float(o.B[k][i / 4][i % 4]);
          C[i] = __uint_as_float(o.C[k][i / 4][i % 4]);
          const float on = FULL || Rows::row(of_dim, i) < N ? fmaf(a, S[i], dx * B) : 0.0f;
          S[i] = WHOLE || half || k0 + at < left ? on : S[i];
        }
        const float part = Rows::chain(begun[k], half, S, C);
        begun[k] = ss_hand_on(part);
        parts[at] = part;
        if (SEGMENTS) {
          decay *= a;
          kept_decay = own == at ? decay : kept_decay;
        }
        if (at == SS_BEHIND - 1) {
          const bool enters = half && begins && k0 == 0;       // (chosen, not branched to: reads are under way)
#pragma unroll
          for (int i = 0; i < ROWS; ++i) S[i] = enters ? second[i] : S[i];
        }
      }
    }
  };
  // behind the work of the chunk's turns k0 .. k0 + 3
  auto add_up = [&](int k0) {
    const float sums = ss_row_sums_of_four(parts[0], parts[1], parts[2], parts[3]);
    kept_sum = (ns & 3) == k0 / 4 ? sums : kept_sum;
  };
  // the outputs of the chunk of turns t0 .. t0 + n - 1 go out at the start of the next: they are on their way while it is worked on
  auto put = [&](int t0, int n) {
    if (half && own_turn < n && t0 + own_turn >= SS_BEHIND && has_p)
      y[(long)(first + t0 + own_turn - SS_BEHIND) * inner + x_col] = fmaf(dskip, kept_x, kept_sum);
    if (SEGMENTS && blockIdx.z == 0 && (int)threadIdx.x < min(SS_CHUNK, count - t0)) cum[(long)(first + t0 + ns) * heads + h] = kept_decay;
  };

  int buffer = 0;
  for (int t0 = 0; t0 < turns; t0 += SS_CHUNK) {
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();      // the chunk is in LDS for every wave; nobody reads the one before any more
    const int left = count - t0, ahead = t0 + SS_CHUNK;        // (left may be below 0: the second half's last tokens)
    const bool more = ahead < turns, begins = t0 == 0;
    const unsigned at = buffer * Chunk::FLOATS * 4;
    if (t0 != 0) put(t0 - SS_CHUNK, SS_CHUNK);
    if (more) ask_rest(buffer ^ 1, ahead);
    SsStaged<OWN> even, odd;
    // x of the lane's own turn, from those of turns 4 (ns % 4) .. + 3: waited for here, before any branch may copy what is under way
    auto own_x = [&]() {
      u32x4 xs[1];
      lds_read16<0>(xs[0], x_at + at + (ns & 3) * 16);
      wait_lgkmcnt<0>();
      use_frags<1>(xs);
      const unsigned lo = ns & 4 ? xs[0][1] : xs[0][0], hi = ns & 4 ? xs[0][3] : xs[0][2];
      kept_x = __uint_as_float(ns & 8 ? hi : lo);
    };
    if (left >= SS_CHUNK) {
      own_x();
      read(even, at, 0, 0);
      arrived(even);
#pragma unroll 1
      for (int k0 = 0; k0 < SS_CHUNK; k0 += 2 * SUB) {      // no read is under way across a branch
        read(odd, at, k0, 1);
        work(even, k0, 0, left, begins, SsNumber<1>());
        arrived(odd);
        if (more && k0 < SS_CHUNK / 2) ask(buffer ^ 1, ahead, 2 * k0, SsNumber<2 * SUB>());
        read(even, at, k0 + 2 * SUB < SS_CHUNK ? k0 + 2 * SUB : 0, 0);
        work(odd, k0, 1, left, begins, SsNumber<1>());
        add_up(k0);
        arrived(even);
        if (more && k0 < SS_CHUNK / 2) ask(buffer ^ 1, ahead, 2 * k0 + 2 * SUB, SsNumber<2 * SUB>());
      }
    } else {                                                // the last chunk, or the last but one
      own_x();
      if (more) {
#pragma unroll
        for (int k = 0; k < SS_BEHIND; ++k) ask(buffer ^ 1, ahead, k, SsNumber<1>());
      }
#pragma unroll 1
      for (int k0 = 0; k0 < min(SS_CHUNK, left + SS_BEHIND); k0 += 2 * SUB) {
        read(even, at, k0, 0);
        read(odd, at, k0, 1);                               // (places of the chunk that nothing was asked for: not used)
        arrived(even);
        arrived(odd);
        work(even, k0, 0, left, begins, SsNumber<0>());
        work(odd, k0, 1, left, begins, SsNumber<0>());
        add_up(k0);
      }
    }
    buffer ^= 1;
  }
  put((turns - 1) / SS_CHUNK * SS_CHUNK, (turns - 1) % SS_CHUNK + 1);
  // a segment's end state goes to the workspace; the fold brings the request's state up to date
  float* end = SEGMENTS ? ends + ((long)blockIdx.x * heads + h) * N * P : to + s_at;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int n = Rows::row(of_dim, i);
    if (has_p && n < N) end[(long)n * P + p] = S[i];
  }
  if (!SEGMENTS && blockIdx.y == 0 && blockIdx.z == 0)
    ss_keep_inputs(from, to, tail_at, conv_in, conv_in_stride, first, count, channels, taps);
}

// Long stretches of tokens in segments.  The walk above then runs every segment of a request side by side:
// the first from the request's state, the others from zero, each leaving its end state E_k in `ends` and
// the running product of its tokens' a in `cum`.  Two more launches make the rest:
//   the fold, per (request, head, eight value dims), over the request's segments in order: the state a
//   segment starts from is I_1 = E_0, I_(k+1) = D_k I_k + E_k (D_k: the segment's whole product), left in
//   `ends` in E_k's place; the last one is the request's new state (and the block (head 0, dims 0) brings
//   the convolution's kept inputs up to date);
//   the carry, per (segment but the first, head, eight value dims): y_t += cum_t (I_k^T C_t), what the
//   state the segment did not start from adds to its outputs; tokens are independent here.
// The sums of a token then differ in order from the walk of one chain, by rounding, and which tokens share a
// segment goes by how the request was cut into steps.
// spans5 [n][5] = (slot, first token, tokens, first segment, segments).
#define SS_THREADS 128      // of the fold and the carry: sixteen lanes a value dim
#define SS_CARRY 32        // tokens of a segment a block of the carry takes
#define SS_AHEAD 4         // tokens whose operands it asks for together
template <int OWN>
__global__ void __launch_bounds__(SS_THREADS)
state_space_fold_kernel(float* __restrict__ ends, const float* __restrict__ cum, const int32_t* __restrict__ spans5,
                        const int32_t* __restrict__ segs, float* __restrict__ state, long state_stride, long copy_elems,
                        long tail_at, const int32_t* __restrict__ positions, const float* __restrict__ conv_in,
                        long conv_in_stride, int heads, int P, int N, int channels, int taps) {
  const int slot = spans5[5 * blockIdx.x], first = spans5[5 * blockIdx.x + 1], count = spans5[5 * blockIdx.x + 2];
  const int seg0 = spans5[5 * blockIdx.x + 3], n_segs = spans5[5 * blockIdx.x + 4];
  const int h = blockIdx.y;
  const int ns = threadIdx.x & 15, p = blockIdx.z * (SS_THREADS / 16) + (threadIdx.x >> 4);
  const bool has_p = p < P;
  const int start = positions[first];
  const float* from = state + (long)slot * state_stride + (long)((start + 1) & 1) * copy_elems;
  float* to = state + (long)slot * state_stride + (long)((start + count - 1) & 1) * copy_elems;
  float I[OWN];
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int n = ns + 16 * i;
    I[i] = has_p && n < N ? ends[((long)seg0 * heads + h) * N * P + (long)n * P + p] : 0.0f;
  }
  for (int k = 1; k < n_segs; ++k) {
    const int seg = seg0 + k;
    const int seg_last = segs[4 * seg + 1] + segs[4 * seg + 2] - 1;
    const float D = cum[(long)seg_last * heads + h];
    float* E = ends + ((long)seg * heads + h) * N * P;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      const int n = ns + 16 * i;
      if (has_p && n < N) {
        const float e = E[(long)n * P + p];
        E[(long)n * P + p] = I[i];
        I[i] = fmaf(D, I[i], e);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int n = ns + 16 * i;
    if (has_p && n < N) to[(long)h * N * P + (long)n * P + p] = I[i];
  }
  if (blockIdx.y == 0 && blockIdx.z == 0) ss_keep_inputs(from, to, tail_at, conv_in, conv_in_stride, first, count, channels, taps);
}

template <int OWN>
__global__ void __launch_bounds__(SS_THREADS)
state_space_carry_kernel(const float* __restrict__ u, const float* __restrict__ ends, const float* __restrict__ cum,
                         const int32_t* __restrict__ segs, float* __restrict__ y, int heads, int groups, int P, int N,
                         int channels, int pieces) {
  // blockIdx.x: (segment, piece of SS_CARRY tokens of it); tokens are independent here
  const int seg = blockIdx.x / pieces, piece = blockIdx.x % pieces;
  if (segs[4 * seg + 3] != 0) return;                 // a request's first segment started from its state
  const int seg_first = segs[4 * seg + 1], seg_count = segs[4 * seg + 2];
  if (piece * SS_CARRY >= seg_count) return;
  const int first = seg_first + piece * SS_CARRY, count = min(SS_CARRY, seg_count - piece * SS_CARRY);
  const int h = blockIdx.y, g = h / (heads / groups);
  const int ns = threadIdx.x & 15, p = blockIdx.z * (SS_THREADS / 16) + (threadIdx.x >> 4);
  const bool has_p = p < P;
  const int inner = heads * P;
  const float* carried = ends + ((long)seg * heads + h) * N * P;
  float I[OWN];
  int n_of[OWN];
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int n = ns + 16 * i;
    I[i] = has_p && n < N ? carried[(long)n * P + p] : 0.0f;
    n_of[i] = min(n, N - 1);
  }
  const long c_col = inner + (long)groups * N + (long)g * N;
  const long out_col = (long)h * P + (has_p ? p : 0);
  for (int t0 = first; t0 < first + count; t0 += SS_AHEAD) {
    float C[SS_AHEAD][OWN], c[SS_AHEAD], was[SS_AHEAD];
#pragma unroll
    for (int k = 0; k < SS_AHEAD; ++k) {
      const int t = min(t0 + k, first + count - 1);
      const float* row = u + (long)t * channels + c_col;
#pragma unroll
      for (int i = 0; i < OWN; ++i) C[k][i] = row[n_of[i]];
      c[k] = cum[(long)t * heads + h];
      was[k] = y[(long)t * inner + out_col];
    }
#pragma unroll
    for (int k = 0; k < SS_AHEAD; ++k) {
      float part = 0.0f;
#pragma unroll
      for (int i = 0; i < OWN; ++i) part = fmaf(I[i], C[k][i], part);
      part = ss_row_sum(part);
      if (t0 + k < first + count && ns == 0 && has_p) y[(long)(t0 + k) * inner + out_col] = fmaf(c[k], part, was[k]);
    }
  }
}

// out[t, part] = ((v / sqrt(mean(v^2) + eps)) gain) with v = y[t, part] silu(z[t, part]): the gate first,
// then the norm of each of `parts` equal parts of a row by its own root mean square.  A block a (token, part):
// a strided chain a thread, a butterfly a wave, the four waves in order.
// KEPT x 256 values of a part are read once, and their gain beside them, not behind the sum; no more than the part has (us, gain behind / four a
// thread / here: 8,192 tokens of four parts of 16 26.4 / 30.0 / 26.4, of 640 53 / 43 / 43, 8 of one part of 1,024 3.2 / 2.6 / 2.6).
template <int KEPT>
__global__ void __launch_bounds__(256)
gated_group_norm_kernel(const float* __restrict__ y, const float* __restrict__ z, long z_stride, const void* __restrict__ gain,
                        int gain_is_f32, float eps, elem_t* __restrict__ out, int width, int parts) {
  __shared__ float partial[256 / AXON_WAVE];
  const int t = blockIdx.x / parts, part = blockIdx.x % parts, size = width / parts;
  const float* ys = y + (long)t * width + (long)part * size;
  const float* zs = z + (long)t * z_stride + (long)part * size;
  float kept[KEPT], gate[KEPT], g[KEPT][1];
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < KEPT; ++c) {
    const int i = min((int)threadIdx.x + 256 * c, size - 1);
    kept[c] = ys[i];
    gate[c] = zs[i];
  }
  load_vec_apart<KEPT, 1, false>(gain, gain_is_f32, part * size, threadIdx.x, 256, (part + 1) * size, g);
#pragma unroll
  for (int c = 0; c < KEPT; ++c) {
    if ((int)threadIdx.x + 256 * c < size) kept[c] *= ss_silu(gate[c]);
    else kept[c] = 0.0f;
    ss = fmaf(kept[c], kept[c], ss);
  }
  for (int i = threadIdx.x + 256 * KEPT; i < size; i += 256) {
    const float v = ys[i] * ss_silu(zs[i]);
    ss = fmaf(v, v, ss);
  }
  const float inv = 1.0f / sqrtf(block_sum_256(ss, partial) / (float)size + eps);
  elem_t* dst = out + (long)t * width + (long)part * size;
#pragma unroll
  for (int c = 0; c < KEPT; ++c) {
    const int i = threadIdx.x + 256 * c;
    if (i < size) dst[i] = from_float((kept[c] * inv) * g[c][0]);
  }
  for (int i = threadIdx.x + 256 * KEPT; i < size; i += 256) {
    const float v = ys[i] * ss_silu(zs[i]);
    dst[i] = from_float((v * inv) * load_vec(gain, gain_is_f32, part * size + i));
  }
}

}  // namespace

extern "C" int axk_state_conv(const float* x, long x_stride, const void* w, const void* bias, int bias_is_f32, int silu,
                              const float* state, long state_stride, long copy_elems, long tail_at, const int32_t* positions,
                              const int32_t* seq_rows, float* u, int n_tokens, int channels, int taps, const float* raw,
                              long raw_stride, const void* dt_bias, int dt_bias_is_f32, const void* a_log, int a_log_is_f32,
                              float* terms, int heads, int single, void* stream) {
  AXK_REQUIRE(n_tokens >= 0 && channels > 0 && taps >= 1 && x_stride >= channels && heads >= 0,
              "state_conv: bad sizes T=%d channels=%d taps=%d heads=%d row stride %ld", n_tokens, channels, taps, heads, x_stride);
  AXK_REQUIRE(tail_at >= 0 && copy_elems >= tail_at + (long)(taps - 1) * channels && state_stride >= 2 * copy_elems,
              "state_conv: a state row of %ld floats does not hold two copies of %ld with %d x %d kept inputs from %ld",
              state_stride, copy_elems, taps - 1, channels, tail_at);
  AXK_REQUIRE(heads == 0 || (raw != nullptr && dt_bias != nullptr && a_log != nullptr && terms != nullptr && raw_stride >= heads),
              "state_conv: step sizes of %d heads need their inputs", heads);
  AXK_REQUIRE(n_tokens <= 65535, "state_conv: %d tokens in one step (at most 65535)", n_tokens);
  if (n_tokens == 0) return 0;
  // Runs want enough of them to fill the chip: 4 million products (tokens x channels x taps), 6.2 where every token asks the state for its
  // earlier inputs.  us, a thread a (token, channel) / runs: four taps of 2,560 channels, 256 tokens of one request, or in twenties, 6.7 / 7.5, 384 8.3 / 8.3,
  // 448 9.3 / 8.4, 600 11.8 / 8.7, single ones 448 8.0 / 10.5, 600 10.7 / 11.0, 700 12.5 / 11.3; 600 of 1,280 7.7 / 7.4, 1,024 11.3 / 8.5, single 10.2 / 10.6; two
  // taps, 600 of 2,560 8.3 / 8.3, 1,024 12.7 / 9.2, single 12.2 / 10.6; four taps 1,024 of 64 2.9 / 12.6.  (Terms of a token's head are stored as a pair.)
  if (n_tokens >= 256 && (long)n_tokens * channels * taps >= (single ? 6200000 : 4000000) && taps >= 2 && taps <= 4 && channels % 4 == 0 &&
      x_stride % 4 == 0 &&
      (((uintptr_t)x | (uintptr_t)u) & 15) == 0 &&
      ((uintptr_t)terms & 7) == 0) {
    AXK_INSTANCE(INST_STATE_CONV, 1);
    auto kernel = taps == 2 ? state_conv_runs_kernel<2> : taps == 3 ? state_conv_runs_kernel<3> : state_conv_runs_kernel<4>;
    kernel<<<dim3(ceil_div(channels / 4 + heads, 128), ceil_div(n_tokens, SS_CONV_RUN)), 128, 0, (hipStream_t)stream>>>(
        x, x_stride, (const elem_t*)w, bias, bias_is_f32, silu, state, state_stride, copy_elems, tail_at, positions, seq_rows, u, n_tokens,
        channels, raw, raw_stride, dt_bias, dt_bias_is_f32, a_log, a_log_is_f32, terms, heads);
    AXK_LAUNCH_CHECK("state_conv");
    return 0;
  }
  AXK_INSTANCE(INST_STATE_CONV, 0);
  dim3 grid(ceil_div(channels + heads, 256), n_tokens);
  state_conv_kernel<<<grid, 256, 0, (hipStream_t)stream>>>(x, x_stride, (const elem_t*)w, bias, bias_is_f32, silu, state,
                                                          state_stride, copy_elems, tail_at, positions, seq_rows, u, channels,
                                                          taps, raw, raw_stride, dt_bias, dt_bias_is_f32, a_log, a_log_is_f32,
                                                          terms, heads);
  AXK_LAUNCH_CHECK("state_conv");
  return 0;
}

extern "C" int axk_state_space_scan(const float* u, const float* terms, const void* d_skip, int d_is_f32, float* state,
                                    long state_stride, long copy_elems, long tail_at, const int32_t* spans, int n_spans,
                                    const int32_t* positions, const int32_t* seq_rows, const float* conv_in, long conv_in_stride,
                                    float* y, int heads, int groups, int vdim, int n_state, int taps, const int32_t* segs,
                                    int n_segs, int longest_seg, const int32_t* spans5, float* ends, float* cum, void* stream) {
  AXK_REQUIRE(n_spans >= 0 && heads > 0 && groups > 0 && heads % groups == 0 && vdim > 0 && n_state > 0 && taps >= 1,
              "state_space_scan: bad sizes spans=%d heads=%d groups=%d vdim=%d state=%d taps=%d", n_spans, heads, groups, vdim,
              n_state, taps);
  AXK_REQUIRE(n_state <= 256, "state_space_scan: a state of %d rows a head (at most 256)", n_state);
  const int channels = heads * vdim + 2 * groups * n_state;
  AXK_REQUIRE(tail_at >= (long)heads * n_state * vdim && copy_elems >= tail_at + (long)(taps - 1) * channels &&
              state_stride >= 2 * copy_elems && conv_in_stride >= channels,
              "state_space_scan: a state row of %ld floats does not hold two copies of %ld (%d x %d x %d, then %d x %d from %ld)",
              state_stride, copy_elems, heads, n_state, vdim, taps - 1, channels, tail_at);
  AXK_REQUIRE((spans != nullptr || seq_rows != nullptr) && positions != nullptr, "state_space_scan: neither spans nor slots, or no positions");
  AXK_REQUIRE(n_spans <= 65535 * 32 && heads <= 65535 && ceil_div(vdim, SS_THREADS / 16) <= 65535, "state_space_scan: %d requests of %d heads", n_spans, heads);
  if (n_spans == 0) return 0;
  AXK_REQUIRE(segs == nullptr || (n_segs >= n_spans && spans5 != nullptr && ends != nullptr && cum != nullptr && spans != nullptr),
              "state_space_scan: %d segments of %d requests come with the requests' list, a workspace and the running products",
              n_segs, n_spans);
  dim3 grid(segs ? n_segs : n_spans, heads, ceil_div(vdim, SS_THREADS / 16));
  dim3 grid_fold(n_spans, heads, ceil_div(vdim, SS_THREADS / 16));
  AXK_REQUIRE(segs == nullptr || longest_seg > 0, "state_space_scan: segments of at most %d tokens", longest_seg);
  const int pieces = segs ? ceil_div(longest_seg, SS_CARRY) : 1;
  dim3 grid_carry((unsigned)((long)(segs ? n_segs : 1) * pieces), heads, ceil_div(vdim, SS_THREADS / 16));
  hipStream_t s = (hipStream_t)stream;
#define SS_LAUNCH(OWN)                                                                              \
  {                                                                                                 \
    if (spans == nullptr)                                                                           \
      state_space_step_kernel<OWN><<<grid, SS_WALKERS, 0, s>>>(u, terms, d_skip, d_is_f32, state, state_stride, copy_elems, tail_at, \
                                                               positions, seq_rows, conv_in, conv_in_stride, y, heads, groups, vdim, \
                                                               n_state, channels, taps);            \
    else if (segs) {                                                                                \
      if (n_state == 16 * OWN) state_space_walk_kernel<OWN, true, true><<<grid, SS_WALKERS, 0, s>>>(SS_ARGS); \
      else state_space_walk_kernel<OWN, false, true><<<grid, SS_WALKERS, 0, s>>>(SS_ARGS);          \
    } else {                                                                                        \
      if (n_state == 16 * OWN) state_space_walk_kernel<OWN, true, false><<<grid, SS_WALKERS, 0, s>>>(SS_ARGS); \
      else state_space_walk_kernel<OWN, false, false><<<grid, SS_WALKERS, 0, s>>>(SS_ARGS);         \
    }                                                                                               \
    if (segs) {                                                                                     \
      state_space_fold_kernel<OWN><<<grid_fold, SS_THREADS, 0, s>>>(ends, cum, spans5, segs, state, state_stride, copy_elems, tail_at, \
                                                                    positions, conv_in, conv_in_stride, heads, vdim, n_state, channels, taps); \
      state_space_carry_kernel<OWN><<<grid_carry, SS_THREADS, 0, s>>>(u, ends, cum, segs, y, heads, groups, vdim, n_state, channels, pieces); \
    }                                                                                               \
  }
#define SS_ARGS u, terms, d_skip, d_is_f32, state, state_stride, copy_elems, tail_at, spans, positions, conv_in, conv_in_stride, y, \
                heads, groups, vdim, n_state, channels, taps, segs, ends, cum
  if (n_state <= 16) SS_LAUNCH(1)
  else if (n_state <= 32) SS_LAUNCH(2)
  else if (n_state <= 64) SS_LAUNCH(4)
  else if (n_state <= 128) SS_LAUNCH(8)
  else SS_LAUNCH(16)
#undef SS_LAUNCH
#undef SS_ARGS
  AXK_LAUNCH_CHECK("state_space_scan");
  return 0;
}

extern "C" int axk_gated_group_norm(const float* y, const float* z, long z_stride, const void* gain, int gain_is_f32, float eps,
                                    void* out, int n_tokens, int width, int parts, void* stream) {
  AXK_REQUIRE(n_tokens >= 0 && width > 0 && parts > 0 && width % parts == 0 && z_stride >= width,
              "gated_group_norm: bad sizes T=%d width=%d parts=%d", n_tokens, width, parts);
  if (n_tokens == 0) return 0;
  AXK_REQUIRE((long)n_tokens * parts <= 2147483647L, "gated_group_norm: %d tokens in %d parts", n_tokens, parts);
  const int size = width / parts;
  auto kernel = size <= 256 ? gated_group_norm_kernel<1> : size <= 512 ? gated_group_norm_kernel<2> : gated_group_norm_kernel<4>;
  kernel<<<(unsigned)((long)n_tokens * parts), 256, 0, (hipStream_t)stream>>>(y, z, z_stride, gain, gain_is_f32, eps, (elem_t*)out, width, parts);
  AXK_LAUNCH_CHECK("gated_group_norm");
  return 0;
}
