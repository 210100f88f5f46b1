// A gated linear recurrence with a short causal convolution in front of it (the recurrent block of
// Griffin-like models): per-request state in 32-bit floats, carried from step to step.
//
// A request's state row holds two copies of ([channels] of recurrent state, then [taps - 1][channels]
// of the convolution's last inputs, oldest first); a new request starts from zeros, which is also
// what the convolution reads before the first token.  The state behind position p lives in copy
// p & 1: a step whose first position is s reads copy (s - 1) & 1 and writes the copy of its last
// position.  A step of one token therefore never writes what it read, and running it again (a
// decoding step is run once before it is captured into a graph) gives the same state and the same
// output.  The tokens of a request are contiguous in a step and a request is in a step once, so
// two tokens belong to one request iff their state slots (seq_rows) are equal.
#include "api.h"
#include "common.h"
#include "instances.h"

namespace {

// u[t, c] = bias[c] + sum_k w[c, k] in(t - (taps - 1 - k)): the last column of w is the current
// token's.  One thread per (token, channel); inputs before the step come from the state.
__global__ void causal_conv_kernel(const elem_t* __restrict__ x, long x_stride, const elem_t* __restrict__ w,
                                   const void* __restrict__ bias, int bias_is_f32, const float* __restrict__ state,
                                   long state_stride, const int32_t* __restrict__ positions,
                                   const int32_t* __restrict__ seq_rows, float* __restrict__ u, int channels, int taps) {
  const int t = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int slot = seq_rows[t];
  // how many earlier tokens of this step belong to the same request (up to taps - 1 matter)
  int inside = 0;
  while (inside < taps - 1 && t - inside - 1 >= 0 && seq_rows[t - inside - 1] == slot) ++inside;
  // the copy behind the position before the request's first of this step (not needed where all taps lie inside the step)
  const int before = (positions[t] - inside + 1) & 1;
  const float* kept = state + (long)slot * state_stride + (long)before * taps * channels + channels;      // [taps - 1][channels]
  float acc = 0.0f;
  for (int k = 0; k < taps; ++k) {
    const int back = taps - 1 - k;            // the input `back` tokens before this one
    float v;
    if (back <= inside) v = to_float(x[(long)(t - back) * x_stride + c]);
    else v = kept[(long)(taps - 1 - (back - inside)) * channels + c];        // the (back - inside)-th last kept input
    acc = fmaf(to_float(w[(long)c * taps + k]), v, acc);
  }
  if (bias) acc += load_vec(bias, bias_is_f32, c);
  u[(long)t * channels + c] = acc;
}

// The same for many tokens: a thread takes four channels of CONV_RUN tokens, whose inputs (and the taps - 1 before them) it
// asks for at once and keeps in registers, where a thread a (token, channel) reads each `taps` times and waits for its
// row's slot first.  Runs in which a request begins also ask for the kept inputs of all their tokens at once.  The sums in
// the same order.  Bound by the three waits (slots, inputs, outputs) of the one round of blocks; 2,560 channels, us, a thread
// a (token, channel) against here: 2,048 tokens of one request 38.7 / 13.4, of requests of 16 37.6 / 15.0, of 2,048 requests
// 31.0 / 20.9; 512 of one 9.3 / 7.6.
#define CONV_RUN 8
#define CONV_TAPS 4           // at most
__global__ void __launch_bounds__(128)
causal_conv_run_kernel(const elem_t* __restrict__ x, long x_stride, const elem_t* __restrict__ w, const void* __restrict__ bias,
                       int bias_is_f32, const float* __restrict__ state, long state_stride, const int32_t* __restrict__ positions,
                       const int32_t* __restrict__ seq_rows, float* __restrict__ u, int n_tokens, int channels, int taps) {
  const int c = 4 * (blockIdx.x * blockDim.x + threadIdx.x), t0 = blockIdx.y * CONV_RUN;
  if (c >= channels) return;
  float in[CONV_RUN + CONV_TAPS - 1][4];             // of tokens t0 - (CONV_TAPS - 1) ..
  int slots[CONV_RUN + CONV_TAPS - 1];
#pragma unroll
  for (int i = 0; i < CONV_RUN + CONV_TAPS - 1; ++i) {
    const int t = min(max(t0 + i - (CONV_TAPS - 1), 0), n_tokens - 1);
    slots[i] = t == t0 + i - (CONV_TAPS - 1) ? seq_rows[t] : -1;
    load4_guarded(x + (long)t * x_stride + c, 4, true, in[i]);
  }
  float wb[CONV_TAPS][4];                            // the weights of the input `back` tokens before
#pragma unroll
  for (int back = 0; back < CONV_TAPS; ++back)
#pragma unroll
    for (int e = 0; e < 4; ++e) wb[back][e] = back < taps ? to_float(w[(long)(c + e) * taps + taps - 1 - back]) : 0.0f;
  float added[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (bias)
#pragma unroll
    for (int e = 0; e < 4; ++e) added[e] = load_vec(bias, bias_is_f32, c + e);

  int inside[CONV_RUN];                              // earlier tokens of this step that belong to the same request
  bool begins = false;
#pragma unroll
  for (int r = 0; r < CONV_RUN; ++r) {
    inside[r] = 0;
#pragma unroll
    for (int b = 1; b < CONV_TAPS; ++b)
      if (b < taps && inside[r] == b - 1 && slots[r + CONV_TAPS - 1 - b] == slots[r + CONV_TAPS - 1]) inside[r] = b;
    begins |= t0 + r < n_tokens && inside[r] < taps - 1;
  }
  float kept[CONV_RUN][CONV_TAPS - 1][4];            // the inputs 1 .. CONV_TAPS - 1 tokens before, from the state
  if (begins) {                                      // the same for the whole block
#pragma unroll
    for (int r = 0; r < CONV_RUN; ++r) {
      const int t = min(t0 + r, n_tokens - 1);
      const int before = (positions[t] - inside[r] + 1) & 1;
      const float* row = state + (long)seq_rows[t] * state_stride + (long)before * taps * channels + channels + c;
#pragma unroll
      for (int back = 1; back < CONV_TAPS; ++back) {
        const bool needed = back < taps && back > inside[r];       // (else any row that is there)
        const float4 v = *reinterpret_cast<const float4*>(row + (needed ? (long)(taps - 1 - (back - inside[r])) * channels : -(long)channels));
        kept[r][back - 1][0] = v.x; kept[r][back - 1][1] = v.y; kept[r][back - 1][2] = v.z; kept[r][back - 1][3] = v.w;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < CONV_RUN; ++r) {
    if (t0 + r >= n_tokens) break;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int back = CONV_TAPS - 1; back >= 0; --back) {
      if (back >= taps) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = back > 0 && begins && back > inside[r] ? kept[r][back > 0 ? back - 1 : 0][e] : in[r + CONV_TAPS - 1 - back][e];
        acc[e] = fmaf(wb[back][e], v, acc[e]);
      }
    }
    if (bias)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += added[e];
    *reinterpret_cast<float4*>(u + (long)(t0 + r) * channels + c) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  }
}

__device__ inline float sigmoid32(float z) { return 1.0f / (1.0f + expf(-z)); }

__device__ inline float gelu_tanh32(float z) {
  const float inner = 0.7978845608028654f * (z + 0.044715f * ((z * z) * z));
  return (0.5f * z) * (1.0f + tanhf(inner));
}

// One thread per (request of the step, channel), walking the request's tokens in order:
//   r = sigmoid(gates[t, r part]), i = sigmoid(gates[t, i part]), log a = -decay r softplus(lam),
//   S = a S + sqrt(1 - a^2) (i u), out[t] = S gelu(y[t]).
// gates [T, blocks, 2 block_width]: a block's r logits, then its i logits.  spans [n][3] = (slot,
// first token, tokens), or null: every token is a request of its own (a decoding step) in slot
// seq_rows[t].  Afterwards the request's state row holds S and the last taps - 1 inputs of the
// convolution.
__global__ void gated_scan_kernel(const float* __restrict__ gates, const float* __restrict__ u,
                                  const elem_t* __restrict__ y, long y_stride, const elem_t* __restrict__ x, long x_stride,
                                  const void* __restrict__ lam, int lam_is_f32, float decay, float* __restrict__ state,
                                  long state_stride, const int32_t* __restrict__ spans, const int32_t* __restrict__ positions,
                                  const int32_t* __restrict__ seq_rows, elem_t* __restrict__ out, int channels, int block_width,
                                  int taps) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  int slot, first, count;
  if (spans) {
    slot = spans[3 * blockIdx.y]; first = spans[3 * blockIdx.y + 1]; count = spans[3 * blockIdx.y + 2];
  } else {
    slot = seq_rows[blockIdx.y]; first = blockIdx.y; count = 1;
  }
  const float l = load_vec(lam, lam_is_f32, c);
  const float softplus = l > 20.0f ? l : log1pf(expf(l));
  const float rate = -decay * softplus;
  const int b = c / block_width, j = c % block_width;
  const long gate_at = (long)b * 2 * block_width + j;
  const int start = positions[first];
  const float* from = state + (long)slot * state_stride + (long)((start + 1) & 1) * taps * channels;
  float* row = state + (long)slot * state_stride + (long)((start + count - 1) & 1) * taps * channels;
  float S = from[c];
  for (int t = first; t < first + count; ++t) {
    const float* g = gates + (long)t * 2 * channels + gate_at;
    const float r = sigmoid32(g[0]), i = sigmoid32(g[block_width]);
    const float log_a = rate * r;
    const float a = expf(log_a);
    const float mult = sqrtf(-expm1f(2.0f * log_a));                 // sqrt(1 - a^2), exact also where a is near 1
    S = fmaf(a, S, (mult * i) * u[(long)t * channels + c]);
    out[(long)t * channels + c] = from_float(S * gelu_tanh32(to_float(y[(long)t * y_stride + c])));
  }
  row[c] = S;
  // the convolution's last taps - 1 inputs: of (what was kept, this step's inputs) the last taps - 1;
  // place i takes what lies `count` places later (where both copies are one: read before it is written, ascending)
  float* kept = row + channels;
  const float* kept_from = from + channels;
  for (int i = 0; i < taps - 1; ++i) {
    const int at = i + count;
    kept[(long)i * channels + c] = at < taps - 1 ? kept_from[(long)at * channels + c]
                                                 : to_float(x[(long)(first + at - (taps - 1)) * x_stride + c]);
  }
}

// The same recurrence for stretches of tokens: a block has `width` channels of a request.  One wave walks S = a S + b, a lane a
// channel, and does nothing else; the others work out, a (token, channel) a lane, what it walks with and what comes of it: a,
// b = (sqrt(1 - a^2) i) u and gelu(y) of the chunk ahead, the outputs of the chunk behind, through LDS, a barrier a chunk.  The
// operations are those of the kernel above, and so are the bits.  Bound by the exponentials and the tangent, some 200 vector
// instructions a (token, channel): 2,048 tokens of 2,560 channels 47 us, where the terms in a launch of their own through memory and
// a walk bound by what one wave issues took 35 + 91; 4,096 243 -> 87, 512 37 -> 16, 64 15 -> 10; five requests of 300 46 -> 34, 64
// of 32 48 -> 40; 5,120 channels 157 -> 67, 1,024 106 -> 40.
#define SCAN_FEEDERS 512
#define SCAN_EACH 2                               // tokens of a chunk that a feeding thread has
#define SCAN_WIDEST 64
// Tokens that the feeding threads have side by side: four at a time, since the walk reads four.
__host__ __device__ inline int scan_rows(int width) { return SCAN_FEEDERS / width / 4 * 4; }
// Channels a block has: of a lone request, or one that outlasts those beside it, as many as give every CU a block, 16 of each of several, 64 of those that are short, 16 of these too while
// all blocks have a place (512).  The short ones have blocks of their own behind the long ones' (where it is not known which they are, as many as if
// they were long, and those that are too many leave at once: a block launched in vain costs some 10 ns); requests take their first channels to the
// XCDs in turn (100 requests of 64 tokens of 64 channels, all on one XCD, 25.8 us, so 13.4).  us by width, 2,560 channels: 2,048 tokens of a request 53.5
// with 8, 46.8 with 10, 50.0 with 16, 91.9 with 32 (5,120 channels 64.1 with 10, 67.1 with 20, 79.1 with 16); requests of 1,000, 700 and 400 38.9 with 10,
// 35.7 with 16, 48.5 with 32; five of 300 39.8, 33.8, 28.7, and 31.7 with 64; 64 of 32 tokens 93.0 with 16, 39.7 with 64; one of 300 and 60 of 64, 1,024
// channels, in vain / not 54 / 35.
#define SCAN_SHORT 128
__host__ inline int scan_width(int channels, int requests) {
  const int width = requests > 1 ? 16 : (channels + 255) / 256;
  return width < 8 ? 8 : width <= 16 ? (width + 1) / 2 * 2 : width <= 20 ? 20 : 32;
}
// Blocks of a request, as many on each XCD.
__host__ __device__ inline int scan_blocks(int channels, int width) { return ((channels + width - 1) / width + 7) / 8 * 8; }
// Floats a channel has in LDS: four more than its tokens, so that lanes side by side meet different banks.
#define SCAN_FLOATS (SCAN_FEEDERS * SCAN_EACH + 4 * SCAN_WIDEST)

__device__ inline void scan_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }   // loads stay under way

__global__ void __launch_bounds__(SCAN_FEEDERS + AXON_WAVE)
gated_scan_stretch_kernel(const float* __restrict__ gates, const float* __restrict__ u, const elem_t* __restrict__ y, long y_stride,
                          const elem_t* __restrict__ x, long x_stride, const void* __restrict__ lam, int lam_is_f32, float decay,
                          float* __restrict__ state, long state_stride, const int32_t* __restrict__ spans,
                          const int32_t* __restrict__ positions, elem_t* __restrict__ out, int channels, int block_width, int taps,
                          int n_long, int width_long, int width_short) {
  __shared__ __align__(16) float as[2][SCAN_FLOATS], bs[2][SCAN_FLOATS], ss[2][SCAN_FLOATS];
  // the blocks of the long requests, request by request, then those of the short ones
  const int per_long = scan_blocks(channels, width_long), per_short = scan_blocks(channels, width_short);
  const bool is_long = (int)blockIdx.x < n_long * per_long;
  const int b = blockIdx.x - (is_long ? 0 : n_long * per_long), per = is_long ? per_long : per_short;
  const int request = b / per + (is_long ? 0 : n_long), place = b % per;
  const int slot = spans[3 * request], first = spans[3 * request + 1], count = spans[3 * request + 2];
  const int width = !is_long || (width_short > width_long && count <= SCAN_SHORT) ? width_short : width_long;
  // neighbouring channels on one XCD: their rows share cache lines; the requests' first ones on all in turn
  const int per_xcd = scan_blocks(channels, width) / 8, c0 = ((place + request) % 8 * per_xcd + place / 8) * width;
  if (place / 8 >= per_xcd || c0 >= channels || count <= 0) return;
  const int rows = scan_rows(width), chunk = SCAN_EACH * rows, pitch = chunk + 4, chunks = (count + chunk - 1) / chunk;
  if (threadIdx.x >= SCAN_FEEDERS) {
    const int lane = threadIdx.x - SCAN_FEEDERS, c = c0 + lane;
    const bool has = lane < width && c < channels;
    const int start = positions[first];
    const float* from = state + (long)slot * state_stride + (long)((start + 1) & 1) * taps * channels;
    float* row = state + (long)slot * state_stride + (long)((start + count - 1) & 1) * taps * channels;
    float S = has ? from[c] : 0.0f;
    for (int it = 0; it < chunks + 2; ++it) {
      if (it > 0 && it <= chunks && has) {
        const int left = count - (it - 1) * chunk, at = lane * pitch;
        const float* A = as[(it - 1) & 1] + at;
        const float* B = bs[(it - 1) & 1] + at;
        float* to = ss[(it - 1) & 1] + at;
        if (left >= chunk) {
          float4 a0 = *reinterpret_cast<const float4*>(A), b0 = *reinterpret_cast<const float4*>(B);
          for (int j = 0; j < chunk; j += 4) {
            const int ahead = min(j + 4, chunk - 4);
            const float4 a1 = *reinterpret_cast<const float4*>(A + ahead), b1 = *reinterpret_cast<const float4*>(B + ahead);
            float4 v;
            S = fmaf(a0.x, S, b0.x); v.x = S;
            S = fmaf(a0.y, S, b0.y); v.y = S;
            S = fmaf(a0.z, S, b0.z); v.z = S;
            S = fmaf(a0.w, S, b0.w); v.w = S;
            *reinterpret_cast<float4*>(to + j) = v;
            a0 = a1; b0 = b1;
          }
        } else {
          for (int j = 0; j < left; ++j) {
            S = fmaf(A[j], S, B[j]);
            to[j] = S;
          }
        }
      }
      scan_barrier();
    }
    if (!has) return;
    row[c] = S;
    float* kept = row + channels;
    const float* kept_from = from + channels;
    for (int i = 0; i < taps - 1; ++i) {
      const int at = i + count;
      kept[(long)i * channels + c] = at < taps - 1 ? kept_from[(long)at * channels + c]
                                                   : to_float(x[(long)(first + at - (taps - 1)) * x_stride + c]);
    }
    return;
  }

  const int ch = threadIdx.x % width, tok = threadIdx.x / width, c = c0 + ch;
  const bool has = tok < rows && c < channels;
  const int cc = min(c, channels - 1);
  const float l = load_vec(lam, lam_is_f32, cc);
  const float softplus = l > 20.0f ? l : log1pf(expf(l));
  const float rate = -decay * softplus;
  const long gate_at = (long)(cc / block_width) * 2 * block_width + cc % block_width;
  struct Inputs { float r, i, u; elem_t y; };
  Inputs next[SCAN_EACH];
  auto ask = [&](int it) {                         // (behind the last token: that one, not used)
#pragma unroll
    for (int e = 0; e < SCAN_EACH; ++e) {
      const long t = first + min(it * chunk + e * rows + tok, count - 1);
      const float* g = gates + t * 2 * channels + gate_at;
      next[e] = Inputs{g[0], g[block_width], u[t * channels + cc], y[t * y_stride + cc]};
    }
  };
  ask(0);
  float gelu[3][SCAN_EACH] = {};                   // of the chunk now fed, of the one walked, of the one put out
  for (int it = 0; it < chunks + 2; ++it) {
#pragma unroll
    for (int e = 0; e < SCAN_EACH; ++e) { gelu[2][e] = gelu[1][e]; gelu[1][e] = gelu[0][e]; }
    if (it < chunks) {
      Inputs now[SCAN_EACH];
#pragma unroll
      for (int e = 0; e < SCAN_EACH; ++e) now[e] = next[e];
      if (it + 1 < chunks) ask(it + 1);
#pragma unroll
      for (int e = 0; e < SCAN_EACH; ++e) {
        const float r = sigmoid32(now[e].r), i = sigmoid32(now[e].i);
        const float log_a = rate * r;
        const float mult = sqrtf(-expm1f(2.0f * log_a));
        const float a = expf(log_a), b = (mult * i) * now[e].u;
        gelu[0][e] = gelu_tanh32(to_float(now[e].y));
        if (has) {
          as[it & 1][ch * pitch + e * rows + tok] = a;
          bs[it & 1][ch * pitch + e * rows + tok] = b;
        }
      }
    }
    if (it >= 2 && has) {
#pragma unroll
      for (int e = 0; e < SCAN_EACH; ++e) {
        const int j = (it - 2) * chunk + e * rows + tok;
        if (j < count) out[(long)(first + j) * channels + c] = from_float(ss[it & 1][ch * pitch + e * rows + tok] * gelu[2][e]);
      }
    }
    scan_barrier();
  }
}

}  // namespace

extern "C" int axk_causal_conv(const void* x, long x_stride, const void* w, const void* bias, int bias_is_f32,
                               const float* state, long state_stride, const int32_t* positions, const int32_t* seq_rows,
                               float* u, int n_tokens, int channels, int taps, void* stream) {
  AXK_REQUIRE(n_tokens >= 0 && channels > 0 && taps >= 1 && x_stride >= channels,
              "causal_conv: bad sizes T=%d channels=%d taps=%d row stride %ld", n_tokens, channels, taps, x_stride);
  AXK_REQUIRE(state_stride >= 2L * taps * channels, "causal_conv: a state row of %ld floats does not hold 2 x %d x %d",
              state_stride, taps, channels);
  AXK_REQUIRE(n_tokens <= 65535, "causal_conv: %d tokens in one step (at most 65535)", n_tokens);
  if (n_tokens == 0) return 0;
  // A step has to be long enough for a run to pay: blocks of 8 tokens x 512 channels wait one after another where a thread a
  // (token, channel) has a wave for every wait.  2,560 channels (us, a thread each against runs): 64 tokens 3.6 / 6.8, 256
  // 6.0 / 7.0, 512 9.3 / 7.6, 512 requests of a token 9.4 / 9.4; 512 channels: 2,048 tokens 8.0 / 7.0, 2,048 requests 6.9 / 7.7.
  const bool by_fours = channels % 4 == 0 && x_stride % 4 == 0 && (uintptr_t)x % (4 * sizeof(elem_t)) == 0 && ((uintptr_t)u & 15) == 0 &&
                        state_stride % 4 == 0 && ((uintptr_t)state & 15) == 0;
  if (by_fours && taps <= CONV_TAPS && (long)n_tokens * channels >= 512 * 2560) {
    AXK_INSTANCE(INST_CAUSAL_CONV, 1);
    causal_conv_run_kernel<<<dim3(ceil_div(channels / 4, 128), ceil_div(n_tokens, CONV_RUN)), 128, 0, (hipStream_t)stream>>>(
        (const elem_t*)x, x_stride, (const elem_t*)w, bias, bias_is_f32, state, state_stride, positions, seq_rows, u, n_tokens, channels, taps);
    AXK_LAUNCH_CHECK("causal_conv");
    return 0;
  }
  AXK_INSTANCE(INST_CAUSAL_CONV, 0);
  dim3 grid(ceil_div(channels, 256), n_tokens);
  causal_conv_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const elem_t*)x, x_stride, (const elem_t*)w, bias, bias_is_f32,
                                                           state, state_stride, positions, seq_rows, u, channels, taps);
  AXK_LAUNCH_CHECK("causal_conv");
  return 0;
}

extern "C" int axk_gated_scan(const float* gates, const float* u, const void* y, long y_stride, const void* x, long x_stride,
                              const void* lam, int lam_is_f32, float decay, float* state, long state_stride,
                              const int32_t* spans, int n_spans, const int32_t* positions, const int32_t* seq_rows, void* out,
                              int channels, int block_width, int taps, void* stream) {
  AXK_REQUIRE(n_spans >= 0 && channels > 0 && block_width > 0 && channels % block_width == 0 && taps >= 1,
              "gated_scan: bad sizes spans=%d channels=%d block width=%d taps=%d", n_spans, channels, block_width, taps);
  AXK_REQUIRE(state_stride >= 2L * taps * channels, "gated_scan: a state row of %ld floats does not hold 2 x %d x %d",
              state_stride, taps, channels);
  AXK_REQUIRE((spans != nullptr || seq_rows != nullptr) && positions != nullptr, "gated_scan: neither spans nor slots, or no positions");
  AXK_REQUIRE(n_spans <= 65535, "gated_scan: %d requests in one step (at most 65535)", n_spans);
  if (n_spans == 0) return 0;
  AXK_INSTANCE(INST_GATED_SCAN, 0);
  dim3 grid(ceil_div(channels, 64), n_spans);
  gated_scan_kernel<<<grid, 64, 0, (hipStream_t)stream>>>(gates, u, (const elem_t*)y, y_stride, (const elem_t*)x, x_stride, lam,
                                                         lam_is_f32, decay, state, state_stride, spans, positions,
                                                         seq_rows, (elem_t*)out, channels, block_width, taps);
  AXK_LAUNCH_CHECK("gated_scan");
  return 0;
}

extern "C" int axk_gated_scan_stretches(const float* gates, const float* u, const void* y, long y_stride, const void* x, long x_stride,
                                        const void* lam, int lam_is_f32, float decay, float* state, long state_stride,
                                        const int32_t* spans, int n_spans, const int32_t* positions, void* out, int channels,
                                        int block_width, int taps, int n_long, int alone, void* stream) {
  AXK_REQUIRE(n_spans >= 0 && channels > 0 && block_width > 0 && channels % block_width == 0 && taps >= 1,
              "gated_scan: bad sizes spans=%d channels=%d block width=%d taps=%d", n_spans, channels, block_width, taps);
  AXK_REQUIRE(state_stride >= 2L * taps * channels, "gated_scan: a state row of %ld floats does not hold 2 x %d x %d",
              state_stride, taps, channels);
  AXK_REQUIRE(spans != nullptr && positions != nullptr, "gated_scan: no spans or no positions");
  AXK_REQUIRE(n_spans <= 65535, "gated_scan: %d requests in one step (at most 65535)", n_spans);
  AXK_REQUIRE(n_long <= n_spans, "gated_scan: %d long ones of %d requests", n_long, n_spans);
  if (n_spans == 0) return 0;
  const int most = n_long < 0 ? n_spans : n_long;       // (not known: as many blocks as if all were long)
  const int width = scan_width(channels, n_spans == 1 || (most == 1 && alone) ? 1 : 2);
  const bool few = (long)most * scan_blocks(channels, width) + (long)(n_spans - most) * scan_blocks(channels, 16) <= 512;
  const int width_short = n_spans == 1 ? width : n_long >= 0 && few ? 16 : SCAN_WIDEST;
  const long blocks = (long)most * scan_blocks(channels, width) + (long)(n_spans - most) * scan_blocks(channels, width_short);
  AXK_REQUIRE(blocks <= 2147483647L, "gated_scan: %ld blocks are more than one launch takes", blocks);
  AXK_INSTANCE(INST_GATED_SCAN, 1);
  gated_scan_stretch_kernel<<<(unsigned)blocks, SCAN_FEEDERS + AXON_WAVE, 0, (hipStream_t)stream>>>(
      gates, u, (const elem_t*)y, y_stride, (const elem_t*)x, x_stride, lam, lam_is_f32, decay, state, state_stride, spans, positions,
      (elem_t*)out, channels, block_width, taps, most, width, width_short);
  AXK_LAUNCH_CHECK("gated_scan_stretches");
  return 0;
}
