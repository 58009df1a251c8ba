// Capacity model: an 8 -> 64 -> 64 -> 64 -> 3 ReLU MLP over per-node
// features, with bfloat16 weights and float32 accumulation, trained and run
// by these kernels. Output j is the log2 of a Poisson rate: the expected
// far-list count, near-list count (leaves) and number of pairs in the peak
// wavefront with this node as target, each divided by a per-output scale.
// Trained on the Poisson negative log-likelihood, the rates are unbiased, so
// their sums estimate the walk's stream sizes in one pass. A misprediction
// only costs a stream growth during the walk (or, for the pair queue, a
// rerun without the prediction): lists never depend on the model.
//
// Parameter layout (P = 9091 floats): W1[64][8] b1[64] W2[64][64] b2[64]
// W3[64][64] b3[64] W4[3][64] b4[3]; W[o][i] multiplies input i into output o.
#include "ygg_common.h"

// The model's arithmetic is not matched against the reference, so products
// and sums may fuse here.
#pragma clang fp contract(fast)

namespace ygg {

constexpr int kIn = 8, kH = 64, kOut = 3;
constexpr int kOffW1 = 0, kOffB1 = kOffW1 + kH * kIn, kOffW2 = kOffB1 + kH,
              kOffB2 = kOffW2 + kH * kH, kOffW3 = kOffB2 + kH, kOffB3 = kOffW3 + kH * kH,
              kOffW4 = kOffB3 + kH, kOffB4 = kOffW4 + kOut * kH, kParams = kOffB4 + kOut;

__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __uint_as_float((uint32_t)h << 16);
}

// Round-to-nearest-even float32 -> bfloat16 (NaN kept quiet).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x7FFFFFu)) return (uint16_t)((u >> 16) | 0x40);
  uint32_t r = u + 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(r >> 16);
}

// ---- inference on the matrix cores --------------------------------------
// Each wavefront runs 16 samples at a time through the four layers with
// 16x16x32 bf16 MFMAs (fp32 accumulate). Operand layouts of
// v_mfma_f32_16x16x32_bf16 on wave64 (lane l, q = l / 16):
//   A[m][k]: lane l holds A[l % 16][8 q + j],  j = 0..7
//   B[k][n]: lane l holds B[8 q + j][l % 16],  j = 0..7
//   D[m][n]: lane l holds D[4 q + j][l % 16],  j = 0..3
// With A = a 16-output slice of W (m = output, k = input) and B = the
// activations (k = input feature, n = sample), the D tiles 2s and 2s + 1 of
// a layer are, lane for lane, the B operand of k-step s of the next one if
// slot (q, j) stands for input 16 (2s + j / 4) + 4 q + j % 4 in A as well:
// no data moves between layers. The weights are exactly bf16; each fp32
// activation is split into bf16 hi + lo (split_bf16) and both halves are
// multiplied, so the products keep 2^-17 relative accuracy and the outputs
// match fp32 arithmetic to ~1e-5. The first layer's eight inputs take one
// k-step for both halves (slots q = 0 the hi, q = 1 the lo parts).
//
// Bound by the chain of splits and MFMAs of a tile (about 220 vector
// instructions and 40 MFMAs): 0.83 us per tile and SIMD with two or three
// wavefronts. Weight fragments live in registers for the whole kernel,
// gathered once through LDS (from global memory the gather had taken 10 us of
// every call), biases in LDS. 524287 nodes take 29 us, against 97 us for the
// 16x16x16 form (80 MFMAs, rounding in integer arithmetic, one wavefront per
// SIMD); with 2 wavefronts per SIMD 31 us, with 4 (spilling) 36 us.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef f32x4_t __attribute__((aligned(4))) f32x4_u;
constexpr int kInferBlocks = 768;

// hi = v rounded to bf16, so v - hi is exact in fp32; lo = that remainder
// rounded: |v - hi - lo| <= 2^-9 |v - hi| <= 2^-18 |v|. Values 2 e and
// 2 e + 1 go to word e.
__device__ __forceinline__ void split_bf16(float v0, float v1, uint32_t& hi, uint32_t& lo) {
  typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
  const pair_t h = {(__bf16)v0, (__bf16)v1};
  hi = __builtin_bit_cast(uint32_t, h);
  asm("" : "+v"(hi));  // else v0 is converted again for its own remainder
  const pair_t r = {(__bf16)(v0 - __uint_as_float(hi << 16)),
                    (__bf16)(v1 - __uint_as_float(hi & 0xFFFF0000u))};
  lo = __builtin_bit_cast(uint32_t, r);
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t __attribute__((aligned(2))) u32_2b_t;  // two bf16 weights, aligned as one

__device__ __forceinline__ f32x4_t mfma32(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// max(v, 0), 0 for NaN, at most the largest bfloat16: one instruction, where
// fmaxf takes two (it quiets its operand first).
__device__ __forceinline__ float relu(float v) {
  return __builtin_amdgcn_fmed3f(v, 0.0f, __uint_as_float(0x7F7F0000u));
}

// One hidden layer: acc (the previous layer's four D tiles) becomes this
// layer's, through ReLU and the split. k-steps run outermost, so consecutive
// MFMAs write different accumulators.
__device__ __forceinline__ void split_relu(const f32x4_t (&acc)[4], u32x4_t (&hi)[2],
                                           u32x4_t (&lo)[2]) {
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x4_t& v = acc[2 * s + e / 2];
      uint32_t h, l;
      split_bf16(relu(v[2 * (e % 2)]), relu(v[2 * (e % 2) + 1]), h, l);
      hi[s][e] = h;
      lo[s][e] = l;
    }
}

template <class Bias>
__device__ __forceinline__ void hidden_layer(const u32x4_t (&a)[4][2], Bias bias,
                                             f32x4_t (&acc)[4]) {
  u32x4_t hi[2], lo[2];
  split_relu(acc, hi, lo);
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = bias(t);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = mfma32(a[t][s], hi[s], acc[t]);
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = mfma32(a[t][s], lo[s], acc[t]);
  }
}

// Feature 4: a parent node's far count (scale * 2^y of its predicted log2
// rate), log-scaled.
__device__ __forceinline__ float far_feature(float far) {
  return log2f(1.0f + fmaxf(far, 0.0f)) / 16.0f;
}

constexpr float kLn2 = 0.69314718055994531f;
constexpr float kMaxLogRate = 30.0f;

// PARENT: feature 4 of node k is not read from x but made from y0, the first
// pass's outputs, at the node's parent (0 for a root), as k_mlp_far_of and
// k_mlp_features make it.
template <bool PARENT>
__global__ __launch_bounds__(256, 3) void k_mlp_infer(const uint16_t* __restrict__ wbf,
                                                      const float* __restrict__ x, int64_t n,
                                                      const int32_t* __restrict__ parent,
                                                      const float* __restrict__ y0, float s0,
                                                      float* __restrict__ y) {
  const unsigned l = lane_id();
  const int r = (int)(l % 16), q = (int)(l / 16);
  // The weights pass through LDS: one coalesced read per workgroup, then each
  // lane gathers its fragments there. Rows of 64 are kept at a pitch of 68.
  constexpr int kPitch = kH + 4;
  __shared__ __align__(16) uint16_t s_w1[kH * kIn], s_w2[kH * kPitch], s_w3[kH * kPitch],
      s_w4[kOut * kPitch];
  __shared__ __align__(16) float s_b[3][kH];
  for (int e = threadIdx.x; e < kH * kH / 2; e += 256) {
    const int at = 2 * e / kH * kPitch + 2 * e % kH;
    *(uint32_t*)(s_w2 + at) = *(const u32_2b_t*)(wbf + kOffW2 + 2 * e);
    *(uint32_t*)(s_w3 + at) = *(const u32_2b_t*)(wbf + kOffW3 + 2 * e);
  }
  {
    const int e = threadIdx.x;  // 256 threads = kH * kIn / 2
    *(uint32_t*)(s_w1 + 2 * e) = *(const u32_2b_t*)(wbf + kOffW1 + 2 * e);
    if (e < kOut * kH) s_w4[e / kH * kPitch + e % kH] = wbf[kOffW4 + e];
    if (e < kH) {
      s_b[0][e] = bf16_to_f32(wbf[kOffB1 + e]);
      s_b[1][e] = bf16_to_f32(wbf[kOffB2 + e]);
      s_b[2][e] = bf16_to_f32(wbf[kOffB3 + e]);
    }
  }
  f32x4_t b4;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float w4 = bf16_to_f32(wbf[kOffB4 + min(4 * q + e, kOut - 1)]);
    b4[e] = 4 * q + e < kOut ? w4 : 0.0f;
  }
  __syncthreads();
  u32x4_t a1[4], a2[4][2], a3[4][2], a4[2];
  // slots (q, 0..3) and (q, 4..7) of k-step s: inputs 32 s + 4 q and
  // 32 s + 16 + 4 q, four each
  auto frag = [&](const uint16_t* row, int s) {
    const uint2 lo = *(const uint2*)(row + 32 * s + 4 * q);
    const uint2 hi = *(const uint2*)(row + 32 * s + 16 + 4 * q);
    return u32x4_t{lo.x, lo.y, hi.x, hi.y};
  };
  constexpr u32x4_t kZero = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const u32x4_t w1 = *(const u32x4_t*)(s_w1 + (16 * t + r) * kIn);
    a1[t] = q < 2 ? w1 : kZero;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      a2[t][s] = frag(s_w2 + (16 * t + r) * kPitch, s);
      a3[t][s] = frag(s_w3 + (16 * t + r) * kPitch, s);
    }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const u32x4_t w4 = frag(s_w4 + min(r, kOut - 1) * kPitch, s);
    a4[s] = r < kOut ? w4 : kZero;
  }
  // biases stay in LDS (one 16-byte read per output tile): in registers they
  // would cost the third wavefront
  auto bias = [&](int layer, int t) { return *(const f32x4_t*)(&s_b[layer][16 * t + 4 * q]); };

  // Wave-uniform loop over 16-sample tiles (every lane reaches every
  // MFMA); the next tile's features are loaded while this one runs, by
  // unconditional loads (a lane past the last sample reads that one and
  // writes nothing; conditional loads had been a branch each).
  const int64_t tiles = (n + 15) / 16;
  const int64_t nw = (int64_t)gridDim.x * (blockDim.x / YGG_WAVE);
  struct In {
    f32x4_u f[2];
  };
  auto load_tile = [&](int64_t tl) {
    int64_t sm = tl * 16 + r;
    sm = sm < n ? sm : n - 1;
    In v;
    v.f[0] = *(const f32x4_u*)(x + sm * kIn);
    v.f[1] = *(const f32x4_u*)(x + sm * kIn + 4);
    if (PARENT) {
      const int32_t p = parent[sm];
      const float far = s0 * exp2f(fminf(y0[kOut * (int64_t)max(p, 0)], kMaxLogRate));
      v.f[1][0] = p >= 0 ? far_feature(far) : 0.0f;
    }
    return v;
  };
  int64_t tile = (int64_t)blockIdx.x * (blockDim.x / YGG_WAVE) + threadIdx.x / YGG_WAVE;
  if (tile >= tiles) return;
  In in_next = load_tile(tile);
  for (; tile < tiles; tile += nw) {
    const In in = in_next;
    if (tile + nw < tiles) in_next = load_tile(tile + nw);
    u32x4_t b;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t hi, lo;
      split_bf16(in.f[e / 2][2 * (e % 2)], in.f[e / 2][2 * (e % 2) + 1], hi, lo);
      b[e] = q == 0 ? hi : (q == 1 ? lo : 0u);
    }
    f32x4_t acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = mfma32(a1[t], b, bias(0, t));
    hidden_layer(a2, [&](int t) { return bias(1, t); }, acc);
    hidden_layer(a3, [&](int t) { return bias(2, t); }, acc);
    u32x4_t hi[2], lo[2];
    split_relu(acc, hi, lo);
    f32x4_t out = b4;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      out = mfma32(a4[s], hi[s], out);
      out = mfma32(a4[s], lo[s], out);
    }
    const int64_t smp = tile * 16 + r;
    if (q == 0 && smp < n) {
#pragma unroll
      for (int j = 0; j < kOut; ++j) y[smp * kOut + j] = out[j];
    }
  }
}

// ---- training: one kernel for a batch's gradients, one for the update ----
// k_train_grads: a workgroup takes kRows batch rows at a time through the
// forward pass, the masked Poisson loss (rate 2^y, y clamped at 30; per
// element m (2^y - t y ln 2) / B, gradient m (2^y - t) ln 2 / B) and the
// backward pass with every activation and delta in LDS, and keeps its weight
// gradients in MFMA accumulators until its last rows. It then writes one
// slice of partial sums (the parameters' layout, the loss after them);
// k_train_update adds the slices in a fixed order and takes the Adam step.
//
// The products run on v_mfma_f32_16x16x4_f32 (fp32 operands and sums):
//   A[m][k]: lane l holds A[l % 16][l / 16]
//   B[k][n]: lane l holds B[l / 16][l % 16]
//   D[m][n]: lane l holds D[4 (l / 16) + j][l % 16], j = 0..3
// and where k runs along a row of LDS, step s of lane group q takes
// k = 16 q + s, so that a lane's operands of four steps are one 16-byte read.
//
// Bound by its own chain of ten phases (each a few thousand MFMA cycles a
// workgroup), no longer by eighteen dependent launches; kRows = 32 gives a
// batch of 4096 a workgroup on every second CU and halves the slices'
// traffic against 16.
// A step of 4096 rows takes 22 us, against
// 208 us for eighteen launches (a layer at a time through memory, 4-byte
// operand reads).
constexpr int kRows = 32;
constexpr int kLd = kH + 4;     // LDS row: 16-byte aligned, bank-shifted
constexpr int kTrainBlocks = 256;
constexpr int kSlice = (kParams + 1 + 15) / 16 * 16;  // floats per slice, loss at kParams

__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// acc[16 x 16] += A-row r times B-row r over k = 0..63 (both rows in LDS).
__device__ __forceinline__ f32x4_t dot_rows(const float* a, const float* b, int q, f32x4_t acc) {
#pragma unroll
  for (int s = 0; s < 16; s += 4) {
    const f32x4_t av = *(const f32x4_t*)(a + 16 * q + s), bv = *(const f32x4_t*)(b + 16 * q + s);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = mfma4(av[j], bv[j], acc);
  }
  return acc;
}

// acc[16 x 16] += A-row r times B-column (LDS rows k, column c) over k = 0..63.
__device__ __forceinline__ f32x4_t dot_cols(const float* a, const float (*b)[kLd], int c, int q,
                                            f32x4_t acc) {
#pragma unroll
  for (int s = 0; s < 16; s += 4) {
    const f32x4_t av = *(const f32x4_t*)(a + 16 * q + s);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = mfma4(av[j], b[16 * q + s + j][c], acc);
  }
  return acc;
}

__global__ __launch_bounds__(256) void k_train_grads(const uint16_t* __restrict__ W,
                                                     const float* __restrict__ x,
                                                     const float* __restrict__ target,
                                                     const float* __restrict__ mask, int64_t B,
                                                     float* __restrict__ partial) {
  __shared__ __align__(16) float s_w2[kH][kLd], s_w3[kH][kLd];
  __shared__ __align__(16) float s_a1[kRows][kLd], s_a2[kRows][kLd], s_a3[kRows][kLd];
  __shared__ __align__(16) float s_d[2][kRows][kLd];
  __shared__ float s_w1[kH][kIn + 1], s_w4[kOut][kH], s_x[kRows][kIn + 1], s_dy[kRows][kOut + 1];
  __shared__ float s_loss[2];
  const int tid = threadIdx.x, lane = (int)lane_id(), r = lane % 16, q = lane / 16;
  const int w = tid / YGG_WAVE, n0 = 16 * w;
  for (int e = tid; e < kH * kH; e += 256) {
    s_w2[e / kH][e % kH] = bf16_to_f32(W[kOffW2 + e]);
    s_w3[e / kH][e % kH] = bf16_to_f32(W[kOffW3 + e]);
  }
  for (int e = tid; e < kH * kIn; e += 256) s_w1[e / kIn][e % kIn] = bf16_to_f32(W[kOffW1 + e]);
  if (tid < kOut * kH) s_w4[tid / kH][tid % kH] = bf16_to_f32(W[kOffW4 + tid]);
  const float bias1 = bf16_to_f32(W[kOffB1 + n0 + r]), bias2 = bf16_to_f32(W[kOffB2 + n0 + r]),
              bias3 = bf16_to_f32(W[kOffB3 + n0 + r]),
              bias4 = r < kOut ? bf16_to_f32(W[kOffB4 + r]) : 0.0f;
  // this workgroup's gradients: wavefront w holds outputs [16 w, 16 w + 16)
  // of the hidden layers, thread tid one weight of the last and one bias
  f32x4_t g1 = {0.0f, 0.0f, 0.0f, 0.0f}, g2[4], g3[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) g2[t] = g3[t] = g1;
  float g4 = 0.0f, gb = 0.0f, loss = 0.0f;

  for (int64_t base = (int64_t)blockIdx.x * kRows; base < B; base += (int64_t)gridDim.x * kRows) {
    const int rows = B - base < kRows ? (int)(B - base) : kRows;
    __syncthreads();  // weights staged; the previous rows' last phase is done
    {
      const int b = tid / kIn, i = tid % kIn;  // 256 threads = kRows x kIn
      s_x[b][i] = b < rows ? x[(base + b) * kIn + i] : 0.0f;
    }
    __syncthreads();
    // rows past the batch hold zeros in every activation and delta
    auto put = [&](float (*dst)[kLd], int rt, const f32x4_t& v) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int b = 16 * rt + 4 * q + j;
        dst[b][n0 + r] = b < rows ? fmaxf(v[j], 0.0f) : 0.0f;
      }
    };
#pragma unroll
    for (int rt = 0; rt < kRows / 16; ++rt) {
      f32x4_t acc = {bias1, bias1, bias1, bias1};
#pragma unroll
      for (int k0 = 0; k0 < kIn; k0 += 4)
        acc = mfma4(s_x[16 * rt + r][k0 + q], s_w1[n0 + r][k0 + q], acc);
      put(s_a1, rt, acc);
    }
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < kRows / 16; ++rt)
      put(s_a2, rt, dot_rows(s_a1[16 * rt + r], s_w2[n0 + r], q, f32x4_t{bias2, bias2, bias2, bias2}));
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < kRows / 16; ++rt)
      put(s_a3, rt, dot_rows(s_a2[16 * rt + r], s_w3[n0 + r], q, f32x4_t{bias3, bias3, bias3, bias3}));
    __syncthreads();
    if (w < kRows / 16) {  // outputs and loss: wavefront w takes rows [16 w, 16 w + 16)
      f32x4_t acc = {bias4, bias4, bias4, bias4};
#pragma unroll
      for (int s = 0; s < 16; s += 4) {
        const f32x4_t av = *(const f32x4_t*)(&s_a3[n0 + r][16 * q + s]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc = mfma4(av[j], r < kOut ? s_w4[r][16 * q + s + j] : 0.0f, acc);
      }
      if (r < kOut) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int b = n0 + 4 * q + j;
          float dy = 0.0f;
          if (b < rows) {
            const int64_t e = (base + b) * kOut + r;
            const float t = target[e], m = mask[e], yv = acc[j];
            const float yc = fminf(yv, kMaxLogRate), lam = exp2f(yc);
            dy = yv > kMaxLogRate ? 0.0f : m * (lam - t) * kLn2 / (float)B;
            loss += m * (lam - t * yc * kLn2) / (float)B;
          }
          s_dy[b][r] = dy;
        }
      }
    }
    __syncthreads();
    // deltas of the third layer, gradients of the last
    for (int e = tid; e < kRows * kH; e += 256) {
      const int b = e / kH, i = e % kH;
      float d = 0.0f;
#pragma unroll
      for (int o = 0; o < kOut; ++o) d += s_dy[b][o] * s_w4[o][i];
      s_d[0][b][i] = s_a3[b][i] > 0.0f ? d : 0.0f;
    }
    if (tid < kOut * kH) {
      const int o = tid / kH, i = tid % kH;
#pragma unroll 8
      for (int b = 0; b < kRows; ++b) g4 += s_dy[b][o] * s_a3[b][i];
    } else if (tid < kOut * kH + kOut) {
      for (int b = 0; b < kRows; ++b) gb += s_dy[b][tid - kOut * kH];
    }
    __syncthreads();
    // weight gradients of a hidden layer (m = output, n = input, k = row),
    // and its bias gradients in 64 threads of their own
    auto weight_grads = [&](const float (*d)[kLd], const float (*a)[kLd], f32x4_t (&g)[4]) {
#pragma unroll
      for (int b0 = 0; b0 < kRows; b0 += 4) {
        const float dv = d[b0 + q][n0 + r];
#pragma unroll
        for (int t = 0; t < 4; ++t) g[t] = mfma4(dv, a[b0 + q][16 * t + r], g[t]);
      }
    };
    auto bias_grads = [&](const float (*d)[kLd], int wave) {
      if (w == wave)
        for (int b = 0; b < kRows; ++b) gb += d[b][lane];
    };
    // deltas of the layer below: d W, where the ReLU passed
    auto down = [&](const float (*d)[kLd], const float (*wt)[kLd], const float (*a)[kLd],
                    float (*out)[kLd]) {
#pragma unroll
      for (int rt = 0; rt < kRows / 16; ++rt) {
        const f32x4_t v = dot_cols(d[16 * rt + r], wt, n0 + r, q, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int b = 16 * rt + 4 * q + j;
          out[b][n0 + r] = a[b][n0 + r] > 0.0f ? v[j] : 0.0f;
        }
      }
    };
    weight_grads(s_d[0], s_a2, g3);
    bias_grads(s_d[0], 0);
    down(s_d[0], s_w3, s_a2, s_d[1]);
    __syncthreads();
    weight_grads(s_d[1], s_a1, g2);
    bias_grads(s_d[1], 1);
    down(s_d[1], s_w2, s_a1, s_d[0]);
    __syncthreads();
#pragma unroll
    for (int b0 = 0; b0 < kRows; b0 += 4)
      g1 = mfma4(s_d[0][b0 + q][n0 + r], r < kIn ? s_x[b0 + q][r] : 0.0f, g1);
    bias_grads(s_d[0], 2);
  }

  float* __restrict__ out = partial + (int64_t)blockIdx.x * kSlice;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int o = n0 + 4 * q + j;
    if (r < kIn) out[kOffW1 + o * kIn + r] = g1[j];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      out[kOffW2 + o * kH + 16 * t + r] = g2[t][j];
      out[kOffW3 + o * kH + 16 * t + r] = g3[t][j];
    }
  }
  if (tid < kOut * kH) out[kOffW4 + tid] = g4;
  // biases: wavefronts 0, 1, 2 hold those of layers 3, 2, 1, and the first
  // kOut threads of wavefront 3 the last layer's
  if (w < 3)
    out[(w == 0 ? kOffB3 : (w == 1 ? kOffB2 : kOffB1)) + lane] = gb;
  else if (lane < kOut)
    out[kOffB4 + lane] = gb;
  loss = wave_sum_f(loss);
  if (lane == 0 && w < 2) s_loss[w] = loss;
  __syncthreads();
  if (tid == 0) out[kParams] = s_loss[0] + s_loss[1];
}

// grads[i] = the sum of the slices' i-th entries (eight interleaved chains,
// added in order), then the Adam step where lr > 0; entry kParams is the
// loss. 32 consecutive entries and 8 chains to a workgroup.
__global__ __launch_bounds__(256) void k_train_update(
    const float* __restrict__ partial, int slices, float* __restrict__ grads,
    float* __restrict__ loss_out, float* __restrict__ p, float* __restrict__ m,
    float* __restrict__ v, uint16_t* __restrict__ pbf, float lr, float b1, float b2, float eps,
    float c1, float c2) {
  __shared__ float s_sum[8][32];
  const int c = threadIdx.x / 32, i = blockIdx.x * 32 + threadIdx.x % 32;
  float acc = 0.0f;
  if (i <= kParams) {
#pragma unroll 4
    for (int s = c; s < slices; s += 8) acc += partial[(int64_t)s * kSlice + i];
  }
  s_sum[c][threadIdx.x % 32] = acc;
  __syncthreads();
  if (c || i > kParams) return;
  float gi = acc;
#pragma unroll
  for (int k = 1; k < 8; ++k) gi += s_sum[k][threadIdx.x];
  if (i == kParams) {
    if (loss_out) *loss_out = gi;
    return;
  }
  grads[i] = gi;
  if (!(lr > 0.0f)) return;
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float upd = lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  const float np = p[i] - upd;
  p[i] = np;
  pbf[i] = f32_to_bf16(np);
}

__global__ void k_to_bf16(const float* __restrict__ p, uint16_t* __restrict__ q, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) q[i] = f32_to_bf16(p[i]);
}

__global__ void k_zero_words(uint32_t* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0u;
}

// ---- per-node features ------------------------------------------------------
// Features of node k of one tree whose arrays start at the given bases
// (root = node 0 of the tree; parent/children/sibling ids local).
__device__ __forceinline__ void node_features(int k, int NI, const int32_t* __restrict__ node_level,
                                              const int32_t* __restrict__ ranges,
                                              const int32_t* __restrict__ parent,
                                              const int32_t* __restrict__ left,
                                              const int32_t* __restrict__ right,
                                              const float* __restrict__ half,
                                              const float* __restrict__ radius,
                                              const float* __restrict__ maxext,
                                              const float* __restrict__ parent_far,
                                              float* __restrict__ o) {
  const float root_ext = maxext[0], root_rad = radius[0];
  const float root_vol = 8.0f * half[0] * half[1] * half[2];
  float cnt = (float)(ranges[2 * k + 1] - ranges[2 * k] + 1);
  int p = parent[k];
  float sib = 0.0f;
  if (p >= 0) {
    int sb = left[p] == k ? right[p] : left[p];
    sib = (float)(ranges[2 * sb + 1] - ranges[2 * sb] + 1);
  }
  float vol = 8.0f * half[3 * k] * half[3 * k + 1] * half[3 * k + 2];
  float pf = (parent_far && p >= 0) ? parent_far[p] : 0.0f;
  o[0] = (float)node_level[k] / 64.0f;
  o[1] = log2f(cnt) / 24.0f;
  o[2] = log2f(maxext[k] / root_ext) / 32.0f + 1.0f;
  o[3] = log2f(radius[k] / root_rad) / 32.0f + 1.0f;
  o[4] = far_feature(pf);
  o[5] = log2f(1.0f + sib) / 24.0f;
  float rel = (cnt / fmaxf(vol, 1e-30f)) / ((float)(ranges[1] + 1) / fmaxf(root_vol, 1e-30f));
  o[6] = fminf(fmaxf(log2f(fmaxf(rel, 1e-30f)) / 64.0f, -1.0f), 1.0f);
  o[7] = k >= NI ? 1.0f : 0.0f;
}

__global__ void k_mlp_features(int T, int NI, const int32_t* __restrict__ node_level,
                               const int32_t* __restrict__ ranges,
                               const int32_t* __restrict__ parent,
                               const int32_t* __restrict__ left,
                               const int32_t* __restrict__ right,
                               const float* __restrict__ half, const float* __restrict__ radius,
                               const float* __restrict__ maxext,
                               const float* __restrict__ parent_far, float* __restrict__ x) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= T) return;
  node_features(k, NI, node_level, ranges, parent, left, right, half, radius, maxext, parent_far,
                x + (int64_t)k * kIn);
}

// Batched: every node of every system, with its own tree's root.
__global__ void k_b_mlp_features(Seg sg, int64_t Ttot, const int32_t* __restrict__ node_level,
                                 const int32_t* __restrict__ ranges,
                                 const int32_t* __restrict__ parent,
                                 const int32_t* __restrict__ left,
                                 const int32_t* __restrict__ right,
                                 const float* __restrict__ half, const float* __restrict__ radius,
                                 const float* __restrict__ maxext,
                                 const float* __restrict__ parent_far, float* __restrict__ x) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (g >= Ttot) return;
  const int s = sg.of_node(g);
  const int64_t n0 = sg.node_off(s), ni0 = sg.ni_off(s);
  node_features((int)(g - n0), sg.L(s) - 1, node_level + n0, ranges + 2 * n0, parent + n0,
                left + ni0, right + ni0, half + 3 * n0, radius + n0, maxext + n0,
                parent_far ? parent_far + n0 : nullptr, x + g * kIn);
}

// Batched totals: output 1 (near) counts each system's leaves.
// Adds a workgroup's three partial sums into tot[0..2]: wavefront
// shuffles, then one LDS row per wavefront and three atomics per workgroup
// (same-address device atomics serialise across XCDs, so the grids of the
// totals kernels are kept at kTotalsBlocks workgroups).
constexpr int kTotalsBlocks = 128;

__device__ __forceinline__ void block_add3(double a0, double a1, double a2, double* tot) {
  __shared__ double red[256 / YGG_WAVE][3];
  for (int off = 32; off > 0; off >>= 1) {
    a0 += __shfl_xor(a0, off, 64);
    a1 += __shfl_xor(a1, off, 64);
    a2 += __shfl_xor(a2, off, 64);
  }
  const int w = threadIdx.x / YGG_WAVE;
  if (lane_id() == 0) {
    red[w][0] = a0;
    red[w][1] = a1;
    red[w][2] = a2;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double v = 0;
    for (int q = 0; q < (int)(blockDim.x / YGG_WAVE); ++q) v += red[q][threadIdx.x];
    atomicAdd(&tot[threadIdx.x], v);
  }
}

__global__ __launch_bounds__(256) void k_b_mlp_totals(Seg sg, const float* __restrict__ y,
                                                      int64_t n, float s0, float s1, float s2,
                                                      double* __restrict__ tot) {
  __shared__ int32_t s_noff[kSegLdsCap];
  const bool staged = seg_stage(s_noff, sg.S, [&](int s) { return (int32_t)sg.node_off(s); });
  __syncthreads();
  double a0 = 0, a1 = 0, a2 = 0;
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n;
       g += (int64_t)gridDim.x * blockDim.x) {
    const int s = staged ? seg_find_lds(s_noff, sg.S, g) : sg.of_node(g);
    a0 += (double)(s0 * exp2f(fminf(y[3 * g], kMaxLogRate)));
    if (g - sg.node_off(s) >= sg.L(s) - 1)
      a1 += (double)(s1 * exp2f(fminf(y[3 * g + 1], kMaxLogRate)));
    a2 += (double)(s2 * exp2f(fminf(y[3 * g + 2], kMaxLogRate)));
  }
  block_add3(a0, a1, a2, tot);
}

// Sum of scale_j 2^y_j per output over [0, n) (stream totals), y row-major
// [n][3]; output 1 (near) counts leaves only.
__global__ __launch_bounds__(256) void k_mlp_totals(const float* __restrict__ y, int64_t n,
                                                    int64_t NI, float s0, float s1, float s2,
                                                    double* __restrict__ tot) {
  double a0 = 0, a1 = 0, a2 = 0;
  for (int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; s < n;
       s += (int64_t)gridDim.x * blockDim.x) {
    a0 += (double)(s0 * exp2f(fminf(y[3 * s], kMaxLogRate)));
    if (s >= NI) a1 += (double)(s1 * exp2f(fminf(y[3 * s + 1], kMaxLogRate)));
    a2 += (double)(s2 * exp2f(fminf(y[3 * s + 2], kMaxLogRate)));
  }
  block_add3(a0, a1, a2, tot);
}

// far[k] = s0 2^y[k][0] (the first pass's far-count prediction).
__global__ void k_mlp_far_of(const float* __restrict__ y, int T, float s0, float* __restrict__ pf) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < T) pf[k] = s0 * exp2f(fminf(y[3 * k], kMaxLogRate));
}

}  // namespace ygg

using namespace ygg;

extern "C" {

int ygg_mlp_num_params(void) { return kParams; }

// 16-sample tiles, four wavefronts per workgroup, at most kInferBlocks
// workgroups: three wavefronts per SIMD (the kernel's occupancy), each
// gathering the weight fragments once and then looping over many tiles.
static dim3 infer_grid(int64_t n) {
  return dim3(grid_for((n + 15) / 16, 256 / YGG_WAVE, kInferBlocks));
}

int ygg_mlp_forward(const uint16_t* params_bf16, const float* features, int64_t n,
                    float* outputs, void* stream) {
  if (n < 0 || !params_bf16) return YGG_ERR_ARG;
  if (n == 0) return YGG_OK;
  hipLaunchKernelGGL(k_mlp_infer<false>, infer_grid(n), dim3(256), 0, (hipStream_t)stream,
                     params_bf16, features, n, nullptr, nullptr, 0.0f, outputs);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

int ygg_mlp_forward_parent(const uint16_t* params_bf16, const float* features, int64_t n,
                           const int32_t* parent, const float* first_outputs, float scale_far,
                           float* outputs, void* stream) {
  if (n < 0 || !params_bf16 || !parent || !first_outputs) return YGG_ERR_ARG;
  if (n == 0) return YGG_OK;
  hipLaunchKernelGGL(k_mlp_infer<true>, infer_grid(n), dim3(256), 0, (hipStream_t)stream,
                     params_bf16, features, n, parent, first_outputs, scale_far, outputs);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

// Workgroups of k_train_grads, and so slices of partial sums, for a batch.
static int64_t train_slices(int64_t B) {
  const int64_t s = (B + kRows - 1) / kRows;
  return s < kTrainBlocks ? s : kTrainBlocks;
}

// One training step on a batch: forward, masked Poisson loss, backward, Adam.
// ws: float workspace of ygg_mlp_train_workspace_floats(B) entries.
int64_t ygg_mlp_train_workspace_floats(int64_t B) { return train_slices(B) * kSlice; }

int ygg_mlp_train_step(float* params, uint16_t* params_bf16, float* adam_m, float* adam_v,
                       int64_t step, float lr, const float* x, const float* target,
                       const float* mask, int64_t B64, float* grads, float* ws,
                       float* loss_out, void* stream) {
  if (B64 < 1 || !params || !grads || !ws) return YGG_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  const int slices = (int)train_slices(B64);
  hipLaunchKernelGGL(k_train_grads, dim3(slices), dim3(256), 0, st, params_bf16, x, target, mask,
                     B64, ws);
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_train_update, dim3((kParams + 1 + 31) / 32), dim3(256), 0, st, ws, slices,
                     grads, loss_out, params, adam_m, adam_v, params_bf16, lr, b1, b2, 1e-8f, c1,
                     c2);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

int ygg_mlp_params_to_bf16(const float* params, uint16_t* params_bf16, void* stream) {
  hipLaunchKernelGGL(k_to_bf16, dim3(grid_for(kParams, 256)), dim3(256), 0, (hipStream_t)stream,
                     params, params_bf16, kParams);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

int ygg_mlp_features(int64_t num_nodes, const int32_t* node_level, const int32_t* node_ranges,
                     const int32_t* parent, const int32_t* left, const int32_t* right,
                     const float* half_extent, const float* radius, const float* max_extent,
                     const float* parent_far, float* features, void* stream) {
  if (num_nodes < 1) return YGG_ERR_ARG;
  int T = (int)num_nodes, NI = (T - 1) / 2;
  hipLaunchKernelGGL(k_mlp_features, dim3(grid_for(T, 256)), dim3(256), 0, (hipStream_t)stream, T,
                     NI, node_level, node_ranges, parent, left, right, half_extent, radius,
                     max_extent, parent_far, features);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

int ygg_mlp_totals(const float* outputs, int64_t num_nodes, float scale_far, float scale_near,
                   float scale_queue, double* totals, void* stream) {
  if (num_nodes < 1 || !outputs || !totals) return YGG_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(64), 0, st, (uint32_t*)totals, 6);
  hipLaunchKernelGGL(k_mlp_totals, dim3(grid_for(num_nodes, 256, kTotalsBlocks)), dim3(256), 0, st,
                     outputs, num_nodes, (num_nodes - 1) / 2, scale_far, scale_near, scale_queue,
                     totals);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

int ygg_mlp_far_counts(const float* outputs, int64_t num_nodes, float scale_far,
                       float* far_counts, void* stream) {
  if (num_nodes < 1 || !outputs || !far_counts) return YGG_ERR_ARG;
  hipLaunchKernelGGL(k_mlp_far_of, dim3(grid_for(num_nodes, 256)), dim3(256), 0,
                     (hipStream_t)stream, outputs, (int)num_nodes, scale_far, far_counts);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

static inline Seg mlp_seg(const YggBatch* b) {
  Seg sg;
  sg.S = b->num_systems;
  sg.leaf_size = b->leaf_size;
  sg.pt = b->point_offsets;
  sg.leaf = b->leaf_offsets;
  return sg;
}

int ygg_batch_mlp_features(const YggBatch* b, const int32_t* node_level,
                           const int32_t* node_ranges, const int32_t* parent, const int32_t* left,
                           const int32_t* right, const float* half_extent, const float* radius,
                           const float* max_extent, const float* parent_far, float* features,
                           void* stream) {
  if (!b || b->num_systems < 1 || !features) return YGG_ERR_ARG;
  const int64_t T = 2 * b->num_leaves - b->num_systems;
  hipLaunchKernelGGL(k_b_mlp_features, dim3(grid_for(T, 256)), dim3(256), 0, (hipStream_t)stream,
                     mlp_seg(b), T, node_level, node_ranges, parent, left, right, half_extent,
                     radius, max_extent, parent_far, features);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

int ygg_batch_mlp_totals(const YggBatch* b, const float* outputs, float scale_far,
                         float scale_near, float scale_queue, double* totals, void* stream) {
  if (!b || b->num_systems < 1 || !outputs || !totals) return YGG_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  const int64_t T = 2 * b->num_leaves - b->num_systems;
  hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(64), 0, st, (uint32_t*)totals, 6);
  hipLaunchKernelGGL(k_b_mlp_totals, dim3(grid_for(T, 256, kTotalsBlocks)), dim3(256), 0, st, mlp_seg(b),
                     outputs, T, scale_far, scale_near, scale_queue, totals);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

}  // extern "C"
