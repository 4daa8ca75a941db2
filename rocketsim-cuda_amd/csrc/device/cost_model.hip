// The learned cost model: a 48 -> 64 -> 64 -> 2 MLP that predicts, from an arena's state, the log of its decision's cost
// (wall-clock ticks of a wave running that arena alone) and a contact logit; and the kernels that regroup arenas by it.
//
//   k_features     48 features per arena from the AoSoA-64 states (positions, velocities, wall and gap distances, counts)
//   k_mlp_infer    inference: bf16 weights and activations, fp32 accumulation, on v_mfma_f32_16x16x16_bf16, weights and
//                  activations in registers
//   k_mlp_train    training forward + backward in fp32 (the same bf16 rounding points as inference; the rounding is treated
//                  as the identity in the backward pass), and each work-group's share of the parameter gradient
//   k_mlp_reduce   the parameter gradient: the sum of the shares
//   k_adam         Adam update of the fp32 master parameters
//   k_gather_words / k_scatter_words / k_gather_states   the regrouping permutations (states stay AoSoA-64)
//
// Parameter vector (fp32): W1[48][64], b1[64], W2[64][64], b2[64], W3[64][2], b3[2] (W[i][j]: input i -> output j).
#include "device/cost_model.h"

namespace rs {
namespace dev {
namespace {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ inline uint16_t bf16_bits(float x) {  // round to nearest even (finite inputs)
  uint32_t u = __builtin_bit_cast(uint32_t, x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ inline float bf16_round(float x) { return __builtin_bit_cast(float, (uint32_t)bf16_bits(x) << 16); }

__device__ inline uint32_t word_of(const uint32_t* buf, uint32_t a, size_t w) {
  return buf[(size_t)(a / AOSOA_LANES) * ARENA_WORDS * AOSOA_LANES + w * AOSOA_LANES + (a % AOSOA_LANES)];
}
__device__ inline float fword(const uint32_t* buf, uint32_t a, size_t byte_off) { return __builtin_bit_cast(float, word_of(buf, a, byte_off / 4)); }
__device__ inline V3 vword(const uint32_t* buf, uint32_t a, size_t byte_off) {
  return V3{fword(buf, a, byte_off), fword(buf, a, byte_off + 4), fword(buf, a, byte_off + 8)};
}
__device__ inline float clamp1(float x) { return x < -4.0f ? -4.0f : (x > 4.0f ? 4.0f : x); }

}  // namespace

// ---- features ------------------------------------------------------------------------------------------------------------------
// One wave per AoSoA block: each lane reads its arena's words (256-byte rows) and computes its features; the rows of 48 then
// leave through LDS, so that the wave writes its 12 KB as one run. Bound by the latency of one round of loads.
constexpr int FEATURE_STRIDE = COST_FEATURES + 1;  // odd: lanes writing the same feature hit distinct banks
__global__ void __launch_bounds__(64) k_features(const uint32_t* __restrict__ states, uint32_t n, float* __restrict__ feat) {
  __shared__ float rows[AOSOA_LANES * FEATURE_STRIDE];
  const uint32_t a0 = blockIdx.x * AOSOA_LANES, a = a0 + threadIdx.x;  // a lane past n reads the padding of its block
  float f[COST_FEATURES];
  const size_t ball = offsetof(ArenaState, ball);
  V3 bp = vword(states, a, ball + offsetof(Ball, pos)), bv = vword(states, a, ball + offsetof(Ball, vel));
  V3 bw = vword(states, a, ball + offsetof(Ball, ang_vel));
  const V3 field = V3{4096.0f, 5120.0f, 2044.0f};
  f[0] = bp.x / field.x, f[1] = bp.y / field.y, f[2] = bp.z / field.z;
  f[3] = bv.x / 6000.0f, f[4] = bv.y / 6000.0f, f[5] = bv.z / 6000.0f;
  f[6] = bw.x / 6.0f, f[7] = bw.y / 6.0f, f[8] = bw.z / 6.0f;
  V3 cp[NUM_CARS];
  for (int c = 0; c < NUM_CARS; ++c) {
    const size_t car = offsetof(ArenaState, cars) + (size_t)c * sizeof(Car);
    V3 p = vword(states, a, car + offsetof(Car, pos)), v = vword(states, a, car + offsetof(Car, vel));
    V3 w = vword(states, a, car + offsetof(Car, ang_vel));
    float up_z = fword(states, a, car + offsetof(Car, rot) + offsetof(M3, c2) + 8);
    float boost = fword(states, a, car + offsetof(Car, boost));
    uint32_t ground = word_of(states, a, (car + offsetof(Car, is_on_ground)) / 4);
    uint32_t demo = word_of(states, a, (car + offsetof(Car, is_demoed)) / 4);
    float* g = f + 9 + 13 * c;
    g[0] = p.x / field.x, g[1] = p.y / field.y, g[2] = p.z / field.z;
    g[3] = v.x / 2300.0f, g[4] = v.y / 2300.0f, g[5] = v.z / 2300.0f;
    g[6] = w.x / 5.5f, g[7] = w.y / 5.5f, g[8] = w.z / 5.5f;
    g[9] = boost / 100.0f, g[10] = ground ? 1.0f : 0.0f, g[11] = up_z, g[12] = demo ? 1.0f : 0.0f;
    cp[c] = p;
  }
  f[35] = (field.x - fabsf(bp.x)) / field.x, f[36] = (field.y - fabsf(bp.y)) / field.y, f[37] = (field.z - bp.z) / field.z;
  f[38] = (field.x - fabsf(cp[0].x)) / field.x, f[39] = (field.y - fabsf(cp[0].y)) / field.y;
  f[40] = (field.x - fabsf(cp[1].x)) / field.x, f[41] = (field.y - fabsf(cp[1].y)) / field.y;
  f[42] = length(cp[0] - cp[1]) / 1000.0f, f[43] = length(cp[0] - bp) / 1000.0f, f[44] = length(cp[1] - bp) / 1000.0f;
  f[45] = (float)word_of(states, a, offsetof(ArenaState, n_pairs) / 4) / 16.0f;
  f[46] = (float)word_of(states, a, offsetof(ArenaState, n_manifolds) / 4) / 16.0f;
  f[47] = (float)word_of(states, a, offsetof(ArenaState, n_dyn_cells) / 4) / 64.0f;
  for (int i = 0; i < COST_FEATURES; ++i) rows[threadIdx.x * FEATURE_STRIDE + i] = clamp1(f[i]);
  __syncthreads();
  const uint32_t words = (n - a0 < AOSOA_LANES ? n - a0 : AOSOA_LANES) * (uint32_t)COST_FEATURES;
  for (uint32_t e = threadIdx.x; e < words; e += 64u)
    feat[(size_t)a0 * COST_FEATURES + e] = rows[e / COST_FEATURES * FEATURE_STRIDE + e % COST_FEATURES];
}

// ---- inference on MFMA ---------------------------------------------------------------------------------------------------------
// v_mfma_f32_16x16x16_bf16 lane layout: A (16x16, rows x k): lane l holds row l % 16, k = 4 (l / 16) + 0..3; B (k x cols):
// col l % 16, k = 4 (l / 16) + 0..3; D (rows x cols): col l % 16, rows 4 (l / 16) + 0..3. The product is taken transposed,
// outputs as rows and arenas as columns: a layer's D is then, lane for lane, the next layer's B, so the activations stay in
// registers from the features to the prediction. The weights stay in registers too, as A operands (a column of 16 outputs'
// weights per lane), and each wave takes every waves-th tile of 16 arenas. Bound by reading the features: 65,536 arenas
// (12.6 MB) took 1,099 us with the weights staged in LDS by every wave of 64 arenas and the activations re-laid through LDS.
constexpr uint32_t INFER_WAVES = 2048;  // two per SIMD: a wave's weights and biases (98 words per lane) pay off over its tiles
__device__ inline v4s weight_frag(const float* __restrict__ w, int in0, int out, int stride, bool used) {
  v4s f = v4s{0, 0, 0, 0};
  if (used)
    for (int i = 0; i < 4; ++i) f[i] = (short)bf16_bits(w[(in0 + i) * stride + out]);
  return f;
}
__device__ inline v4s hidden_frag(v4f acc, v4f bias) {  // the layer's activation, rounded as the next layer's input
  v4s f;
  for (int i = 0; i < 4; ++i) {
    const float v = acc[i] + bias[i];
    f[i] = (short)bf16_bits(v > 0.0f ? v : 0.0f);
  }
  return f;
}
__global__ void __launch_bounds__(64) k_mlp_infer(const float* __restrict__ params, const float* __restrict__ feat, uint32_t n,
                                                  float* __restrict__ out) {
  const int l = threadIdx.x, lr = l % 16, lk = 4 * (l / 16);
  const float *W1 = params + COST_W1, *B1 = params + COST_B1, *W2 = params + COST_W2, *B2 = params + COST_B2,
              *W3 = params + COST_W3, *B3 = params + COST_B3;
  constexpr int K1 = COST_FEATURES / 16;  // 16-wide input steps of the first layer
  v4s w1[4][K1], w2[4][4], w3[4];
  v4f b1[4], b2[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int ks = 0; ks < K1; ++ks) w1[j][ks] = weight_frag(W1, ks * 16 + lk, j * 16 + lr, 64, true);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) w2[j][ks] = weight_frag(W2, ks * 16 + lk, j * 16 + lr, 64, true);
    w3[j] = weight_frag(W3, j * 16 + lk, lr, 2, lr < 2);
    for (int i = 0; i < 4; ++i) b1[j][i] = B1[j * 16 + lk + i], b2[j][i] = B2[j * 16 + lk + i];
  }
  const float b30 = B3[0], b31 = B3[1];
  for (uint32_t t = blockIdx.x; t < (n + 15) / 16; t += gridDim.x) {
    const uint32_t a = t * 16 + lr;
    v4s x[K1];
#pragma unroll
    for (int ks = 0; ks < K1; ++ks) {
      const float* row = feat + (size_t)(a < n ? a : n - 1) * COST_FEATURES + ks * 16 + lk;
      for (int i = 0; i < 4; ++i) x[ks][i] = (short)bf16_bits(row[i]);
    }
    v4s h1[4], h2[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v4f acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int ks = 0; ks < K1; ++ks) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w1[j][ks], x[ks], acc, 0, 0, 0);
      h1[j] = hidden_frag(acc, b1[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v4f acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w2[j][ks], h1[ks], acc, 0, 0, 0);
      h2[j] = hidden_frag(acc, b2[j]);
    }
    v4f y = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) y = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w3[ks], h2[ks], y, 0, 0, 0);
    if (l < 16 && a < n) {
      out[(size_t)a * 2] = y[0] + b30;
      out[(size_t)a * 2 + 1] = y[1] + b31;
    }
  }
}

// ---- training ------------------------------------------------------------------------------------------------------------------
// One work-group per TRAIN_ROWS batch rows (and every gridDim.x * TRAIN_ROWS further ones): the forward pass in fp32 with
// bf16-rounded weights and activations (the inference kernel's rounding points; each sum runs over its inputs in order, as
// one accumulator), the losses (squared error on the normalised log cost, logistic loss on the contact flag, both averaged
// over the batch), the backward pass, and the rows' share of the parameter gradient, kept in registers over the group's
// rows and written once. k_mlp_reduce sums the groups' shares in a fixed order.
//
// Forward: lane j of each wave holds column j of W1 and W2 in registers and takes eight rows, whose inputs it reads from LDS
// as broadcasts. The layer-1 gradient and the two weight gradients are contractions in fp32 and run on
// v_mfma_f32_16x16x4_f32 (A: row l % 16, k = l / 16; B: k = l / 16, column l % 16; D: rows 4 (l / 16) + 0..3, column
// l % 16). 4,096 rows: 128 groups, one wave per SIMD on half the CUs; bound by the forward's instruction chain. Before, one
// lane per row wrote its activations to memory and one thread per parameter summed 4,096 rows in turn: 1,340 us.
constexpr uint32_t TRAIN_ROWS = 32, TRAIN_MAX_GROUPS = 256;
constexpr int TS = 80;  // LDS row stride of the 64-wide activations: the four rows an MFMA operand reads fall in distinct banks
__global__ void __launch_bounds__(256) k_mlp_train(const float* __restrict__ params, const float* __restrict__ feat,
                                                   const float* __restrict__ target, const float* __restrict__ contact,
                                                   uint32_t b, float* __restrict__ shares, float* __restrict__ loss) {
  __shared__ float4 x4[TRAIN_ROWS * COST_FEATURES / 4], h14[TRAIN_ROWS * TS / 4], h24[TRAIN_ROWS * TS / 4];
  __shared__ float d1[TRAIN_ROWS * TS], d2[TRAIN_ROWS * TS], dy[TRAIN_ROWS * 2];
  float *x = (float*)x4, *h1 = (float*)h14, *h2 = (float*)h24;
  const float *W1 = params + COST_W1, *B1 = params + COST_B1, *W2 = params + COST_W2, *B2 = params + COST_B2,
              *W3 = params + COST_W3, *B3 = params + COST_B3;
  constexpr int F = COST_FEATURES, PER = (int)TRAIN_ROWS / 4;  // rows per wave
  const int tid = threadIdx.x, l = tid % 64, wave = tid / 64, lr = l % 16, lk = l / 16;
  float w1[F], w2[64], w2r[16];
#pragma unroll
  for (int i = 0; i < F; ++i) w1[i] = bf16_round(W1[i * 64 + l]);
#pragma unroll
  for (int i = 0; i < 64; ++i) w2[i] = bf16_round(W2[i * 64 + l]);
#pragma unroll
  for (int k = 0; k < 16; ++k) w2r[k] = bf16_round(W2[(wave * 16 + lr) * 64 + 4 * k + lk]);  // dh1's B operand: W2 transposed
  const float b1 = B1[l], b2 = B2[l], w3a = bf16_round(W3[l * 2]), w3b = bf16_round(W3[l * 2 + 1]);
  const float inv_b = 1.0f / (float)b;
  v4f g1[3] = {}, g2[4] = {};
  float g_vec = 0.0f, g_b3 = 0.0f;
  for (uint32_t r0 = blockIdx.x * TRAIN_ROWS; r0 < b; r0 += gridDim.x * TRAIN_ROWS) {
    const uint32_t rows = b - r0 < TRAIN_ROWS ? b - r0 : TRAIN_ROWS;
    for (uint32_t e = tid; e < TRAIN_ROWS * F; e += 256)  // rows past the batch: zeros, and no share below
      x[e] = e < rows * F ? bf16_round(feat[(size_t)r0 * F + e]) : 0.0f;
    __syncthreads();
    // two rows at a time: enough independent sums to fill the pipeline without holding all rows' inputs in registers
#pragma unroll 1
    for (int r = wave * PER; r < (wave + 1) * PER; r += 2) {
      float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
      for (int i = 0; i < F; i += 4) {
        const float4 v = x4[(r * F + i) / 4], u = x4[((r + 1) * F + i) / 4];
        s0 += w1[i] * v.x, s1 += w1[i] * u.x;
        s0 += w1[i + 1] * v.y, s1 += w1[i + 1] * u.y;
        s0 += w1[i + 2] * v.z, s1 += w1[i + 2] * u.z;
        s0 += w1[i + 3] * v.w, s1 += w1[i + 3] * u.w;
      }
      s0 += b1, s1 += b1;
      h1[r * TS + l] = (uint32_t)r < rows ? bf16_round(s0 > 0.0f ? s0 : 0.0f) : 0.0f;
      h1[(r + 1) * TS + l] = (uint32_t)r + 1 < rows ? bf16_round(s1 > 0.0f ? s1 : 0.0f) : 0.0f;
    }
    __syncthreads();
#pragma unroll 1
    for (int r = wave * PER; r < (wave + 1) * PER; r += 2) {
      float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
      for (int i = 0; i < 64; i += 4) {
        const float4 v = h14[(r * TS + i) / 4], u = h14[((r + 1) * TS + i) / 4];
        s0 += w2[i] * v.x, s1 += w2[i] * u.x;
        s0 += w2[i + 1] * v.y, s1 += w2[i + 1] * u.y;
        s0 += w2[i + 2] * v.z, s1 += w2[i + 2] * u.z;
        s0 += w2[i + 3] * v.w, s1 += w2[i + 3] * u.w;
      }
      s0 += b2, s1 += b2;
      h2[r * TS + l] = (uint32_t)r < rows ? bf16_round(s0 > 0.0f ? s0 : 0.0f) : 0.0f;
      h2[(r + 1) * TS + l] = (uint32_t)r + 1 < rows ? bf16_round(s1 > 0.0f ? s1 : 0.0f) : 0.0f;
    }
    __syncthreads();
    if (l < 2 * PER) {  // one lane per (row, output): its sum over h2 in order, then the row's losses and their gradients
      const int r = wave * PER + l / 2, k = l % 2;
      float y = 0.0f;
      for (int i = 0; i < 64; i += 4) {
        const float4 v = h24[(r * TS + i) / 4];
        y += bf16_round(W3[i * 2 + k]) * v.x;
        y += bf16_round(W3[(i + 1) * 2 + k]) * v.y;
        y += bf16_round(W3[(i + 2) * 2 + k]) * v.z;
        y += bf16_round(W3[(i + 3) * 2 + k]) * v.w;
      }
      y += B3[k];
      const bool valid = (uint32_t)r < rows;
      const float want = valid ? (k == 0 ? target[r0 + r] : contact[r0 + r]) : 0.0f;
      float part, grad;
      if (k == 0) {
        const float e = y - want;
        part = e * e;
        grad = 2.0f * e * inv_b;
      } else {
        const float sig = 1.0f / (1.0f + expf(-y));
        const float sp = y > 0.0f ? y + log1pf(expf(-y)) : log1pf(expf(y));  // softplus
        part = sp - want * y;
        grad = (sig - want) * inv_b;
      }
      const float other = __shfl_xor(part, 1);
      if (valid && k == 0) loss[r0 + r] = part + other;
      dy[r * 2 + k] = valid ? grad : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int r = wave * PER + q;
      const float g = w3a * dy[r * 2] + w3b * dy[r * 2 + 1];
      d2[r * TS + l] = h2[r * TS + l] > 0.0f ? g : 0.0f;
    }
    __syncthreads();
    v4f acc[2] = {};  // dh1 = dh2 W2^T: this wave's 16 columns of all rows
#pragma unroll
    for (int k = 0; k < 16; ++k)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(d2[(t * 16 + lr) * TS + 4 * k + lk], w2r[k], acc[t], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int at = (t * 16 + 4 * lk + i) * TS + wave * 16 + lr;
        d1[at] = h1[at] > 0.0f ? acc[t][i] : 0.0f;
      }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < (int)TRAIN_ROWS / 4; ++k) {  // the weights' shares: input activations transposed times output gradients
      const int r = 4 * k + lk;
      const float ah = h1[r * TS + wave * 16 + lr], bd = d1[r * TS + wave * 16 + lr];
#pragma unroll
      for (int j = 0; j < 4; ++j) g2[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah, d2[r * TS + j * 16 + lr], g2[j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 3; ++i) g1[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[r * F + i * 16 + lr], bd, g1[i], 0, 0, 0);
    }
    // the rest, one per thread: W3 (128), b1 (64), b2 (64); b3 beside them
    for (int r = 0; r < (int)TRAIN_ROWS; ++r)
      g_vec += tid < 128 ? h2[r * TS + tid / 2] * dy[r * 2 + tid % 2] : tid < 192 ? d1[r * TS + l] : d2[r * TS + l];
    if (tid < 2)
      for (int r = 0; r < (int)TRAIN_ROWS; ++r) g_b3 += dy[r * 2 + tid];
    __syncthreads();  // the next rows overwrite the LDS
  }
  float* out = shares + (size_t)blockIdx.x * COST_PARAMS;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) out[COST_W2 + (wave * 16 + 4 * lk + i) * 64 + j * 16 + lr] = g2[j][i];
#pragma unroll
    for (int t = 0; t < 3; ++t) out[COST_W1 + (t * 16 + 4 * lk + i) * 64 + wave * 16 + lr] = g1[t][i];
  }
  out[tid < 128 ? COST_W3 + tid : tid < 192 ? COST_B1 + l : COST_B2 + l] = g_vec;
  if (tid < 2) out[COST_B3 + tid] = g_b3;
}

// grad[p] = the groups' shares summed: 64 parameters per work-group, each by four threads over every fourth share.
__global__ void __launch_bounds__(256) k_mlp_reduce(const float* __restrict__ shares, uint32_t groups, float* __restrict__ grad) {
  __shared__ float part[4][64];
  const uint32_t l = threadIdx.x % 64, q = threadIdx.x / 64, p = blockIdx.x * 64 + l;
  float s = 0.0f;
  if (p < (uint32_t)COST_PARAMS) {
#pragma unroll 8
    for (uint32_t g = q; g < groups; g += 4) s += shares[(size_t)g * COST_PARAMS + p];
  }
  part[q][l] = s;
  __syncthreads();
  if (q == 0 && p < (uint32_t)COST_PARAMS) grad[p] = (part[0][l] + part[1][l]) + (part[2][l] + part[3][l]);
}

__global__ void __launch_bounds__(256) k_adam(float* __restrict__ params, float* __restrict__ m, float* __restrict__ v,
                                              const float* __restrict__ grad, float lr, float bc1, float bc2) {
  uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= COST_PARAMS) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  float g = grad[p];
  float mp = b1 * m[p] + (1.0f - b1) * g, vp = b2 * v[p] + (1.0f - b2) * g * g;
  m[p] = mp;
  v[p] = vp;
  params[p] -= lr * (mp / bc1) / (sqrtf(vp / bc2) + eps);
}

// ---- regrouping ----------------------------------------------------------------------------------------------------------------
// dst item i = src item perm[i] (words per item contiguous) and its inverse.
__global__ void __launch_bounds__(256) k_gather_words(const uint32_t* __restrict__ src, const uint32_t* __restrict__ perm,
                                                      uint32_t* __restrict__ dst, uint32_t n, uint32_t words) {
  size_t e = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= (size_t)n * words) return;
  size_t i = e / words, w = e % words;
  uint32_t j = perm[i];
  if (j < n) dst[e] = src[(size_t)j * words + w];  // a permutation never fails this; a bad index reads nothing
}
__global__ void __launch_bounds__(256) k_scatter_words(const uint32_t* __restrict__ src, const uint32_t* __restrict__ perm,
                                                       uint32_t* __restrict__ dst, uint32_t n, uint32_t words) {
  size_t e = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= (size_t)n * words) return;
  size_t i = e / words, w = e % words;
  uint32_t j = perm[i];
  if (j < n) dst[(size_t)j * words + w] = src[e];
}
// AoSoA-64 states: arena i of dst (n arenas) = arena perm[i] of src (n_src arenas); an index past src leaves that arena of
// dst as it was. The grid walks the words, so all arenas of one word are copied together and the source lines they share
// are read from HBM once. With XCD, word w's work-groups are all w % 8 modulo 8, on one XCD and its L2: eight words in x,
// their eights in y. (A launch takes fewer than 2^32 work-items in x, which one dimension for all words would pass at
// 1,542,657 arenas.)
template <bool XCD>
__global__ void __launch_bounds__(256) k_gather_states(const uint32_t* __restrict__ src, uint32_t n_src,
                                                       const uint32_t* __restrict__ perm, uint32_t* __restrict__ dst, uint32_t n) {
  const uint32_t w = XCD ? blockIdx.y * 8u + blockIdx.x % 8u : blockIdx.y;
  const uint32_t i = (XCD ? blockIdx.x / 8u : blockIdx.x) * 256u + threadIdx.x;
  if (i >= n || w >= (uint32_t)ARENA_WORDS) return;
  uint32_t a = perm[i];
  if (a < n_src) dst[aosoa_index(i, w)] = src[aosoa_index(a, w)];
}
// From a sample of one arena in GATHER_SPARSE on, the 32 arenas of a source line have enough readers for the one L2 to pay;
// a sparser sample of a source past the caches reads most lines for one arena, and a word's reads spread over all XCDs are
// faster (us without / with: 131,072 to 1,310 arenas 81 / 88, to 3,932 208 / 217, to 6,553 303 / 302, to 9,175 430 / 365,
// to all 2,554 / 1,855; 800,000 to 24,000 1,240 / 1,325, to 40,000 1,939 / 1,873; but 30,000 to 900 47 / 35, 65,536 to
// 655 35.0 / 33.5).
constexpr uint32_t GATHER_SPARSE = 20, GATHER_CACHED = 65536;
// The same row by row: 4-byte reads at random places, one L2 request each, bound the kernel above (65,536 arenas: 1,148 us
// without its XCD mapping, 971 us with it). Here a work-group takes one word of all of dst's arenas (up to ROW_DST): the
// source's row of that word passes through LDS in parts of ROW_PART arenas, read from HBM as whole lines, and every thread
// picks its arenas' values there, holds them in registers over the parts and writes whole lines at the end (65,536 arenas:
// 758 us; a copy of the buffer 292 us). The group has read the whole row before it writes any of it, so dst may be src.
constexpr uint32_t ROW_PART = 32768, ROW_THREADS = 1024, ROW_EACH = 64, ROW_DST = ROW_THREADS * ROW_EACH;
constexpr uint32_t ROW_LOADS = ROW_PART / (4 * ROW_THREADS);
// Rows from here on: a smaller row stays in L2 and fills few of a group's threads (16,384 arenas: rows 172 us, words 219 us;
// 8,192 arenas: words 71 us). A sample of a source is gathered word by word too, and a batch past ROW_DST, where every group
// would read several parts for each of several chunks (131,072 arenas: rows 2,473 us, words 1,897 us).
constexpr uint32_t ROW_MIN = 12288;
__global__ void __launch_bounds__(ROW_THREADS) k_gather_rows(const uint32_t* src, uint32_t n_src,
                                                             const uint32_t* __restrict__ perm, uint32_t* dst, uint32_t n) {
  extern __shared__ uint4 row4[];  // ROW_PART words
  const uint32_t* row = (const uint32_t*)row4;
  const uint32_t tid = threadIdx.x, w = blockIdx.x;
  const uint32_t quads = (n_src + AOSOA_LANES - 1) / AOSOA_LANES * (AOSOA_LANES / 4);  // of the row, padding lanes included
  uint32_t v[ROW_EACH];
  const uint32_t parts = (n_src + ROW_PART - 1) / ROW_PART;
  for (uint32_t part = 0; part < parts; ++part) {
#pragma unroll
    for (uint32_t k = 0; k < ROW_LOADS; ++k) {
      const uint32_t g = part * (ROW_PART / 4) + k * ROW_THREADS + tid;  // arenas 4 g .. 4 g + 3
      row4[k * ROW_THREADS + tid] = g < quads ? *(const uint4*)(src + aosoa_index(4 * g, w)) : uint4{0u, 0u, 0u, 0u};
    }
    __syncthreads();
    uint32_t first = tid;
    asm volatile("" : "+v"(first));  // not the same in every round to the compiler: 64 addresses kept over the rounds would spill
#pragma unroll
    for (uint32_t k = 0; k < ROW_EACH; ++k) {
      const uint32_t i = first + k * ROW_THREADS;
      if (k % 8 == 0) asm volatile("" ::: "memory");  // at most eight indices in flight: more would spill the values
      if (k * ROW_THREADS < n) {  // the same for the whole work-group
        const uint32_t at = (i < n ? perm[i] : 0u) - part * ROW_PART;
        if (at < ROW_PART) v[k] = row[at];
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (uint32_t k = 0; k < ROW_EACH; ++k) {
    const uint32_t i = k * ROW_THREADS + tid;
    if (k % 8 == 0) asm volatile("" ::: "memory");
    if (i < n && perm[i] < n_src) dst[aosoa_index(i, w)] = v[k];
  }
}

// ---- the order by predicted cost ---------------------------------------------------------------------------------------------
// A stable counting sort on the device: each arena's predicted normalised log cost falls into one of ORDER_BUCKETS
// buckets (bucket 0 the most expensive); ranks are stable within a bucket (slot order), so the order is deterministic.
// k_order_count: per-block bucket histograms, stored bucket-major (counts[b * blocks + block]). k_order_scan: each bucket's
// row scanned. k_order_place: each arena's rank = the buckets before its own (their totals scanned by every work-group) + its
// bucket's arenas in earlier blocks + its rank among the block's earlier arenas of the same bucket (wave ballots, then the
// earlier waves' counts), mapped to a slot by the mode.
__device__ inline uint32_t order_bucket(float p) {
  float q = (ORDER_HI - p) * ORDER_SCALE;
  return q != q ? ORDER_BUCKETS - 1u : q <= 0.0f ? 0u : q >= (float)(ORDER_BUCKETS - 1) ? ORDER_BUCKETS - 1u : (uint32_t)q;
}

__device__ inline uint32_t order_slot(uint32_t s, uint32_t n, int mode) {
  if (mode != ORDER_BALANCED) return s;
  // rank s is dealt round-robin over the W waves; the last wave holds r lanes, so after r rounds it is skipped
  const uint32_t W = (n + AOSOA_LANES - 1) / AOSOA_LANES, r = n - AOSOA_LANES * (W - 1);
  if (s < r * W) return (s % W) * AOSOA_LANES + s / W;
  const uint32_t t = s - r * W;  // W > 1 here: with one wave, r * W = n > s
  return (t % (W - 1)) * AOSOA_LANES + r + t / (W - 1);
}

__global__ void __launch_bounds__(ORDER_BLOCK) k_order_count(const float* __restrict__ pred, uint32_t n, uint32_t* __restrict__ counts) {
  __shared__ uint32_t h[ORDER_BUCKETS];
  const uint32_t t = threadIdx.x, blocks = gridDim.x;
  for (uint32_t b = t; b < ORDER_BUCKETS; b += ORDER_BLOCK) h[b] = 0;
  __syncthreads();
  const uint32_t a = blockIdx.x * ORDER_BLOCK + t;
  if (a < n) atomicAdd(&h[order_bucket(pred[2 * (size_t)a])], 1u);
  __syncthreads();
  for (uint32_t b = t; b < ORDER_BUCKETS; b += ORDER_BLOCK) counts[(size_t)b * blocks + blockIdx.x] = h[b];
}

// One work-group per bucket: the inclusive scan of its row of block counts, in place, ORDER_BLOCK at a time. A bucket's total
// is then its row's last word, and a block's first rank within the bucket the word before its own. (A scan of the whole
// array by one work-group took 109 us of the order's 120 at 65,536 arenas.)
__global__ void __launch_bounds__(ORDER_BLOCK) k_order_scan(uint32_t* __restrict__ counts, uint32_t blocks) {
  __shared__ uint32_t s[ORDER_BLOCK];
  const uint32_t t = threadIdx.x;
  uint32_t* v = counts + (size_t)blockIdx.x * blocks;
  uint32_t carry = 0;
  for (uint32_t lo = 0; lo < blocks; lo += ORDER_BLOCK) {
    s[t] = lo + t < blocks ? v[lo + t] : 0u;
    __syncthreads();
    for (uint32_t d = 1; d < ORDER_BLOCK; d <<= 1) {  // Hillis-Steele inclusive scan
      const uint32_t x = t >= d ? s[t - d] : 0u;
      __syncthreads();
      s[t] += x;
      __syncthreads();
    }
    if (lo + t < blocks) v[lo + t] = carry + s[t];
    carry += s[ORDER_BLOCK - 1];
    __syncthreads();
  }
}

__global__ void __launch_bounds__(ORDER_BLOCK) k_order_place(const float* __restrict__ pred, uint32_t n, const uint32_t* __restrict__ counts,
                                                             int mode, uint32_t* __restrict__ perm) {
  constexpr uint32_t WAVES = ORDER_BLOCK / AOSOA_LANES;
  __shared__ uint32_t wc[WAVES][ORDER_BUCKETS];
  const uint32_t t = threadIdx.x, lane = t % AOSOA_LANES, wave = t / AOSOA_LANES;
  __shared__ uint32_t first[ORDER_BUCKETS];  // the rank of the bucket's first arena in this block
  static_assert(ORDER_BUCKETS == ORDER_BLOCK, "one thread per bucket");
  for (uint32_t e = t; e < WAVES * ORDER_BUCKETS; e += ORDER_BLOCK) wc[e / ORDER_BUCKETS][e % ORDER_BUCKETS] = 0;
  const uint32_t* mine = counts + (size_t)t * gridDim.x;
  const uint32_t total = mine[gridDim.x - 1], earlier = blockIdx.x ? mine[blockIdx.x - 1] : 0u;
  first[t] = total;
  __syncthreads();
  for (uint32_t d = 1; d < ORDER_BUCKETS; d <<= 1) {
    const uint32_t x = t >= d ? first[t - d] : 0u;
    __syncthreads();
    first[t] += x;
    __syncthreads();
  }
  first[t] += earlier - total;
  __syncthreads();
  const uint32_t a = blockIdx.x * ORDER_BLOCK + t;
  const bool valid = a < n;
  const uint32_t b = valid ? order_bucket(pred[2 * (size_t)a]) : 0u;
  uint64_t peers = __ballot(valid);  // every lane of the wave takes part in each ballot
  for (uint32_t bit = 0; (1u << bit) < ORDER_BUCKETS; ++bit) {
    const bool on = (b >> bit) & 1u;
    const uint64_t m = __ballot(on);
    peers &= on ? m : ~m;
  }
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const uint32_t rank_in_wave = (uint32_t)__popcll(peers & below);
  if (valid && rank_in_wave == 0) wc[wave][b] = (uint32_t)__popcll(peers);  // the bucket's first lane records its count
  __syncthreads();
  if (!valid) return;
  uint32_t rank = rank_in_wave;
  for (uint32_t w = 0; w < wave; ++w) rank += wc[w][b];
  const uint32_t s = first[b] + rank;
  if (s < n) perm[order_slot(s, n, mode)] = a;  // s < n always (the counts sum to n); the check keeps a stray rank out
}

// The cost of an AoSoA block of 64 arenas for the block queue (k_run_queue): the largest predicted cost among its arenas
// (a wave lasts about as long as its slowest lane), written as a prediction row (cost, 0) so the block order is the
// arenas' counting sort applied to blocks. NaN predictions are skipped (a block of NaNs keeps NaN, which sorts last).
__global__ void __launch_bounds__(256) k_block_cost(const float* __restrict__ pred, uint32_t n, float* __restrict__ out) {
  const uint32_t b = blockIdx.x * 256 + threadIdx.x, nb = (n + AOSOA_LANES - 1) / AOSOA_LANES;
  if (b >= nb) return;
  float m = __builtin_nanf("");
  for (uint32_t a = b * AOSOA_LANES; a < n && a < (b + 1) * AOSOA_LANES; ++a) {
    const float c = pred[2 * (size_t)a];
    if (c == c && !(c <= m)) m = c;  // m NaN: the first non-NaN cost; afterwards the larger
  }
  out[2 * (size_t)b] = m;
  out[2 * (size_t)b + 1] = 0.0f;
}

// ---- launchers -----------------------------------------------------------------------------------------------------------------
static unsigned blocks_of(size_t n, unsigned b) { return (unsigned)((n + b - 1) / b > 0 ? (n + b - 1) / b : 1); }
uint64_t order_work_words(uint32_t n) { return (uint64_t)ORDER_BUCKETS * blocks_of(n, ORDER_BLOCK); }
// The fixed workspace of launch_cost_order for callers that cannot allocate: the bucket counts of up to ORDER_SCRATCH_MAX_N
// arenas (1 MiB). Each GPU holds its own copy for the life of the process; host code must not pass this name to a kernel
// (on the host it is a stand-in, not a device address) but the address order_scratch_address returns for the current
// device. The counts are overwritten whole by every order (k_order_count writes every (bucket, block) word it scans), so
// nothing needs clearing between calls; two orders in flight on one GPU at once would race on it.
static __device__ __align__(256) uint32_t scratch[ORDER_SCRATCH_WORDS];
hipError_t order_scratch_address(uint32_t** out) { return hipGetSymbolAddress((void**)out, HIP_SYMBOL(scratch)); }

hipError_t launch_cost_order(hipStream_t st, const float* pred, uint32_t n, int mode, uint32_t* work, uint32_t* perm) {
  const unsigned blocks = blocks_of(n, ORDER_BLOCK);
  k_order_count<<<blocks, ORDER_BLOCK, 0, st>>>(pred, n, work);
  k_order_scan<<<ORDER_BUCKETS, ORDER_BLOCK, 0, st>>>(work, blocks);
  k_order_place<<<blocks, ORDER_BLOCK, 0, st>>>(pred, n, work, mode, perm);
  return hipGetLastError();
}
uint64_t block_order_work_words(uint32_t n) {
  const uint32_t nb = (n + AOSOA_LANES - 1) / AOSOA_LANES;
  return 2ull * nb + order_work_words(nb);
}
hipError_t launch_block_order(hipStream_t st, const float* pred, uint32_t n, uint32_t* work, uint32_t* order) {
  const uint32_t nb = (n + AOSOA_LANES - 1) / AOSOA_LANES;
  float* block_pred = reinterpret_cast<float*>(work);
  k_block_cost<<<blocks_of(nb, 256), 256, 0, st>>>(pred, n, block_pred);
  return launch_cost_order(st, block_pred, nb, ORDER_SORTED, work + 2ull * nb, order);
}
hipError_t launch_features(hipStream_t st, const uint32_t* states, uint32_t n, float* feat) {
  k_features<<<blocks_of(n, AOSOA_LANES), AOSOA_LANES, 0, st>>>(states, n, feat);
  return hipGetLastError();
}
hipError_t launch_mlp_infer(hipStream_t st, const float* params, const float* feat, uint32_t n, float* out) {
  const uint32_t tiles = blocks_of(n, 16);
  k_mlp_infer<<<tiles < INFER_WAVES ? tiles : INFER_WAVES, 64, 0, st>>>(params, feat, n, out);
  return hipGetLastError();
}
hipError_t launch_mlp_train(hipStream_t st, const float* params, const float* feat, const float* target, const float* contact,
                            uint32_t b, float* acts, float* loss, float* grad) {
  // as many groups as have rows, the chip has CUs for, and the scratch (COST_ACT_WORDS per row) has room for shares of
  const uint32_t rows = (b + TRAIN_ROWS - 1) / TRAIN_ROWS, room = (uint32_t)((uint64_t)b * COST_ACT_WORDS / COST_PARAMS);
  uint32_t groups = rows < TRAIN_MAX_GROUPS ? rows : TRAIN_MAX_GROUPS;
  if (groups > room) groups = room;
  if (groups <= 1) {  // one group's share is the gradient
    k_mlp_train<<<1, 256, 0, st>>>(params, feat, target, contact, b, grad, loss);
    return hipGetLastError();
  }
  k_mlp_train<<<groups, 256, 0, st>>>(params, feat, target, contact, b, acts, loss);
  k_mlp_reduce<<<blocks_of(COST_PARAMS, 64), 256, 0, st>>>(acts, groups, grad);
  return hipGetLastError();
}
hipError_t launch_adam(hipStream_t st, float* params, float* m, float* v, const float* grad, float lr, float bc1, float bc2) {
  k_adam<<<blocks_of(COST_PARAMS, 256), 256, 0, st>>>(params, m, v, grad, lr, bc1, bc2);
  return hipGetLastError();
}
hipError_t launch_gather_words(hipStream_t st, const uint32_t* src, const uint32_t* perm, uint32_t* dst, uint32_t n, uint32_t words,
                               bool scatter) {
  const size_t blocks = ((size_t)n * words + 255) / 256;  // in rows of 2^20: a launch takes fewer than 2^32 work-items in x
  const unsigned x = blocks < (1u << 20) ? (unsigned)blocks : 1u << 20;
  const dim3 g(x, (unsigned)((blocks + x - 1) / x));
  if (scatter) k_scatter_words<<<g, 256, 0, st>>>(src, perm, dst, n, words);
  else k_gather_words<<<g, 256, 0, st>>>(src, perm, dst, n, words);
  return hipGetLastError();
}
hipError_t launch_gather_states(hipStream_t st, const uint32_t* src, uint32_t n_src, const uint32_t* perm, uint32_t* dst,
                                uint32_t n) {
  static_assert(ARENA_WORDS % 8 == 0, "eight words in flight, one per XCD");
  if (n_src >= ROW_MIN && n_src <= ROW_DST && n >= n_src / 2 && n <= ROW_DST)
    k_gather_rows<<<ARENA_WORDS, ROW_THREADS, ROW_PART * sizeof(uint32_t), st>>>(src, n_src, perm, dst, n);
  else if (n_src <= GATHER_CACHED || n >= n_src / GATHER_SPARSE)
    k_gather_states<true><<<dim3(blocks_of(n, 256) * 8u, ARENA_WORDS / 8), 256, 0, st>>>(src, n_src, perm, dst, n);
  else
    k_gather_states<false><<<dim3(blocks_of(n, 256), ARENA_WORDS), 256, 0, st>>>(src, n_src, perm, dst, n);
  return hipGetLastError();
}

hipError_t launch_permute_states(hipStream_t st, uint32_t* states, uint32_t* spare, const uint32_t* perm, uint32_t n) {
  if (n >= ROW_MIN && n <= ROW_DST) {
    k_gather_rows<<<ARENA_WORDS, ROW_THREADS, ROW_PART * sizeof(uint32_t), st>>>(states, n, perm, states, n);
    return hipGetLastError();
  }
  hipError_t e = launch_gather_states(st, states, n, perm, spare, n);
  return e == hipSuccess ? launch_copy_words(st, spare, states, aosoa_words(n)) : e;
}

}  // namespace dev
}  // namespace rs
