// Learned subgrid closure: a 10 -> 128 -> 128 -> 128 -> 6 MLP with GELU on
// the hidden layers (no counterpart in the reference).
//
// Inference (k_mlp_infer) runs on the matrix cores in bfloat16 with float32
// accumulation: every layer is H_out^T = W H_in^T + b with the 16 points of a
// tile as the N dimension of v_mfma_f32_16x16x16_bf16 (layer 1, K = 16) and
// v_mfma_f32_16x16x32_bf16 (layers 2-4, K = 32).  In that orientation
// the 16x16 float32 result tile (lane l: rows 4(l/16)..+3, column l%16) is
// already the B operand of the next layer for the matching 16-feature
// K-block (lane l: k = 4(l/16)..+3, column l%16), so activations never leave
// the registers between layers.  The weights, packed per 16x16 block in
// A-operand order (lane l: row l%16, k = 4(l/16)..+3), sit in LDS for the
// whole persistent workgroup.
//
// Training runs in float32 on the matrix cores: one kernel takes points
// through the network and back, a second sums the gradients and applies Adam.
#include "chan_internal.h"
#include <cmath>

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
// two 4-value operands side by side as one 8-value operand
__device__ __forceinline__ bf16x8 cat8(bf16x4 a, bf16x4 b) {
  const s16x8 r = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, r);
}
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float gelu_f(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad_f(float x) {
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * expf(-0.5f * x * x) * 0.39894228040143268f;
}

// Packed bf16 weights: layer 1 (8 out tiles x 1 k-block: 10 inputs padded to
// 16), layers 2 and 3 (8 x 8), layer 4 (1 x 8: 6 outputs padded to 16);
// 512 B per block.
#define MLP_BLK1 0
#define MLP_BLK2 8
#define MLP_BLK3 72
#define MLP_BLK4 136
#define MLP_NBLK 144

// Parameter offsets (floats) in the float32 vector W1,b1,W2,b2,W3,b3,W4,b4.
#define MLP_W1 0
#define MLP_B1 1280
#define MLP_W2 1408
#define MLP_B2 17792
#define MLP_W3 17920
#define MLP_B3 34304
#define MLP_W4 34432
#define MLP_B4 35200
#define MLP_NPARAM 35206

// Four float32 values rounded to bf16 (nearest even) by the hardware
// conversion, as one MFMA operand.
typedef __bf16 bf16x2h __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ bf16x4 to_bf16x4(float a, float b, float c, float d) {
  const bf16x2h lo = {(__bf16)a, (__bf16)b}, hi = {(__bf16)c, (__bf16)d};
  const u32x2 w = {__builtin_bit_cast(unsigned int, lo), __builtin_bit_cast(unsigned int, hi)};
  return __builtin_bit_cast(bf16x4, w);
}

// Layer 1 (K = 16, v_mfma_f32_16x16x16_bf16): block ot holds lane l's A
// operand (row l%16 of output tile ot, k = 4(l/16)..+3).  Layers 2-4
// (K = 32, v_mfma_f32_16x16x32_bf16): the two 512-byte blocks of K-block kb of
// output tile ot hold lane l's 8 values (row l%16, logical k = 8(l/16)..+7) at
// entries 2l, 2l+1.  Logical k = 8q + j stands for input feature
// 32 kb + 16 (j/4) + 4q + j%4, so that a lane's B operand is its two result
// tiles of the previous layer side by side (features 4q..4q+3 of tiles 2kb
// and 2kb+1).
__global__ void k_mlp_pack(const float* __restrict__ p, bf16x4* __restrict__ packed) {
  const int blk = blockIdx.x, l = threadIdx.x;  // 64 threads
  int wofs, nin, nout, row, f0;
  if (blk < MLP_BLK2) {
    wofs = MLP_W1; nin = 10; nout = 128;
    row = blk * 16 + (l & 15);
    f0 = 4 * (l >> 4);
  } else {
    const int b0 = blk < MLP_BLK3 ? MLP_BLK2 : (blk < MLP_BLK4 ? MLP_BLK3 : MLP_BLK4);
    wofs = blk < MLP_BLK3 ? MLP_W2 : (blk < MLP_BLK4 ? MLP_W3 : MLP_W4);
    nin = 128;
    nout = blk < MLP_BLK4 ? 128 : 6;
    const int pi = (blk - b0) / 2, hb = (blk - b0) % 2;
    const int ot = pi / 4, kb = pi % 4;
    const int L = 32 * hb + l / 2, part = l % 2;   // lane of the operand, half of its 8 values
    row = ot * 16 + (L & 15);
    f0 = 32 * kb + 16 * part + 4 * (L >> 4);
  }
  // the hidden layers' weights halved (exactly: a power of two), so that
  // their products are x/2 for the GELU (gelu_half)
  const float h = blk < MLP_BLK4 ? 0.5f : 1.0f;
  float w[4];
  for (int t = 0; t < 4; ++t) {
    const int k = f0 + t;
    w[t] = (row < nout && k < nin) ? h * p[wofs + row * nin + k] : 0.0f;
  }
  packed[blk * 64 + l] = to_bf16x4(w[0], w[1], w[2], w[3]);
}

// GELU for the bf16 inference path, without transcendental instructions or
// branches, from y = x/2: the hidden layers run with halved weights and
// biases, which halves every product, sum and rounding exactly (a power of
// two), so their accumulators hold x/2 bit for bit.  GELU(x) = x/2 + |x| e(w)
// = y + |y| 2e(w), e(w) = erf(4.5 w/sqrt 2)/2 at w = min(|y|/2.25, 1) =
// min(|x|/4.5, 1), with 2e a degree-9 polynomial in w (a least-squares
// Chebyshev fit weighted by t = 4.5 w, made for this kernel, converted to
// monomials in w and doubled).  Doubling the coefficients and halving y are
// exact, so the result is that of the same polynomial on x, rounded once at
// the last fused multiply-add.  In float32 its GELU error is <= 6.3e-5
// absolute for |x| <= 8 and below 1e-5 relative beyond (erf(4.5/sqrt 2)
// differs from 1 by 7e-6), far inside the 2^-9 relative rounding of the bf16
// result the value feeds.  11 VALU operations per value: w is one multiply
// with the clamp-to-[0,1] output modifier (|y| is a source modifier), then
// 9 fused multiply-adds and the last fused multiply-add.
__device__ __forceinline__ float gelu_half(float y) {
  const float w = __builtin_amdgcn_fmed3f(fabsf(y) * (1.0f / 2.25f), 0.0f, 1.0f);
  float e = 2.110172653e+01f;
  e = fmaf(e, w, -1.103641815e+02f);
  e = fmaf(e, w, 2.381811523e+02f);
  e = fmaf(e, w, -2.659908447e+02f);
  e = fmaf(e, w, 1.515909576e+02f);
  e = fmaf(e, w, -2.882330894e+01f);
  e = fmaf(e, w, -7.994132996e+00f);
  e = fmaf(e, w, -2.997743785e-01f);
  e = fmaf(e, w, 3.598392963e+00f);
  e = fmaf(e, w, 1.978126056e-05f);
  return fmaf(fabsf(y), e, y);
}

// GELU on a result tile of a hidden layer (x/2, its halved bias already in
// the accumulator), rounded to bf16 as the next B operand.
__device__ __forceinline__ bf16x4 act_tile(f32x4 acc) {
  return to_bf16x4(gelu_half(acc[0]), gelu_half(acc[1]), gelu_half(acc[2]), gelu_half(acc[3]));
}

// The bias of rows 4(lane/16)..+3 of output tile ot: the accumulator's
// starting value, so the products add onto it.
__device__ __forceinline__ f32x4 bias_tile(const float* __restrict__ bias, int ot, int lane) {
  const float* bb = bias + ot * 16 + 4 * (lane >> 4);
  return f32x4{bb[0], bb[1], bb[2], bb[3]};
}

#define MLP_NT 3  // point tiles of 16 per wavefront (each weight operand read from LDS serves all of them)

// Two workgroups per compute unit (their 2 x 75 KB of LDS fill it): the bound
// keeps the kernel within 256 registers, so it runs at two wavefronts per SIMD
// with its accumulators in VGPRs (175, no AGPRs, no spills), instead of 196
// VGPRs + 72 AGPRs at one wavefront per SIMD with a copy out of the AGPRs
// before every GELU (114 -> 103 us at 589 824 points).  Six-wavefront
// workgroups, three wavefronts per SIMD, are slower (120 us).  What bounds the
// kernel is its vector work: per 48 points 3666 VALU instructions (the GELU's
// 12 per value over 3 x 128 values, at 4 cycles per wavefront instruction
// without packed FP32) against 228 matrix products.
#define MLP_WAVES 4
__global__ __launch_bounds__(64 * MLP_WAVES, 2) void k_mlp_infer(const bf16x4* __restrict__ packed, const float* __restrict__ p, int n,
                                                   const float* __restrict__ x, float* __restrict__ y) {
  __shared__ __align__(16) bf16x4 W[MLP_NBLK * 64];
  const bf16x8* W8 = reinterpret_cast<const bf16x8*>(W);
  __shared__ float bias[128 * 3 + 16];
  for (int i = threadIdx.x; i < MLP_NBLK * 64; i += blockDim.x) W[i] = packed[i];
  for (int i = threadIdx.x; i < 128; i += blockDim.x) {
    bias[i] = 0.5f * p[MLP_B1 + i];  // halved with the hidden layers' weights
    bias[128 + i] = 0.5f * p[MLP_B2 + i];
    bias[256 + i] = 0.5f * p[MLP_B3 + i];
  }
  if (threadIdx.x < 16) bias[384 + threadIdx.x] = threadIdx.x < 6 ? p[MLP_B4 + threadIdx.x] : 0.0f;
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int nw = gridDim.x * (blockDim.x >> 6);
  const int q = lane >> 4, col = lane & 15;
  // features 4q..4q+3 of the points b + 16 nt + col (zero past n and past
  // feature 10), loaded without branches from clamped in-range addresses (n >= 1)
  float xv[MLP_NT][4];
  auto load_x = [&](long b) {
#pragma unroll
    for (int nt = 0; nt < MLP_NT; ++nt) {
      const long pt = b + 16 * nt + col;
      const float* xp = x + (pt < n ? pt : (long)n - 1) * 10;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int f = 4 * q + t;
        const float v = xp[f < 10 ? f : 9];
        xv[nt][t] = (pt < n && f < 10) ? v : 0.0f;
      }
    }
  };
  for (long base = ((long)blockIdx.x * (blockDim.x >> 6) + wv) * 16 * MLP_NT; base < n; base += (long)nw * 16 * MLP_NT) {
    bf16x4 h[MLP_NT][8];
    // layer 1: B operand = features 4q..4q+3 of point base + 16 nt + col
    load_x(base);
#pragma unroll
    for (int nt = 0; nt < MLP_NT; ++nt) h[nt][0] = to_bf16x4(xv[nt][0], xv[nt][1], xv[nt][2], xv[nt][3]);
    // Each layer is software-pipelined over its 8 output tiles: the matrix
    // products of tile ot+1 are issued before the GELU of tile ot, so that the
    // wavefront's vector instructions run while its products are in flight.
    f32x4 acc[2][MLP_NT];
    bf16x4 g[MLP_NT][8];
    auto layer1 = [&](int ot, f32x4 (&o)[MLP_NT]) {
      const bf16x4 a = W[(MLP_BLK1 + ot) * 64 + lane];
      const f32x4 b0 = bias_tile(bias, ot, lane);
#pragma unroll
      for (int nt = 0; nt < MLP_NT; ++nt) o[nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, h[nt][0], b0, 0, 0, 0);
    };
    layer1(0, acc[0]);
#pragma unroll
    for (int ot = 0; ot < 8; ++ot) {
      if (ot + 1 < 8) layer1(ot + 1, acc[(ot + 1) & 1]);
#pragma unroll
      for (int nt = 0; nt < MLP_NT; ++nt) g[nt][ot] = act_tile(acc[ot & 1][nt]);
      if (ot + 1 < 8) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int i = 0; i < MLP_NT; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 48, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int nt = 0; nt < MLP_NT; ++nt)
#pragma unroll
      for (int ot = 0; ot < 8; ++ot) h[nt][ot] = g[nt][ot];
    // layers 2 and 3
#pragma unroll
    for (int layer = 0; layer < 2; ++layer) {
      const int blk0 = layer == 0 ? MLP_BLK2 : MLP_BLK3;
      const float* bl = bias + 128 * (layer + 1);
      auto products = [&](int ot, f32x4 (&o)[MLP_NT]) {
        const f32x4 b0 = bias_tile(bl, ot, lane);
#pragma unroll
        for (int nt = 0; nt < MLP_NT; ++nt) o[nt] = b0;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const bf16x8 a = W8[(blk0 + (ot * 4 + kb) * 2) * 32 + lane];
#pragma unroll
          for (int nt = 0; nt < MLP_NT; ++nt)
            o[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, cat8(h[nt][2 * kb], h[nt][2 * kb + 1]), o[nt], 0, 0, 0);
        }
      };
      products(0, acc[0]);
#pragma unroll
      for (int ot = 0; ot < 8; ++ot) {
        if (ot + 1 < 8) products(ot + 1, acc[(ot + 1) & 1]);
#pragma unroll
        for (int nt = 0; nt < MLP_NT; ++nt) g[nt][ot] = act_tile(acc[ot & 1][nt]);
        if (ot + 1 < 8) {
          // the weight and bias reads, then each product followed by its
          // share of the GELU's vector instructions
          __builtin_amdgcn_sched_group_barrier(0x100, 5, 0);
#pragma unroll
          for (int i = 0; i < 4 * MLP_NT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 12, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int nt = 0; nt < MLP_NT; ++nt)
#pragma unroll
        for (int ot = 0; ot < 8; ++ot) h[nt][ot] = g[nt][ot];
    }
    // layer 4 (linear): rows 4q..4q+3 of the output tile are outputs, column = point
    const f32x4 b4 = bias_tile(bias + 384, 0, lane);
#pragma unroll
    for (int nt = 0; nt < MLP_NT; ++nt) {
      f32x4 o = b4;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W8[(MLP_BLK4 + kb * 2) * 32 + lane],
                                                    cat8(h[nt][2 * kb], h[nt][2 * kb + 1]), o, 0, 0, 0);
      const long pt = base + 16 * nt + col;
      if (pt < n)
        for (int i = 0; i < 4; ++i) {
          const int f = 4 * q + i;
          if (f < 6) y[pt * 6 + f] = o[i];
        }
    }
  }
}

// ---------------------------------------------------------------------------
// float32 training
//
// k_mlp_grad takes 16 points at a time through the whole network and back
// (forward only without GRAD), on the float32 matrix cores
// (v_mfma_f32_16x16x4_f32: full float32 products and sums).  The activations
// and GELU derivatives of the 16 points stay in LDS, the weights in registers
// (each loaded once, in the order of use; the backward pass takes a layer's
// from a copy in LDS), and a workgroup's weight gradients stay in accumulators
// over all its points; it writes them once, as one partial gradient, and
// k_mlp_update sums the partial gradients in a fixed order (and applies Adam).
//
// A mini-batch is small (1024 points: 0.2 GFLOP, 1.4 us of matrix work), so
// what counts is the number of launches and of workgroups: two launches per
// batch, one workgroup per 16 points.  One tiled product per layer and
// direction took 24 launches, its weight gradients on 4 workgroups that ran
// over all points (175 us each), and a wait for the loss: 835 us a batch of
// 1024 against 32 us now (22 us in k_mlp_grad, of which 5 us are the weights'
// first loads, and 6 us in k_mlp_update).
// ---------------------------------------------------------------------------
#define MLP_TP 16              // points per tile
#define MLP_LD 132             // LDS row of 128 features (16-byte aligned, 4 banks apart)
#define MLP_LX 20              // LDS row of 16 values
#define MLP_MAXWG 256          // partial gradients

struct MlpLds {
  float wt[128][MLP_LD];            // the weights the backward pass is at
  float x[MLP_TP][MLP_LX];          // inputs, 10 padded to 16
  float a[3][MLP_TP][MLP_LD];       // activations of the hidden layers
  float g[3][MLP_TP][MLP_LD];       // their GELU derivatives
  float d[2][MLP_TP][MLP_LD];       // dL/dz of the current layer
  float d4[MLP_TP][MLP_LX];         // dL/dy, 6 padded to 16
  float y4[8][MLP_TP][MLP_LX];      // output layer, one part per wavefront
};

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Operand layout of the 16x16x4 product: lane l = 16 g + r holds row r of A
// and column r of B at k = g; a k-block of 16 is fed as four products whose
// k = g stands for element 4g + j.  Result: column r, rows 4g .. 4g+3.
template <bool GRAD>
__global__ __launch_bounds__(512) void k_mlp_grad(const float* __restrict__ p, int n, const float* __restrict__ x,
                                                  const float* __restrict__ t, float* __restrict__ y, float sc,
                                                  float* __restrict__ part, double* __restrict__ lpart) {
  extern __shared__ float4 mlp_lds[];
  MlpLds& L = *reinterpret_cast<MlpLds*>(mlp_lds);
  const int tid = threadIdx.x, w = tid >> 6, g = (tid & 63) >> 4, r = tid & 15;
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  const int o = 16 * w + r;   // the lane's feature: wavefront w has features 16w .. 16w+15 of every layer
  // weight-gradient tiles of the wavefront: its output tile of layers 1-3 by
  // every input tile, its input tile of layer 4
  f32x4 w1 = zero, w2[8], w3[8], w4 = zero;
  float b1 = 0.0f, b2 = 0.0f, b3 = 0.0f, b4 = 0.0f;
  double loss = 0.0;
#pragma unroll
  for (int v = 0; v < 8; ++v) w2[v] = w3[v] = zero;
  // A tile's inputs and targets: threads below 256 = (point, value).  The
  // first tile's go ahead of the weights, whose loads are issued in the order
  // of their use and stay in registers over all tiles.
  const int ti = tid >> 4, tk = tid & 15;
  auto xload = [&](long base) { return (tid < 256 && tk < 10 && base + ti < n) ? x[(base + ti) * 10 + tk] : 0.0f; };
  auto tload = [&](long base) {
    return (GRAD && tid < 256 && tk < 6 && base + ti < n) ? t[(base + ti) * 6 + tk] : 0.0f;
  };
  float xv = xload((long)blockIdx.x * MLP_TP), tv = tload((long)blockIdx.x * MLP_TP);
  __builtin_amdgcn_sched_barrier(0);
  float q1[4], q4b[4];
  float4 q2[8], q3[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) q1[j] = 4 * g + j < 10 ? p[MLP_W1 + o * 10 + 4 * g + j] : 0.0f;
  const float c1 = p[MLP_B1 + o], c2 = p[MLP_B2 + o], c3 = p[MLP_B3 + o];
#pragma unroll
  for (int k = 0; k < 8; ++k) q2[k] = *reinterpret_cast<const float4*>(p + MLP_W2 + o * 128 + 16 * k + 4 * g);
#pragma unroll
  for (int k = 0; k < 8; ++k) q3[k] = *reinterpret_cast<const float4*>(p + MLP_W3 + o * 128 + 16 * k + 4 * g);
  const float4 q4 = r < 6 ? *reinterpret_cast<const float4*>(p + MLP_W4 + r * 128 + 16 * w + 4 * g)
                          : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float c4 = tk < 6 ? p[MLP_B4 + tk] : 0.0f;
  if (GRAD) {
#pragma unroll
    for (int j = 0; j < 4; ++j) q4b[j] = 4 * g + j < 6 ? p[MLP_W4 + (4 * g + j) * 128 + o] : 0.0f;
  }
  // hidden layer of 128 inputs `in` with weights q and bias b into (a, gelu')
  auto hidden = [&](const float (*in)[MLP_LD], const float4 (&q)[8], float b, float (*oa)[MLP_LD],
                    float (*og)[MLP_LD]) {
    f32x4 c = zero;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float4 a = *reinterpret_cast<const float4*>(&in[r][16 * k + 4 * g]);
      c = mfma_f32(a.x, q[k].x, c); c = mfma_f32(a.y, q[k].y, c);
      c = mfma_f32(a.z, q[k].z, c); c = mfma_f32(a.w, q[k].w, c);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float z = c[i] + b;
      oa[4 * g + i][o] = gelu_f(z);
      if (GRAD) og[4 * g + i][o] = gelu_grad_f(z);
    }
  };
  // weights (rows o, as the forward pass holds them) to LDS for the backward
  // pass, which takes them by columns
  auto stage = [&](const float4 (&q)[8]) {
#pragma unroll
    for (int k = 0; k < 8; ++k) *reinterpret_cast<float4*>(&L.wt[o][16 * k + 4 * g]) = q[k];
  };
  // dL/dz of the layer below: (D W) gelu', W in L.wt
  auto back = [&](const float (*D)[MLP_LD], const float (*gp)[MLP_LD], float (*out)[MLP_LD]) {
    f32x4 c = zero;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float4 a = *reinterpret_cast<const float4*>(&D[r][16 * k + 4 * g]);
      const float(*W)[MLP_LD] = L.wt + 16 * k + 4 * g;
      c = mfma_f32(a.x, W[0][o], c); c = mfma_f32(a.y, W[1][o], c);
      c = mfma_f32(a.z, W[2][o], c); c = mfma_f32(a.w, W[3][o], c);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) out[4 * g + i][o] = c[i] * gp[4 * g + i][o];
  };
  // acc[v] += D^T A over the 16 points, the wavefront's output tile by input tile v
  auto wgrad = [&](const float (*D)[MLP_LD], const float (*A)[MLP_LD], f32x4 (&acc)[8]) {
    float dv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) dv[j] = D[4 * g + j][o];
#pragma unroll
    for (int v = 0; v < 8; ++v)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[v] = mfma_f32(dv[j], A[4 * g + j][16 * v + r], acc[v]);
  };
  auto colsum = [&](const float (*D)[MLP_LD]) {
    float v = 0.0f;
#pragma unroll
    for (int i = 0; i < MLP_TP; ++i) v += D[i][tid & 127];
    return v;
  };

  const int ntile = (n + MLP_TP - 1) / MLP_TP;
  for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const long base = (long)tile * MLP_TP;
    const float target = tv;
    if (tid < 256) L.x[ti][tk] = xv;
    __syncthreads();
    xv = xload(base + (long)gridDim.x * MLP_TP);
    tv = tload(base + (long)gridDim.x * MLP_TP);
    {  // layer 1, K = 10 padded to 16
      const float4 a = *reinterpret_cast<const float4*>(&L.x[r][4 * g]);
      const float av[4] = {a.x, a.y, a.z, a.w};
      f32x4 c = zero;
#pragma unroll
      for (int j = 0; j < 4; ++j) c = mfma_f32(av[j], q1[j], c);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float z = c[i] + c1;
        L.a[0][4 * g + i][o] = gelu_f(z);
        if (GRAD) L.g[0][4 * g + i][o] = gelu_grad_f(z);
      }
    }
    __syncthreads();
    hidden(L.a[0], q2, c2, L.a[1], L.g[1]);
    __syncthreads();
    hidden(L.a[1], q3, c3, L.a[2], L.g[2]);
    if (GRAD) stage(q3);
    __syncthreads();
    {  // output layer, 6 padded to 16: wavefront w sums its own features
      f32x4 c = zero;
      const float4 a = *reinterpret_cast<const float4*>(&L.a[2][r][16 * w + 4 * g]);
      c = mfma_f32(a.x, q4.x, c); c = mfma_f32(a.y, q4.y, c);
      c = mfma_f32(a.z, q4.z, c); c = mfma_f32(a.w, q4.w, c);
#pragma unroll
      for (int i = 0; i < 4; ++i) L.y4[w][4 * g + i][r] = c[i];
    }
    __syncthreads();
    if (tid < 256) {
      const int i = ti, k = tk;
      const bool ok = k < 6 && base + i < n;
      float d = 0.0f;
      if (ok) {
        const float v = ((L.y4[0][i][k] + L.y4[1][i][k]) + (L.y4[2][i][k] + L.y4[3][i][k])) +
                        ((L.y4[4][i][k] + L.y4[5][i][k]) + (L.y4[6][i][k] + L.y4[7][i][k])) + c4;
        const long at = (base + i) * 6 + k;
        if (GRAD) {
          const float e = v - target;
          d = sc * e;
          loss += (double)e * (double)e;
        } else {
          y[at] = v;
        }
      }
      if (GRAD) L.d4[i][k] = d;
    }
    if (GRAD) {
      __syncthreads();
      {  // layer 4: its weight gradient, and dL/dz of layer 3
        const float4 a = *reinterpret_cast<const float4*>(&L.d4[r][4 * g]);
        const float av[4] = {a.x, a.y, a.z, a.w};
        f32x4 c = zero;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          w4 = mfma_f32(L.d4[4 * g + j][r], L.a[2][4 * g + j][o], w4);
          c = mfma_f32(av[j], q4b[j], c);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) L.d[0][4 * g + i][o] = c[i] * L.g[2][4 * g + i][o];
        if (tid < 6) {
#pragma unroll
          for (int i = 0; i < MLP_TP; ++i) b4 += L.d4[i][tid];
        }
      }
      __syncthreads();
      wgrad(L.d[0], L.a[1], w3);
      b3 += colsum(L.d[0]);
      back(L.d[0], L.g[1], L.d[1]);
      __syncthreads();
      stage(q2);
      wgrad(L.d[1], L.a[0], w2);
      b2 += colsum(L.d[1]);
      __syncthreads();
      back(L.d[1], L.g[0], L.d[0]);
      __syncthreads();
#pragma unroll
      for (int j = 0; j < 4; ++j) w1 = mfma_f32(L.d[0][4 * g + j][o], L.x[4 * g + j][r], w1);
      b1 += colsum(L.d[0]);
    }
    __syncthreads();   // the tile's LDS is free
  }
  if (!GRAD) return;
  float* q = part + (long)blockIdx.x * MLP_NPARAM;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 16 * w + 4 * g + i;
    if (r < 10) q[MLP_W1 + row * 10 + r] = w1[i];
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      q[MLP_W2 + row * 128 + 16 * v + r] = w2[v][i];
      q[MLP_W3 + row * 128 + 16 * v + r] = w3[v][i];
    }
    if (4 * g + i < 6) q[MLP_W4 + (4 * g + i) * 128 + o] = w4[i];
  }
  if (tid < 128) {
    q[MLP_B1 + tid] = b1;
    q[MLP_B2 + tid] = b2;
    q[MLP_B3 + tid] = b3;
  }
  if (tid < 6) q[MLP_B4 + tid] = b4;
  __shared__ double red[8];
  for (int s = 32; s > 0; s >>= 1) loss += __shfl_xor(loss, s, 64);
  if ((tid & 63) == 0) red[w] = loss;
  __syncthreads();
  if (tid == 0) lpart[blockIdx.x] = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
}

// g = sum of the nw partial gradients (in double, in order), loss = sum of the
// nw partial losses; with ADAM one step t >= 1 of Adam (Kingma & Ba 2015,
// Algorithm 1) on the parameters.
// A workgroup has 64 parameters; wavefront w sums every fourth partial.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_mlp_update(int nw, const float* __restrict__ part,
                                                    const double* __restrict__ lpart, float* __restrict__ g,
                                                    double* __restrict__ loss, float* __restrict__ p,
                                                    float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                                    float b2, float eps, float c1, float c2) {
  __shared__ double red[4][64];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + l, ic = min(i, MLP_NPARAM - 1);
  const bool own = w == 0 && i < MLP_NPARAM;
  const float m0 = ADAM && own ? m[i] : 0.0f, v0 = ADAM && own ? v[i] : 0.0f, p0 = ADAM && own ? p[i] : 0.0f;
  double s = 0.0;
#pragma unroll 16
  for (int k = w; k < nw; k += 4) s += (double)part[(long)k * MLP_NPARAM + ic];
  red[w][l] = s;
  if (blockIdx.x == 0 && threadIdx.x == 64) {
    double e = 0.0;
    for (int k = 0; k < nw; ++k) e += lpart[k];
    *loss = e;
  }
  __syncthreads();
  if (!own) return;
  const float gi = (float)((red[0][l] + red[1][l]) + (red[2][l] + red[3][l]));
  g[i] = gi;
  if (ADAM) {
    const float mi = b1 * m0 + (1.0f - b1) * gi;
    const float vi = b2 * v0 + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] = p0 - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct chan_mlp {
  hipStream_t stream = nullptr;
  float* d_p = nullptr;      // float32 parameters
  float* d_g = nullptr;      // gradients
  float* d_m = nullptr;      // Adam moments
  float* d_v = nullptr;
  bf16x4* d_packed = nullptr;
  bool packed_ok = false;
  int adam_t = 0;
  // work buffers (capacity in points)
  long cap = 0;
  float *d_x = nullptr, *d_y = nullptr, *d_t = nullptr;
  // partial gradients and losses of the training workgroups, and the loss
  float* d_part = nullptr;
  double* d_lpart = nullptr;
  std::string last_error;
};

namespace {

void mchk(hipError_t e, const char* what) {
  if (e != hipSuccess) throw chan_error(std::string(what) + ": " + hipGetErrorString(e));
}

template <class T>
void mfree(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

void ensure_cap(chan_mlp* m, long n) {
  if (n <= m->cap) return;
  mfree(m->d_x); mfree(m->d_y); mfree(m->d_t);
  m->cap = 0;
  mchk(hipMalloc(&m->d_x, sizeof(float) * 10 * n), "hipMalloc");
  mchk(hipMalloc(&m->d_y, sizeof(float) * 6 * n), "hipMalloc");
  mchk(hipMalloc(&m->d_t, sizeof(float) * 6 * n), "hipMalloc");
  m->cap = n;
}

void ensure_partials(chan_mlp* m) {
  if (!m->d_part) mchk(hipMalloc(&m->d_part, sizeof(float) * (size_t)MLP_NPARAM * MLP_MAXWG), "hipMalloc");
  if (!m->d_lpart) mchk(hipMalloc(&m->d_lpart, sizeof(double) * (MLP_MAXWG + 1)), "hipMalloc");
}

int tile_blocks(long n) { return (int)std::min<long>(MLP_MAXWG, (n + MLP_TP - 1) / MLP_TP); }

// Gradient of the mean squared error of n points (inputs x, targets t on the
// device) into d_g and its sum of squares into d_lpart[MLP_MAXWG]; with
// adam_t > 0 that step of Adam on the parameters.  Queued, not waited for.
void gradient32(chan_mlp* m, int n, const float* x, const float* t, int adam_t, float lr) {
  const int nw = tile_blocks(n);
  hipLaunchKernelGGL((k_mlp_grad<true>), dim3(nw), dim3(512), sizeof(MlpLds), m->stream, m->d_p, n, x, t, nullptr,
                     2.0f / (float)(6L * n), m->d_part, m->d_lpart);
  LAUNCH_CHECK("k_mlp_grad");
  const dim3 grid((MLP_NPARAM + 63) / 64);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  if (adam_t > 0) {
    const float c1 = 1.0f - std::pow(b1, (float)adam_t), c2 = 1.0f - std::pow(b2, (float)adam_t);
    hipLaunchKernelGGL((k_mlp_update<true>), grid, dim3(256), 0, m->stream, nw, m->d_part, m->d_lpart, m->d_g,
                       m->d_lpart + MLP_MAXWG, m->d_p, m->d_m, m->d_v, lr, b1, b2, eps, c1, c2);
  } else {
    hipLaunchKernelGGL((k_mlp_update<false>), grid, dim3(256), 0, m->stream, nw, m->d_part, m->d_lpart, m->d_g,
                       m->d_lpart + MLP_MAXWG, m->d_p, m->d_m, m->d_v, lr, b1, b2, eps, 1.0f, 1.0f);
  }
  LAUNCH_CHECK("k_mlp_update");
}

// the loss of the last gradient32 of n points (waits for it)
double last_loss(chan_mlp* m, int n) {
  double s = 0.0;
  mchk(hipMemcpyAsync(&s, m->d_lpart + MLP_MAXWG, sizeof(double), hipMemcpyDeviceToHost, m->stream), "copy");
  mchk(hipStreamSynchronize(m->stream), "sync");
  return s / (double)(6L * n);
}

void pack(chan_mlp* m) {
  if (m->packed_ok) return;
  hipLaunchKernelGGL(k_mlp_pack, dim3(MLP_NBLK), dim3(64), 0, m->stream, m->d_p, m->d_packed);
  LAUNCH_CHECK("k_mlp_pack");
  m->packed_ok = true;
}

template <class F>
int mguard(chan_mlp* m, F&& f) {
  if (!m) return 1;
  try {
    f();
    return 0;
  } catch (const chan_error& e) {
    m->last_error = e.msg;
  } catch (const std::exception& e) {
    m->last_error = e.what();
  }
  return 1;
}

}  // namespace

// Workgroups of the persistent inference kernel: as many as fit on the device
// at once (its 75 KB of LDS weights allow two per CU), so that every
// workgroup loads the weights once.
static int mlp_blocks(long n) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
    cus = 256;
  const long tiles = (n + 16 * MLP_NT - 1) / (16 * MLP_NT);
  return (int)std::max<long>(1, std::min<long>(2L * cus, (tiles + MLP_WAVES - 1) / MLP_WAVES));
}

void mlp_prepare_device(chan_mlp* m) {
  pack(m);
  mchk(hipStreamSynchronize(m->stream), "sync");
}

// inference of n points already on the device, on the caller's stream
// (weights changed since the last packing are packed first, synchronised)
void mlp_infer_device(chan_mlp* m, long n, const float* x, float* y, hipStream_t s) {
  if (!m->packed_ok) mlp_prepare_device(m);
  if (n <= 0) return;
  if (n > 0x7fffffffL) throw chan_error("too many points for one inference");
  hipLaunchKernelGGL(k_mlp_infer, dim3(mlp_blocks(n)), dim3(64 * MLP_WAVES), 0, s, m->d_packed, m->d_p, (int)n, x, y);
  LAUNCH_CHECK("k_mlp_infer");
}

extern "C" {

int chan_mlp_create(chan_mlp** out) {
  if (!out) return 1;
  *out = nullptr;
  chan_mlp* m = new chan_mlp();
  if (mguard(m, [&] {
        mchk(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking), "stream");
        mchk(hipMalloc(&m->d_p, sizeof(float) * MLP_NPARAM), "hipMalloc");
        mchk(hipMalloc(&m->d_g, sizeof(float) * MLP_NPARAM), "hipMalloc");
        mchk(hipMalloc(&m->d_m, sizeof(float) * MLP_NPARAM), "hipMalloc");
        mchk(hipMalloc(&m->d_v, sizeof(float) * MLP_NPARAM), "hipMalloc");
        mchk(hipMalloc(&m->d_packed, sizeof(bf16x4) * MLP_NBLK * 64), "hipMalloc");
        mchk(hipMemset(m->d_p, 0, sizeof(float) * MLP_NPARAM), "memset");
        mchk(hipMemset(m->d_m, 0, sizeof(float) * MLP_NPARAM), "memset");
        mchk(hipMemset(m->d_v, 0, sizeof(float) * MLP_NPARAM), "memset");
      })) {
    chan_mlp_destroy(m);
    return 1;
  }
  *out = m;
  return 0;
}

int chan_mlp_destroy(chan_mlp* m) {
  if (!m) return 0;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  mfree(m->d_p); mfree(m->d_g); mfree(m->d_m); mfree(m->d_v); mfree(m->d_packed);
  mfree(m->d_x); mfree(m->d_y); mfree(m->d_t); mfree(m->d_part); mfree(m->d_lpart);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return 0;
}

const char* chan_mlp_last_error(const chan_mlp* m) { return m ? m->last_error.c_str() : "null network"; }

int chan_mlp_num_params(void) { return MLP_NPARAM; }

int chan_mlp_set_params(chan_mlp* m, const float* p) {
  return mguard(m, [&] {
    if (!p) throw chan_error("null argument");
    mchk(hipMemcpyAsync(m->d_p, p, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice, m->stream), "copy");
    mchk(hipMemsetAsync(m->d_m, 0, sizeof(float) * MLP_NPARAM, m->stream), "memset");
    mchk(hipMemsetAsync(m->d_v, 0, sizeof(float) * MLP_NPARAM, m->stream), "memset");
    mchk(hipStreamSynchronize(m->stream), "sync");
    m->adam_t = 0;
    m->packed_ok = false;
  });
}

int chan_mlp_get_params(chan_mlp* m, float* p) {
  return mguard(m, [&] {
    if (!p) throw chan_error("null argument");
    mchk(hipMemcpyAsync(p, m->d_p, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost, m->stream), "copy");
    mchk(hipStreamSynchronize(m->stream), "sync");
  });
}

int chan_mlp_infer(chan_mlp* m, int n, const float* x, float* y) {
  return mguard(m, [&] {
    if (n < 0 || (n && (!x || !y))) throw chan_error("invalid arguments");
    if (n == 0) return;
    ensure_cap(m, n);
    pack(m);
    mchk(hipMemcpyAsync(m->d_x, x, sizeof(float) * 10 * n, hipMemcpyHostToDevice, m->stream), "copy");
    hipLaunchKernelGGL(k_mlp_infer, dim3(mlp_blocks(n)), dim3(64 * MLP_WAVES), 0, m->stream, m->d_packed, m->d_p, n, m->d_x,
                       m->d_y);
    LAUNCH_CHECK("k_mlp_infer");
    mchk(hipMemcpyAsync(y, m->d_y, sizeof(float) * 6 * n, hipMemcpyDeviceToHost, m->stream), "copy");
    mchk(hipStreamSynchronize(m->stream), "sync");
  });
}

int chan_mlp_forward_fp32(chan_mlp* m, int n, const float* x, float* y) {
  return mguard(m, [&] {
    if (n < 1 || !x || !y) throw chan_error("invalid arguments");
    ensure_cap(m, n);
    mchk(hipMemcpyAsync(m->d_x, x, sizeof(float) * 10 * n, hipMemcpyHostToDevice, m->stream), "copy");
    hipLaunchKernelGGL((k_mlp_grad<false>), dim3(tile_blocks(n)), dim3(512), sizeof(MlpLds), m->stream, m->d_p, n,
                       m->d_x, nullptr, m->d_y, 0.0f, nullptr, nullptr);
    LAUNCH_CHECK("k_mlp_grad");
    mchk(hipMemcpyAsync(y, m->d_y, sizeof(float) * 6 * n, hipMemcpyDeviceToHost, m->stream), "copy");
    mchk(hipStreamSynchronize(m->stream), "sync");
  });
}

int chan_mlp_gradient(chan_mlp* m, int n, const float* x, const float* t, float* grad, double* loss) {
  return mguard(m, [&] {
    if (n < 1 || !x || !t) throw chan_error("invalid arguments");
    ensure_cap(m, n);
    ensure_partials(m);
    mchk(hipMemcpyAsync(m->d_x, x, sizeof(float) * 10 * n, hipMemcpyHostToDevice, m->stream), "copy");
    mchk(hipMemcpyAsync(m->d_t, t, sizeof(float) * 6 * n, hipMemcpyHostToDevice, m->stream), "copy");
    gradient32(m, n, m->d_x, m->d_t, 0, 0.0f);
    if (grad)
      mchk(hipMemcpyAsync(grad, m->d_g, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost, m->stream), "copy");
    const double l = last_loss(m, n);
    if (loss) *loss = l;
  });
}

// Mini-batch Adam on n points (in the given order, batches of `batch`, the
// incomplete last batch dropped) for `epochs` passes; loss_out receives the
// loss of the last batch.
int chan_mlp_train(chan_mlp* m, int n, const float* x, const float* t, int epochs, int batch, double lr,
                   double* loss_out) {
  return mguard(m, [&] {
    if (n < 1 || !x || !t || epochs < 1 || batch < 1 || batch > n) throw chan_error("invalid arguments");
    ensure_cap(m, n);
    ensure_partials(m);
    mchk(hipMemcpyAsync(m->d_x, x, sizeof(float) * 10 * n, hipMemcpyHostToDevice, m->stream), "copy");
    mchk(hipMemcpyAsync(m->d_t, t, sizeof(float) * 6 * n, hipMemcpyHostToDevice, m->stream), "copy");
    m->packed_ok = false;
    const int nb = n / batch;
    for (int e = 0; e < epochs; ++e)
      for (int bi = 0; bi < nb; ++bi) {
        m->adam_t += 1;
        gradient32(m, batch, m->d_x + (long)bi * batch * 10, m->d_t + (long)bi * batch * 6, m->adam_t, (float)lr);
      }
    const double l = last_loss(m, batch);
    if (loss_out) *loss_out = l;
  });
}

}  // extern "C"
