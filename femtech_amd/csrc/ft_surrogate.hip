// ft_surrogate.hip -- the constitutive surrogate network on the matrix cores
// (no counterpart in the reference).
//
//   k_mlp_infer  all five layers of a 32-sample slab per wavefront in one
//                launch: BF16 operands on v_mfma_f32_32x32x16_bf16, FP32
//                accumulation, bias and SiLU on the accumulators, and the
//                layer-to-layer hand-over kept in registers (the weights of
//                layers 1-4 are stored with their input columns permuted to
//                the accumulator layout, so one layer's output tile is the
//                next layer's B operand as it stands).
//   k_mlp_train  forward, loss and backward of 32 samples per block in one
//                launch, leaving every layer's activations and dZ.
//   k_mlp_grad   weight gradients per 256 samples, bias gradients.
//   k_mlp_update gradients summed, Adam, BF16 weight copies.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/femtech_amd.h"
#include "ft_mlp.h"

extern "C" void ft_internal_set_error(const char *msg);

namespace ft {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

int mfail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
int mfail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  ft_internal_set_error(buf);
  // reported here, so not by the check behind a later launch
  if (code == FT_ERR_HIP || code == FT_ERR_ALLOC) (void)hipGetLastError();
  return code;
}

#define MCHK(call)                                                                      \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess)                                                               \
      return mfail(FT_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                   __FILE__, __LINE__);                                                 \
  } while (0)

// Flat FP32 parameter vector: per layer W_l [out][in] row-major, then b_l.
__host__ __device__ constexpr int layer_in(int l) { return l == 0 ? kMlpIn : kMlpHid; }
__host__ __device__ constexpr int layer_out(int l) { return l == kMlpLayers - 1 ? kMlpOut : kMlpHid; }
__host__ __device__ constexpr int w_off(int l) {
  return l == 0 ? 0 : w_off(l - 1) + layer_out(l - 1) * (layer_in(l - 1) + 1);
}
__host__ __device__ constexpr int b_off(int l) { return w_off(l) + layer_out(l) * layer_in(l); }
constexpr int kParams = w_off(kMlpLayers);
static_assert(kParams == 52744, "parameter layout");

// Inference copy (BF16): layer 0 [128][16] as is; layers 1-3 [128][128] and
// layer 4 [32][128] (rows past 8 zero) with permuted input columns.
__host__ __device__ constexpr int wi_off(int l) { return l == 0 ? 0 : kMlpHid * kMlpIn + (l - 1) * kMlpHid * kMlpHid; }
constexpr int kWi = wi_off(kMlpLayers - 1) + 32 * kMlpHid;

// Accumulator layout of the 32x32 product (lane l, h = l / 32): element
// 4 j + r of the 16 holds row 8 j + 4 h + r, column l % 32.  The B operand of
// a 16-deep step takes 8 values per lane at depth 8 h + i.  Handing the 16
// accumulators of output tile t over as two B operands (values 0-7 and
// 8-15) feeds depth position p of step s = 2 t + q with the feature below;
// the next layer's weights are stored with their columns in this order.
__host__ __device__ inline int chain_feature(int kpos) {
  const int s = kpos >> 4, p = kpos & 15, h = p >> 3, pp = p & 7;
  return 32 * (s >> 1) + 16 * (s & 1) + 8 * (pp >> 2) + 4 * h + (pp & 3);
}

// Training copies (BF16): weights as they stand (Pb, the parameter layout) and
// transposed, Wt: layers 1-3 [in][out], layer 4 [in][16] (outputs past 8 zero).
__host__ __device__ constexpr int wt_off(int l) { return (l - 1) * kMlpHid * kMlpHid; }
constexpr int kWt = wt_off(4) + kMlpHid * 16;

// Layer of a parameter and its place there.
__device__ inline int layer_of(int i) {
  int l = 0;
  while (l < kMlpLayers - 1 && i >= w_off(l + 1)) ++l;
  return l;
}

// The BF16 copies of parameter i (value v).
__device__ inline void store_copies(int i, float v, __bf16 *Pb, __bf16 *Wt) {
  Pb[i] = (__bf16)v;
  const int l = layer_of(i);
  if (l == 0 || i >= b_off(l)) return;
  const int row = (i - w_off(l)) / kMlpHid, col = (i - w_off(l)) % kMlpHid;
  Wt[wt_off(l) + col * (l == kMlpLayers - 1 ? 16 : kMlpHid) + row] = (__bf16)v;
}

__global__ void k_refresh(const float *P, __bf16 *Pb, __bf16 *Wi, __bf16 *Wt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kParams) store_copies(i, P[i], Pb, Wt);
  if (i < kMlpHid * 8) Wt[wt_off(4) + (i / 8) * 16 + 8 + i % 8] = (__bf16)0.0f;
  if (i < kWi) {
    int l, row, col;
    if (i < wi_off(1)) {
      l = 0;
      row = i / kMlpIn;
      col = i % kMlpIn;
    } else {
      l = 1 + (i - wi_off(1)) / (kMlpHid * kMlpHid);
      const int r = i - wi_off(l);
      row = r / kMlpHid;
      col = chain_feature(r % kMlpHid);
    }
    float v = 0.0f;
    if (row < layer_out(l)) v = P[w_off(l) + row * layer_in(l) + col];
    Wi[i] = (__bf16)v;
  }
}

// SiLU for inference: hardware exponential and reciprocal (1 ulp), the
// BF16 rounding of the result dominates the error.
__device__ inline float silu_fast(float z) { return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

// Accumulators of the four output tiles of a layer started at the bias (the
// lane's rows 8 j + 4 h + r hold 4 consecutive biases: one 16-byte read).
__device__ inline void bias_init(f32x16 (&acc)[4], const float *b, int h) {
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 v = *reinterpret_cast<const float4 *>(b + 32 * t + 8 * j + 4 * h);
      acc[t][4 * j] = v.x;
      acc[t][4 * j + 1] = v.y;
      acc[t][4 * j + 2] = v.z;
      acc[t][4 * j + 3] = v.w;
    }
}

// SiLU on the four output tiles of one 32-sample column tile (bias already
// in the accumulators), then the hand-over to the next layer's eight B
// operands.
__device__ inline void act_chain(const f32x16 (&acc)[4], bf16x8 (&B)[8]) {
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) B[2 * t + (j >> 1)][(j & 1) * 4 + r] = (__bf16)silu_fast(acc[t][4 * j + r]);
}

// y[n][8] = network(x[n][16]).  Persistent blocks of 8 wavefronts: the
// block stages all weights (BF16, 117 KB) and biases in LDS once, then each
// wavefront walks 32-sample slabs, the A operands coming from LDS.
// NT column tiles of 32 samples per wavefront, THREADS per block: one tile at
// two wavefronts per SIMD, so that the SiLU evaluations of one overlap the
// matrix products of the other.  Weight rows in LDS are padded by 16 bytes:
// the 8 rows of one phase of a 16-byte read then fall on different banks
// (unpadded, 256-byte rows put them all on the same four, and each fragment
// read took eight turns).  1.40M samples: 381 us unpadded with two tiles at one
// wavefront per SIMD, 321 us padded, 244 us with one tile at two (0.60 PFLOP/s;
// two tiles at two, with spills: 15 us slower).
constexpr int kInferTiles = 1;
constexpr int kInferThreads = 512;
constexpr int kPadIn = kMlpIn + 8, kPadW = kMlpHid + 8;
constexpr int kWiLds = kMlpHid * kPadIn + (3 * kMlpHid + 32) * kPadW;

template <int NT, int THREADS>
__global__ __launch_bounds__(THREADS) void k_mlp_infer(const __bf16 *x, long n, const __bf16 *wi, const float *P,
                                                       float *y) {
  __shared__ __attribute__((aligned(16))) __bf16 sw[kWiLds];
  __shared__ float sb[kMlpLayers * kMlpHid];
  for (int i = threadIdx.x; i < wi_off(1) / 8; i += blockDim.x)
    *reinterpret_cast<bf16x8 *>(sw + i / 2 * kPadIn + i % 2 * 8) = reinterpret_cast<const bf16x8 *>(wi)[i];
  for (int i = threadIdx.x; i < (kWi - wi_off(1)) / 8; i += blockDim.x)
    *reinterpret_cast<bf16x8 *>(sw + kMlpHid * kPadIn + i / 16 * kPadW + i % 16 * 8) =
        reinterpret_cast<const bf16x8 *>(wi + wi_off(1))[i];
  for (int i = threadIdx.x; i < kMlpLayers * kMlpHid; i += blockDim.x) {
    const int l = i / kMlpHid, r = i % kMlpHid;
    sb[i] = r < layer_out(l) ? P[b_off(l) + r] : 0.0f;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, h = lane >> 5, c32 = lane & 31;
  constexpr int waves = THREADS / 64, slab_n = 32 * NT;
  const long slabs = (n + slab_n - 1) / slab_n;
  const bf16x8 zero8 = {};
  const f32x16 zero16 = {};
  for (long slab = (long)blockIdx.x * waves + (threadIdx.x >> 6); slab < slabs; slab += (long)gridDim.x * waves) {
    const long base = slab * slab_n;
    bf16x8 B[NT][8];
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      const long s = base + 32 * c + c32;
      B[c][0] = s < n ? *reinterpret_cast<const bf16x8 *>(x + s * kMlpIn + 8 * h) : zero8;
    }
    f32x16 acc[NT][4];
    bias_init(acc[0], sb, h);
#pragma unroll
    for (int c = 1; c < NT; ++c)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[c][t] = acc[0][t];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bf16x8 a = *reinterpret_cast<const bf16x8 *>(sw + (32 * t + c32) * kPadIn + 8 * h);
#pragma unroll
      for (int c = 0; c < NT; ++c) acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, B[c][0], acc[c][t], 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < NT; ++c) act_chain(acc[c], B[c]);
#pragma unroll 1
    for (int l = 1; l < kMlpLayers - 1; ++l) {
      const __bf16 *w = sw + kMlpHid * kPadIn + (l - 1) * kMlpHid * kPadW;
      bias_init(acc[0], sb + l * kMlpHid, h);
#pragma unroll
      for (int c = 1; c < NT; ++c)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[c][t] = acc[0][t];
      // depth-step outer, tiles inner: independent accumulation chains in
      // flight behind each other on the matrix core
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const bf16x8 a = *reinterpret_cast<const bf16x8 *>(w + (32 * t + c32) * kPadW + 16 * s + 8 * h);
#pragma unroll
          for (int c = 0; c < NT; ++c)
            acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, B[c][s], acc[c][t], 0, 0, 0);
        }
#pragma unroll
      for (int c = 0; c < NT; ++c) act_chain(acc[c], B[c]);
    }
    const __bf16 *w = sw + kMlpHid * kPadIn + (kMlpLayers - 2) * kMlpHid * kPadW;
    f32x16 o[NT];
#pragma unroll
    for (int c = 0; c < NT; ++c) o[c] = zero16;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const bf16x8 a = *reinterpret_cast<const bf16x8 *>(w + c32 * kPadW + 16 * s + 8 * h);
#pragma unroll
      for (int c = 0; c < NT; ++c) o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, B[c][s], o[c], 0, 0, 0);
    }
    const float *b4 = sb + (kMlpLayers - 1) * kMlpHid;
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      const long s = base + 32 * c + c32;
      if (s < n) {  // rows 4 h + r of the first row group are outputs 4 h + r
        float4 v;
        v.x = o[c][0] + b4[4 * h];
        v.y = o[c][1] + b4[4 * h + 1];
        v.z = o[c][2] + b4[4 * h + 2];
        v.w = o[c][3] + b4[4 * h + 3];
        *reinterpret_cast<float4 *>(y + s * kMlpOut + 4 * h) = v;
      }
    }
  }
}

__device__ inline uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// ---------------------------------------------------------------------------
// Training
// ---------------------------------------------------------------------------
// k_mlp_train: one block takes 32 samples through forward, loss and backward.
// Its 4 wavefronts each own 32 of a layer's 128 rows: weights as A operands
// straight from the cache into registers, a layer ahead, against the block's
// samples as B operands.  A tile's accumulators (lane half h: rows 8 j + 4 h +
// r) become B operands (depth 8 h + i) by one v_permlane32_swap per packed
// pair and go to the other wavefronts through LDS, two buffers, one barrier per
// layer; SiLU' stays in registers.  For the weight gradients, whose depth is
// the samples, activations and dZ go to memory sample-contiguous; k_mlp_grad
// spreads their 56 tiles per 256 samples over the chip.  Every sum keeps its
// order: products in steps of 16, weight gradients in blocks of 256 samples
// added in order, bias gradients by 256 strided sums and a tree, so a step does
// not depend on how samples are spread over blocks.
// A step is a chain of small products: bound by latency and by the SiLU
// evaluations, not by the matrix cores, so the rows are split, not only the
// samples.  A step at a batch of 1,024 / 4,096 / 16,384 / 65,536: 28 / 37 / 65 /
// 303 us (all steps of a call but its first); 59 / 82 us at 1,024 / 4,096 and
// 378 at 65,536 with 32 samples and all rows per wavefront (4 to a block,
// weights staged in LDS, SiLU' spilled); 540 us at 4,096 as 37 launches of
// single products and elementwise passes.  At 2 wavefronts per SIMD (44 bytes of
// spills) instead of 1, 65,536 took 295 instead of 323 us, 4,096 the same.
constexpr int kTrainTile = 32;      // samples per block
constexpr int kTrainThreads = 256;  // 4 wavefronts x 32 rows of a layer
constexpr int kGradChunk = 256;     // samples per weight-gradient block
constexpr int kAtRows = kMlpIn + 4 * kMlpHid, kDzRows = 4 * kMlpHid + kMlpOut;

struct TrainArgs {
  const __bf16 *x;      // [n_data][16]
  const float *t;       // [n_data][8]
  long n_data;          // > 0: samples drawn by `key`; 0: sample i of the batch is row i
  uint64_t key;
  int n;                // batch size
  size_t ld;            // samples rounded up to kGradChunk
  const __bf16 *Pb, *Wt;
  const float *P;
  __bf16 *at;           // activations [input 16, layers 1-4 128 each][ld]; zero past n
  __bf16 *dzb;          // dZ of layers 0-4 (128, ..., 8 rows) [ld], BF16 and FP32; zero past n
  float *dz;
  double *lpart;        // squared errors by block of samples
};

// Accumulators of a 32-row tile (rows 8 j + 4 h + r) as the two B operands of
// its 16-deep steps (depth 8 h + i), BF16.
__device__ __forceinline__ void tile_to_operands(const float (&v)[16], bf16x8 (&B)[2]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    unsigned a[2], b[2];  // rows 16 q + 4 h + {0..3}, 16 q + 8 + 4 h + {0..3}
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      bf16x2 lo = {(__bf16)v[8 * q + 2 * k], (__bf16)v[8 * q + 2 * k + 1]};
      bf16x2 hi = {(__bf16)v[8 * q + 4 + 2 * k], (__bf16)v[8 * q + 4 + 2 * k + 1]};
      a[k] = __builtin_bit_cast(unsigned, lo);
      b[k] = __builtin_bit_cast(unsigned, hi);
    }
    // upper half of a <-> lower half of b
    unsigned o[4];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const auto r = __builtin_amdgcn_permlane32_swap(a[k], b[k], false, false);
      o[k] = r[0];
      o[2 + k] = r[1];
    }
    struct Four { unsigned u[4]; };
    B[q] = __builtin_bit_cast(bf16x8, Four{{o[0], o[1], o[2], o[3]}});
  }
}

// SiLU and its derivative as z / (1 + e^-z) and s (1 + z (1 - s)), s = 1 / (1 +
// e^-z): the reciprocal refined to full precision serves both divisions.  It is
// taken of the denominator scaled down by a power of two: from 2^126 on (z below
// -87) a reciprocal is too small for the instruction, but not the quotients.
// (The same with the scaling only where it is needed and div_fixup for infinite
// operands: 428 bytes of spills instead of 44, 376 against 300 us per step at a
// batch of 65,536.)
__device__ __forceinline__ void silu_both(float z, float &v, float &d) {
  constexpr float kDown = 0x1p-64f;
  const float t = __expf(-z), ez = 1.0f + t, e = fmaf(t, kDown, kDown);
  float s = __builtin_amdgcn_rcpf(e);
  s = fmaf(fmaf(-e, s, 1.0f), s, s) * kDown;
  const bool finite = ez < INFINITY;
  s = finite ? s : 0.0f;
  const float q = z * s, w = fmaf(fmaf(-q, ez, z), s, q);
  v = z > 0x1p24f ? z : (finite ? w : q);  // (z itself, also where it is infinite)
  d = s * (1.0f + z * (1.0f - s));
}

// Weights of this lane's row of a product (16 STEPS deep), as A operands.
template <int STEPS>
__device__ __forceinline__ void fetch_row(const __bf16 *row, int h, bf16x8 (&A)[8]) {
#pragma unroll
  for (int k = 0; k < STEPS; ++k) A[k] = *reinterpret_cast<const bf16x8 *>(row + 16 * k + 8 * h);
}

template <int STEPS>
__device__ __forceinline__ f32x16 row_product(const bf16x8 (&A)[8], const bf16x8 (&B)[8]) {
  f32x16 acc = {};
#pragma unroll
  for (int k = 0; k < STEPS; ++k) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[k], B[k], acc, 0, 0, 0);
  return acc;
}

__global__ __launch_bounds__(kTrainThreads, 2) void k_mlp_train(TrainArgs g) {
  __shared__ bf16x8 ex[2][8][64];  // a layer's output as the next one's B operands, [32-row tile, half][lane]
  const int lane = threadIdx.x & 63, h = lane >> 5, c32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r0 = 32 * w + c32;                                // this lane's row of A in a product
  const size_t i = (size_t)blockIdx.x * kTrainTile + c32;     // sample in the batch (below ld)
  const bool valid = i < (size_t)g.n;
  const bf16x8 zero8 = {};
  bf16x8 A[2][8], B[8];  // weights of a layer and of the next
  fetch_row<1>(g.Pb + w_off(0) + r0 * kMlpIn, h, A[0]);
  size_t row = i;
  if (g.n_data > 0) row = (size_t)(mix64(g.key ^ (uint64_t)i * 0xD1B54A32D192ED03ull) % (uint64_t)g.n_data);
  B[0] = valid ? *reinterpret_cast<const bf16x8 *>(g.x + row * kMlpIn + 8 * h) : zero8;
  const float4 tv = valid ? *reinterpret_cast<const float4 *>(g.t + row * kMlpOut + 4 * h) : float4{0, 0, 0, 0};
  if (w == 0) {
#pragma unroll
    for (int k = 0; k < 8; ++k) g.at[(8 * h + k) * g.ld + i] = B[0][k];
  }
  // ---- forward: Z_l = W_l A_{l-1} + b_l, A_l = SiLU(Z_l)
  float zg[4][16];  // SiLU'(Z_l), l = 0-3
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    float4 b4[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) b4[j] = *reinterpret_cast<const float4 *>(g.P + b_off(l) + 32 * w + 8 * j + 4 * h);
    if (l < 3) {
      fetch_row<8>(g.Pb + w_off(l + 1) + r0 * kMlpHid, h, A[(l + 1) & 1]);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) A[0][k] = zero8;
      if (c32 < kMlpOut) fetch_row<8>(g.Pb + w_off(4) + c32 * kMlpHid, h, A[0]);
    }
    const f32x16 acc = l == 0 ? row_product<1>(A[0], B) : row_product<8>(A[l & 1], B);
    __bf16 *al = g.at + (size_t)(kMlpIn + l * kMlpHid + 32 * w) * g.ld + i;
    float v[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float bb[4] = {b4[j].x, b4[j].y, b4[j].z, b4[j].w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = 4 * j + r;
        silu_both(acc[e] + bb[r], v[e], zg[l][e]);
        al[(size_t)(8 * j + 4 * h + r) * g.ld] = valid ? (__bf16)v[e] : (__bf16)0.0f;
      }
    }
    bf16x8 two[2];
    tile_to_operands(v, two);
    ex[l & 1][2 * w][lane] = two[0];
    ex[l & 1][2 * w + 1][lane] = two[1];
    __syncthreads();  // (buffer l & 1 is written again two layers on, past the next barrier)
#pragma unroll
    for (int k = 0; k < 8; ++k) B[k] = ex[l & 1][k][lane];
  }
  // ---- output layer and loss, alike in every wavefront: mean squared error over the 6 used outputs
  const float4 bo = *reinterpret_cast<const float4 *>(g.P + b_off(4) + 4 * h);
  fetch_row<1>(g.Wt + wt_off(4) + r0 * 16, h, A[1]);
  const f32x16 o = row_product<8>(A[0], B);
  fetch_row<8>(g.Wt + wt_off(3) + r0 * kMlpHid, h, A[0]);
  float dy[4];
  double e2 = 0.0;
  {
    const float tt[4] = {tv.x, tv.y, tv.z, tv.w}, bb[4] = {bo.x, bo.y, bo.z, bo.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 4 * h + r;
      const float d = (o[r] + bb[r]) - tt[r];
      const bool use = valid && k < kMlpUsedOut;
      dy[r] = use ? 2.0f * d / (float)(kMlpUsedOut * (long)g.n) : 0.0f;
      if (use) e2 += (double)d * d;
    }
  }
  // dZ of the output layer: to memory, and as the B operand (depth 8: the lower half holds all 8)
  B[0] = zero8;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float other = __shfl_xor(dy[r], 32);
    B[0][r] = h ? (__bf16)0.0f : (__bf16)dy[r];
    B[0][4 + r] = h ? (__bf16)0.0f : (__bf16)other;
  }
  if (w == 0) {
    for (int m = 32; m > 0; m >>= 1) e2 += __shfl_xor(e2, m);
    if (lane == 0) g.lpart[blockIdx.x] = e2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const size_t at = (size_t)(4 * kMlpHid + 4 * h + r) * g.ld + i;
      g.dz[at] = dy[r];
      g.dzb[at] = (__bf16)dy[r];
    }
  }
  // ---- backward: dA_{l-1} = W_l^T dZ_l; dZ_{l-1} = dA SiLU'(Z_{l-1})
#pragma unroll
  for (int l = 4; l >= 1; --l) {
    const f32x16 acc = l == 4 ? row_product<1>(A[1], B) : row_product<8>(A[(l + 1) & 1], B);
    if (l == 4 || l == 3) fetch_row<8>(g.Wt + wt_off(l - 2) + r0 * kMlpHid, h, A[(l + 1) & 1]);
    float v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const size_t at = (size_t)((l - 1) * kMlpHid + 32 * w + 8 * (e >> 2) + 4 * h + (e & 3)) * g.ld + i;
      v[e] = valid ? acc[e] * zg[l - 1][e] : 0.0f;
      g.dz[at] = v[e];
      g.dzb[at] = (__bf16)v[e];
    }
    if (l > 1) {
      bf16x8 two[2];
      tile_to_operands(v, two);
      ex[l & 1][2 * w][lane] = two[0];
      ex[l & 1][2 * w + 1][lane] = two[1];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 8; ++k) B[k] = ex[l & 1][k][lane];
    }
  }
}

// Weight and bias gradients from k_mlp_train's arrays.  The first kDzRows
// blocks: the bias gradients, one row of dZ each, summed in a fixed order into
// db.  Then 14 blocks x per 256 samples z: weight gradients of samples [256 z,
// + 256), dW_l[o][i] = sum_s dZ_l[o][s] A_{l-1}[i][s], a 32x32 tile per
// wavefront (layer 0: x 0, one output tile per wavefront; layers 1-3: x 1-12,
// an output tile each, an input tile per wavefront; layer 4: x 13), into
// parts[z].  (Numbered through: as a grid of (14 + kDzRows) x chunks all but
// the first chunk's bias blocks were empty; a training step at a batch of 4,096
// / 16,384: 40 / 68 us, then 35 / 63 us.)
constexpr int kGradTiles = 14;
__global__ __launch_bounds__(256) void k_mlp_grad(const __bf16 *at, const __bf16 *dzb, const float *dz, size_t ld,
                                                  float *parts, float *db) {
  const int w = threadIdx.x >> 6;
  if (blockIdx.x < kDzRows) {
    __shared__ float sh[256];
    const float *src = dz + (size_t)blockIdx.x * ld;
    float q = 0.0f;
    for (size_t k = threadIdx.x; k < ld; k += 256) q += src[k];
    sh[threadIdx.x] = q;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
      __syncthreads();
    }
    if (threadIdx.x == 0) db[blockIdx.x] = sh[0];
    return;
  }
  const int x = (blockIdx.x - kDzRows) % kGradTiles, z = (blockIdx.x - kDzRows) / kGradTiles;
  const int l = x == 0 ? 0 : (x == 13 ? 4 : 1 + (x - 1) / 4);
  const int ot = x == 0 ? w : (x == 13 ? 0 : (x - 1) % 4), it = x == 0 ? 0 : w;
  const int in = layer_in(l), out = layer_out(l);
  const int lane = threadIdx.x & 63, h = lane >> 5, c32 = lane & 31;
  const int r = 32 * ot + c32, c = 32 * it + c32;
  const size_t s0 = (size_t)z * kGradChunk + 8 * h;
  const __bf16 *ap = dzb + (size_t)(l * kMlpHid + r) * ld + s0;
  const __bf16 *bp = at + (size_t)((l == 0 ? 0 : kMlpIn + (l - 1) * kMlpHid) + c) * ld + s0;
  const bf16x8 zero8 = {};
  bf16x8 a[kGradChunk / 16], b[kGradChunk / 16];
#pragma unroll
  for (int k = 0; k < kGradChunk / 16; ++k) {
    a[k] = r < out ? *reinterpret_cast<const bf16x8 *>(ap + 16 * k) : zero8;
    b[k] = c < in ? *reinterpret_cast<const bf16x8 *>(bp + 16 * k) : zero8;
  }
  f32x16 acc = {};
#pragma unroll
  for (int k = 0; k < kGradChunk / 16; ++k) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[k], b[k], acc, 0, 0, 0);
  if (c >= in) return;
  float *dst = parts + (size_t)z * kParams + w_off(l) + c;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int o = 32 * ot + 8 * (e >> 2) + 4 * h + (e & 3);
    if (o < out) dst[o * in] = acc[e];
  }
}

// Gradients: the weights' parts added in order, the biases' as they are; with
// `adam`, the parameter update and its BF16 copies.
__global__ void k_mlp_update(const float *parts, int nz, const float *db, float *G, int adam, float *P, float *m,
                             float *v, float lr, float c1, float c2, __bf16 *Pb, __bf16 *Wt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kParams) return;
  const int l = layer_of(i);
  float g = 0.0f;
  if (i >= b_off(l)) {
    g = db[l * kMlpHid + i - b_off(l)];
  } else {
    int z = 0;
    for (; z + 8 <= nz; z += 8) {  // 8 loads in flight
      float q[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) q[k] = parts[(size_t)(z + k) * kParams + i];
#pragma unroll
      for (int k = 0; k < 8; ++k) g += q[k];
    }
    for (; z < nz; ++z) g += parts[(size_t)z * kParams + i];
  }
  G[i] = g;
  if (!adam) return;
  const float mi = 0.9f * m[i] + 0.1f * g;
  const float vi = 0.999f * v[i] + 0.001f * g * g;
  m[i] = mi;
  v[i] = vi;
  const float p = P[i] - lr * (mi * c1) / (sqrtf(vi * c2) + 1e-8f);
  P[i] = p;
  store_copies(i, p, Pb, Wt);
}

__global__ void k_to_bf16(const float *x, size_t n, __bf16 *y) {
  const size_t i = 4 * ((size_t)blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= n) return;  // n is a multiple of 16
  const float4 v = *reinterpret_cast<const float4 *>(x + i);
  y[i] = (__bf16)v.x;
  y[i + 1] = (__bf16)v.y;
  y[i + 2] = (__bf16)v.z;
  y[i + 3] = (__bf16)v.w;
}

int blocks(long n, int b = 256) { return (int)((n + b - 1) / b); }

}  // namespace

struct MlpNet {
  float *P = nullptr, *G = nullptr, *m = nullptr, *v = nullptr;
  __bf16 *Pb = nullptr, *Wi = nullptr, *Wt = nullptr;
  bool wi_stale = false;  // Wi (inference) is behind P
  int adam_t = 0;
  int n_cu = 0;  // compute units (persistent inference grid)
  // training workspace for batches up to `ld` samples
  size_t ld = 0;
  __bf16 *at = nullptr, *dzb = nullptr;
  float *dz = nullptr, *parts = nullptr, *db = nullptr;
  double *lpart = nullptr;
};

namespace {

void free_ws(MlpNet *n) {
  for (void *p : {(void *)n->at, (void *)n->dzb, (void *)n->dz, (void *)n->parts, (void *)n->db, (void *)n->lpart})
    if (p) (void)hipFree(p);
  n->at = n->dzb = nullptr;
  n->dz = n->parts = n->db = nullptr;
  n->lpart = nullptr;
  n->ld = 0;
}

size_t train_ld(int batch) { return ((size_t)batch + kGradChunk - 1) / kGradChunk * kGradChunk; }

int ensure_ws(MlpNet *n, int batch) {
  const size_t ld = train_ld(batch);
  if (ld <= n->ld) return 0;
  free_ws(n);
  MCHK(hipMalloc(&n->at, kAtRows * ld * sizeof(__bf16)));
  MCHK(hipMalloc(&n->dzb, kDzRows * ld * sizeof(__bf16)));
  MCHK(hipMalloc(&n->dz, kDzRows * ld * sizeof(float)));
  MCHK(hipMalloc(&n->parts, ld / kGradChunk * kParams * sizeof(float)));
  MCHK(hipMalloc(&n->db, kDzRows * sizeof(float)));
  MCHK(hipMalloc(&n->lpart, ld / kTrainTile * sizeof(double)));
  n->ld = ld;
  return 0;
}

int refresh(MlpNet *net, hipStream_t st) {
  hipLaunchKernelGGL(k_refresh, dim3(blocks(std::max(kParams, kWi))), dim3(256), 0, st, net->P, net->Pb, net->Wi,
                     net->Wt);
  MCHK(hipGetLastError());
  net->wi_stale = false;
  return 0;
}

struct AdamStep {
  float lr, c1, c2;
};

// One batch: gradients into G and, with `adam`, the parameter update.
// n_data > 0 draws the batch from (x, t) by `key`, else it is their first n
// rows.
int train_batch(MlpNet *net, const __bf16 *x, const float *t, long n_data, uint64_t key, int n, const AdamStep *adam,
                hipStream_t st) {
  int rc;
  if ((rc = ensure_ws(net, n))) return rc;
  const size_t ld = train_ld(n);
  const TrainArgs g{x, t, n_data, key, n, ld, net->Pb, net->Wt, net->P, net->at, net->dzb, net->dz, net->lpart};
  hipLaunchKernelGGL(k_mlp_train, dim3((unsigned)(ld / kTrainTile)), dim3(kTrainThreads), 0, st, g);
  MCHK(hipGetLastError());
  const int nz = (int)(ld / kGradChunk);
  hipLaunchKernelGGL(k_mlp_grad, dim3(kDzRows + kGradTiles * nz), dim3(256), 0, st, net->at, net->dzb, net->dz, ld,
                     net->parts, net->db);
  MCHK(hipGetLastError());
  hipLaunchKernelGGL(k_mlp_update, dim3(blocks(kParams)), dim3(256), 0, st, net->parts, nz, net->db, net->G,
                     adam ? 1 : 0, net->P, net->m, net->v, adam ? adam->lr : 0.0f, adam ? adam->c1 : 0.0f,
                     adam ? adam->c2 : 0.0f, net->Pb, net->Wt);
  MCHK(hipGetLastError());
  if (adam) net->wi_stale = true;
  return 0;
}

int read_loss(MlpNet *net, int n, hipStream_t st, double *loss) {
  std::vector<double> part(train_ld(n) / kTrainTile);
  MCHK(hipMemcpyAsync(part.data(), net->lpart, part.size() * sizeof(double), hipMemcpyDeviceToHost, st));
  MCHK(hipStreamSynchronize(st));
  double s = 0.0;
  for (size_t k = 0; k < part.size(); k += 4) s += part[k] + part[k + 1] + part[k + 2] + part[k + 3];
  *loss = s / ((double)n * kMlpUsedOut);
  return 0;
}

}  // namespace

int mlp_param_count() { return kParams; }

int mlp_create(unsigned long long seed, MlpNet **out) {
  MlpNet *n = new MlpNet();
  *out = nullptr;
  auto bail = [&](int rc) {
    mlp_destroy(n);
    return rc;
  };
  if (hipMalloc(&n->P, kParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&n->G, kParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&n->m, kParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&n->v, kParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&n->Pb, kParams * sizeof(__bf16)) != hipSuccess ||
      hipMalloc(&n->Wi, kWi * sizeof(__bf16)) != hipSuccess ||
      hipMalloc(&n->Wt, kWt * sizeof(__bf16)) != hipSuccess)
    return bail(mfail(FT_ERR_ALLOC, "network allocation failed"));
  // Glorot-uniform weights from a 64-bit mix of (seed, index), zero biases
  std::vector<float> h(kParams, 0.0f);
  for (int l = 0; l < kMlpLayers; ++l) {
    const int fi = l == 0 ? kMlpUsedIn : layer_in(l), fo = l == kMlpLayers - 1 ? kMlpUsedOut : layer_out(l);
    const double a = sqrt(6.0 / (fi + fo));
    for (int o = 0; o < fo; ++o)
      for (int i = 0; i < fi; ++i) {
        uint64_t z = seed * 0x9E3779B97F4A7C15ull + (uint64_t)(w_off(l) + o * layer_in(l) + i) + 1;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        const double u = (double)(z >> 11) * (1.0 / 9007199254740992.0);
        h[w_off(l) + o * layer_in(l) + i] = (float)((2.0 * u - 1.0) * a);
      }
  }
  int rc = mlp_set_params(n, h.data());
  if (rc) return bail(rc);
  *out = n;
  return 0;
}

void mlp_destroy(MlpNet *n) {
  if (!n) return;
  (void)hipDeviceSynchronize();
  free_ws(n);
  for (void *p : {(void *)n->P, (void *)n->G, (void *)n->m, (void *)n->v, (void *)n->Pb, (void *)n->Wi,
                  (void *)n->Wt})
    if (p) (void)hipFree(p);
  delete n;
}

int mlp_get_params(MlpNet *net, float *host) {
  MCHK(hipMemcpy(host, net->P, kParams * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

int mlp_set_params(MlpNet *net, const float *host) {
  MCHK(hipMemcpy(net->P, host, kParams * sizeof(float), hipMemcpyHostToDevice));
  MCHK(hipMemset(net->m, 0, kParams * sizeof(float)));
  MCHK(hipMemset(net->v, 0, kParams * sizeof(float)));
  MCHK(hipMemset(net->G, 0, kParams * sizeof(float)));
  net->adam_t = 0;
  int rc = refresh(net, nullptr);
  if (rc) return rc;
  MCHK(hipDeviceSynchronize());
  return 0;
}

int mlp_copy_gradients(MlpNet *net, float *host) {
  MCHK(hipMemcpy(host, net->G, kParams * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

int mlp_infer(MlpNet *net, const __bf16 *x, long n, float *y, hipStream_t st) {
  if (n <= 0) return 0;
  int rc;
  if (net->wi_stale && (rc = refresh(net, st))) return rc;
  if (!net->n_cu) {
    int dev = 0;
    MCHK(hipGetDevice(&dev));
    MCHK(hipDeviceGetAttribute(&net->n_cu, hipDeviceAttributeMultiprocessorCount, dev));
  }
  const long slabs = (n + 32 * kInferTiles - 1) / (32 * kInferTiles), per_block = kInferThreads / 64;
  const long blocks_needed = (slabs + per_block - 1) / per_block;
  const unsigned grid = (unsigned)std::min<long>(blocks_needed, (long)net->n_cu);
  hipLaunchKernelGGL((k_mlp_infer<kInferTiles, kInferThreads>), dim3(grid), dim3(kInferThreads), 0, st, x, n,
                     net->Wi, net->P, y);
  MCHK(hipGetLastError());
  return 0;
}

int mlp_gradients(MlpNet *net, const __bf16 *x, const float *t, int n, hipStream_t st, double *loss) {
  if (n <= 0) return mfail(FT_ERR_ARG, "empty batch");
  int rc;
  if ((rc = train_batch(net, x, t, 0, 0, n, nullptr, st))) return rc;
  return loss ? read_loss(net, n, st, loss) : 0;
}

int mlp_train(MlpNet *net, const __bf16 *x, const float *t, long n_data, int steps, int batch, float lr,
              unsigned long long seed, hipStream_t st, double *final_loss) {
  if (n_data <= 0 || batch <= 0 || steps < 0) return mfail(FT_ERR_ARG, "empty training set or batch");
  int rc;
  double acc = 0.0;
  int nacc = 0;
  for (int k = 0; k < steps; ++k) {
    const uint64_t key = seed * 0x9E3779B97F4A7C15ull ^ ((uint64_t)k << 20);
    const float lr_k = lr * (0.02f + 0.98f * 0.5f * (1.0f + cosf(3.14159265f * (float)k / (float)steps)));
    const int at = net->adam_t + 1;
    const AdamStep a{lr_k, (float)(1.0 / (1.0 - pow(0.9, at))), (float)(1.0 / (1.0 - pow(0.999, at)))};
    if ((rc = train_batch(net, x, t, n_data, key, batch, &a, st))) return rc;
    net->adam_t = at;  // (a step that could not be launched is none)
    // the loss is read back (a synchronisation) only over the last 1 % of steps
    if (final_loss && k >= steps - std::max(1, steps / 100)) {
      double l = 0.0;
      if ((rc = read_loss(net, batch, st, &l))) return rc;
      acc += l;
      ++nacc;
    }
  }
  if (net->wi_stale && (rc = refresh(net, st))) return rc;
  MCHK(hipStreamSynchronize(st));
  if (final_loss) *final_loss = nacc ? acc / nacc : 0.0;
  return 0;
}

}  // namespace ft

// ---------------------------------------------------------------------------
// C ABI of the stand-alone network (host arrays; tests and tools)
// ---------------------------------------------------------------------------
struct ft_mlp {
  ft::MlpNet *net = nullptr;
};

namespace {

int to_device_f32(const float *host, size_t count, float **dev) {
  if (hipMalloc(dev, count * sizeof(float)) != hipSuccess) return ft::mfail(FT_ERR_ALLOC, "allocation failed");
  if (hipMemcpy(*dev, host, count * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
    return ft::mfail(FT_ERR_HIP, "copy failed");
  return 0;
}

// Rounded on the device: the host's conversion loop took longer than the copy.
int to_device_bf16(const float *host, size_t count, __bf16 **dev) {
  float *f = nullptr;
  int rc = to_device_f32(host, count, &f);
  if (!rc && hipMalloc(dev, count * sizeof(__bf16)) != hipSuccess) rc = ft::mfail(FT_ERR_ALLOC, "allocation failed");
  if (!rc) {
    hipLaunchKernelGGL(ft::k_to_bf16, dim3((unsigned)((count / 4 + 255) / 256)), dim3(256), 0, nullptr, f, count, *dev);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess)
      rc = ft::mfail(FT_ERR_HIP, "conversion failed");
  }
  if (f) (void)hipFree(f);
  return rc;
}

int device_ok() {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return ft::mfail(FT_ERR_HIP, "no HIP device available");
  return 0;
}

}  // namespace

extern "C" {

int ft_mlp_param_count(void) { return ft::kParams; }

int ft_mlp_create(unsigned long long seed, ft_mlp **out) {
  if (!out) return ft::mfail(FT_ERR_ARG, "null argument");
  *out = nullptr;
  int rc;
  if ((rc = device_ok())) return rc;
  ft_mlp *m = new ft_mlp();
  if ((rc = ft::mlp_create(seed, &m->net))) {
    delete m;
    return rc;
  }
  *out = m;
  return 0;
}

int ft_mlp_destroy(ft_mlp *m) {
  if (!m) return 0;
  ft::mlp_destroy(m->net);
  delete m;
  return 0;
}

int ft_mlp_get_params(ft_mlp *m, float *params) {
  if (!m || !params) return ft::mfail(FT_ERR_ARG, "null argument");
  return ft::mlp_get_params(m->net, params);
}

int ft_mlp_set_params(ft_mlp *m, const float *params) {
  if (!m || !params) return ft::mfail(FT_ERR_ARG, "null argument");
  return ft::mlp_set_params(m->net, params);
}

int ft_mlp_forward(ft_mlp *m, const float *x, int n, float *y) {
  if (!m || !x || !y || n < 0) return ft::mfail(FT_ERR_ARG, "bad argument");
  if (n == 0) return 0;
  __bf16 *dx = nullptr;
  float *dy = nullptr;
  int rc = to_device_bf16(x, (size_t)n * ft::kMlpIn, &dx);
  if (!rc && hipMalloc(&dy, (size_t)n * ft::kMlpOut * sizeof(float)) != hipSuccess)
    rc = ft::mfail(FT_ERR_ALLOC, "allocation failed");
  if (!rc) rc = ft::mlp_infer(m->net, dx, n, dy, nullptr);
  if (!rc && hipMemcpy(y, dy, (size_t)n * ft::kMlpOut * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
    rc = ft::mfail(FT_ERR_HIP, "copy failed");
  if (dx) (void)hipFree(dx);
  if (dy) (void)hipFree(dy);
  return rc;
}

int ft_mlp_gradients(ft_mlp *m, const float *x, const float *t, int n, double *loss, float *grad) {
  if (!m || !x || !t || n <= 0) return ft::mfail(FT_ERR_ARG, "bad argument");
  __bf16 *dx = nullptr;
  float *dt = nullptr;
  int rc = to_device_bf16(x, (size_t)n * ft::kMlpIn, &dx);
  if (!rc) rc = to_device_f32(t, (size_t)n * ft::kMlpOut, &dt);
  if (!rc) rc = ft::mlp_gradients(m->net, dx, dt, n, nullptr, loss);
  if (!rc && grad) rc = ft::mlp_copy_gradients(m->net, grad);
  if (dx) (void)hipFree(dx);
  if (dt) (void)hipFree(dt);
  return rc;
}

int ft_mlp_train(ft_mlp *m, const float *x, const float *t, int n_data, int steps, int batch, double lr,
                 unsigned long long seed, double *final_loss) {
  if (!m || !x || !t || n_data <= 0) return ft::mfail(FT_ERR_ARG, "bad argument");
  __bf16 *dx = nullptr;
  float *dt = nullptr;
  int rc = to_device_bf16(x, (size_t)n_data * ft::kMlpIn, &dx);
  if (!rc) rc = to_device_f32(t, (size_t)n_data * ft::kMlpOut, &dt);
  if (!rc) rc = ft::mlp_train(m->net, dx, dt, n_data, steps, batch, (float)lr, seed, nullptr, final_loss);
  if (dx) (void)hipFree(dx);
  if (dt) (void)hipFree(dt);
  return rc;
}

}  // extern "C"
