// MLP surrogate kernels: a batch's forward and backward pass (bf16 matrix-core products with FP32 accumulation, Fourier
// features, SiLU, loss), weight and bias gradients, Adam, and table prediction.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "surrogate.hpp"

namespace sfsim {

namespace {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kEw = 256;  // elementwise block size

__host__ __device__ inline uint16_t f2bf(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// SiLU and its derivative with the hardware reciprocal (1 ulp) instead of an IEEE division: the
// results are rounded to bf16 for the products anyway.
__device__ __forceinline__ float sigmoid(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

__device__ __forceinline__ float silu(float z) { return z * sigmoid(z); }

__device__ __forceinline__ float dsilu(float z) {
  float s = sigmoid(z);
  return s * (1.0f + z * (1.0f - s));
}

__host__ __device__ inline uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// The 17 Fourier features of one input x: x, then sin / cos (2^b pi x) for b = 0..7 (bf16).
__device__ inline uint16_t encode_feature(float v, int q) {
  if (q == 0) return f2bf(v);
  float sn, cs;
  sincosf(ldexpf(3.14159265358979f * v, (q - 1) >> 1), &sn, &cs);
  return f2bf(q & 1 ? sn : cs);
}

__device__ inline void entry_coords(const GridShape& P, long long entry, float* x) {
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  int ia = (int)(entry % NA);
  long long q = entry / NA;
  int is = (int)(q % NL);
  q /= NL;
  int ie = (int)(q % NE);
  int ih = (int)(q / NE);
  x[0] = (float)ih / (NH - 1);
  x[1] = (float)ie / (NE - 1);
  x[2] = (float)is / (NL - 1);
  x[3] = (float)ia / (NA - 1);
}

struct SumTables {
  const float4* p[kMlpOrders];
};

__global__ void targets_kernel(const SumTables sums, long long entries, float* __restrict__ t) {
  long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= entries) return;
  for (int k = 0; k < kMlpOrders; ++k) {
    const float4 v = sums.p[k][e];
    t[e * kMlpUsed + 3 * k + 0] = logf(fmaxf(v.x, 0.f) + kMlpEps) + kMlpShift;
    t[e * kMlpUsed + 3 * k + 1] = logf(fmaxf(v.y, 0.f) + kMlpEps) + kMlpShift;
    t[e * kMlpUsed + 3 * k + 2] = logf(fmaxf(v.z, 0.f) + kMlpEps) + kMlpShift;
  }
}

// out[c] = mean over rows of T[row][c] for the kMlpUsed target columns (row stride kMlpUsed), FP64
// partial sums in a fixed order: the output biases' initial values.
__global__ void __launch_bounds__(kEw) target_mean_kernel(const float* __restrict__ T, long long rows,
                                                          float* __restrict__ out) {
  __shared__ double red[kEw / 64];
  const int c = blockIdx.x;
  double s = 0.0;
  for (long long r = threadIdx.x; r < rows; r += blockDim.x) s += T[r * kMlpUsed + c];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kEw / 64; ++w) t += red[w];
    out[c] = (float)(t / (double)rows);
  }
}

// ---- one pass over a batch: forward, loss and backward --------------------------------------------
// Every product runs on v_mfma_f32_32x32x8bf16_1k, K in ascending steps of 8.  Operand layout of that instruction: lane l
// supplies A(l % 32, 4 (l / 32) + i) and B(4 (l / 32) + i, l % 32), i = 0..3; accumulator element e of lane l is
// C(8 (e / 4) + 4 (l / 32) + e % 4, l % 32).  Operands that come from memory lie there as "fragments": for each tile of 32
// and step of 8 the 64 lanes' 4 values side by side (8 bytes per lane, one coalesced read per step).  What a
// lane's accumulator holds of 32 rows, rows 8 g + 4 h + i of one column, is its fragment of the products that sum over
// the rows (the weight gradients), for steps g = 0..3: it is written as it stands.
constexpr int kRows = 32;  // rows of the batch per workgroup
constexpr int kFragWaves = 4;

// Weight fragments in units of one step of one tile (256 values): forward layers (B operand W(k, n)), then the backward
// products dA = dZ W^T of layers 2, 3 and 4 (B operand W(n, k)).
struct FragLayout {
  static constexpr int f1 = 0, f2 = f1 + 4 * kMlpFeat / 8, f3 = f2 + 4 * kMlpHidden / 8, f4 = f3 + 4 * kMlpHidden / 8;
  static constexpr int b2 = f4 + kMlpHidden / 8, b3 = b2 + 4 * kMlpHidden / 8, b4 = b3 + 4 * kMlpHidden / 8;
  static constexpr int total = b4 + 4 * kMlpOut / 8;
};
static_assert(FragLayout::total * 256 == kMlpFragments, "size of the weight fragments");

__device__ __forceinline__ int frag_index(int tile, int steps, int k, int n) {
  return (tile * steps + k / 8) * 256 + ((n & 31) + 32 * ((k & 7) >> 2)) * 4 + (k & 3);
}

// The bf16 copies of weight i (a row-major one and its fragments); biases have none.
__device__ __forceinline__ void store_bf16(size_t i, uint16_t v, uint16_t* __restrict__ bf, uint16_t* __restrict__ frag) {
  bf[i] = v;
  const size_t off[4] = {MlpLayout::W1, MlpLayout::W2, MlpLayout::W3, MlpLayout::W4};
  const int kin[4] = {kMlpFeat, kMlpHidden, kMlpHidden, kMlpHidden}, out[4] = {kMlpHidden, kMlpHidden, kMlpHidden, kMlpOut};
  const int fwd[4] = {FragLayout::f1, FragLayout::f2, FragLayout::f3, FragLayout::f4};
  const int bwd[4] = {-1, FragLayout::b2, FragLayout::b3, FragLayout::b4};
#pragma unroll
  for (int l = 0; l < 4; ++l)
    if (i >= off[l] && i < off[l] + (size_t)kin[l] * out[l]) {
      const int k = (int)(i - off[l]) / out[l], n = (int)(i - off[l]) % out[l];
      frag[fwd[l] * 256 + frag_index(n / 32, kin[l] / 8, k, n)] = v;
      if (bwd[l] >= 0) frag[bwd[l] * 256 + frag_index(k / 32, out[l] / 8, n, k)] = v;
    }
}

// A tile's weight fragments in registers, and its product over STEPS steps with the rows' values in LDS (row pitch in
// values).
template <int STEPS>
struct Frags {
  short4_t v[STEPS];
};

template <int STEPS>
__device__ __forceinline__ Frags<STEPS> load_frags(const uint16_t* __restrict__ frag, int lane) {
  Frags<STEPS> f;
#pragma unroll
  for (int k = 0; k < STEPS; ++k) f.v[k] = *(const short4_t*)(frag + (k * 64 + lane) * 4);
  return f;
}

template <int STEPS>
__device__ __forceinline__ float16_t tile_product(const uint16_t* a, int pitch, const Frags<STEPS>& w, int lane) {
  float16_t acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  const uint16_t* row = a + (lane & 31) * pitch + 4 * (lane >> 5);
#pragma unroll
  for (int k = 0; k < STEPS; ++k)
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(*(const short4_t*)(row + 8 * k), w.v[k], acc, 0, 0, 0);
  return acc;
}

// Four rows of a lane's column: into the LDS tile of the next product and the fragments of the weight gradient.
__device__ __forceinline__ void store_rows(const float (&v)[4], uint16_t* lds, int pitch, uint16_t* __restrict__ frag) {
  uint16_t b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    b[i] = f2bf(v[i]);
    if (lds) lds[i * pitch] = b[i];
  }
  *(uint2*)frag = make_uint2(b[0] | (uint32_t)b[1] << 16, b[2] | (uint32_t)b[3] << 16);
}

// Row pitches (values) of the LDS tiles: 2 dwords modulo the 32 banks, so that 16 rows' 8-byte reads do not collide.
constexpr int kPitchX = kMlpFeat + 4, kPitchH = kMlpHidden + 4, kPitchY = kMlpOut + 4;

// Forward, loss and backward of 32 rows by one workgroup of 4 wavefronts, wavefront w computing columns 32 w .. 32 w + 31 of
// every hidden layer: activations stay in LDS (bf16, as the products take them) and pre-activations in
// registers.  The rows are given (in, with targets T) or drawn from the training data.  One launch for what had
// been gather, four products, loss, three products, three activation derivatives, each through memory.
__global__ void __launch_bounds__(64 * kFragWaves) pass_kernel(const PassSource src, int rows, const uint16_t* __restrict__ wfrag,
                                                               const float* __restrict__ theta, const PassOutputs out) {
  __shared__ __align__(16) uint16_t s_x[kRows * kPitchX];
  __shared__ __align__(16) uint16_t s_a[2][kRows * kPitchH];
  __shared__ __align__(16) uint16_t s_dy[kRows * kPitchY];
  __shared__ float s_y[kRows][kMlpOut], s_t[kRows][kMlpOut], s_in[kRows][kMlpIn];
  __shared__ float s_red[kFragWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, col = 32 * wave + (lane & 31);
  const int row0 = blockIdx.x * kRows, steps = gridDim.x * (kRows / 8), step0 = blockIdx.x * (kRows / 8);
  // the weights of a layer are requested a layer (the first two: the whole input stage) before they are needed: a
  // workgroup has its CU to itself, so nothing else hides their latency, and registers are free
  const auto w1 = load_frags<kMlpFeat / 8>(wfrag + (FragLayout::f1 + wave * (kMlpFeat / 8)) * 256, lane);
  const auto w2 = load_frags<kMlpHidden / 8>(wfrag + (FragLayout::f2 + wave * (kMlpHidden / 8)) * 256, lane);
  const float bias1 = theta[MlpLayout::b1 + col], bias2 = theta[MlpLayout::b2 + col], bias3 = theta[MlpLayout::b3 + col];
  // inputs and targets
  if (tid < kRows) {
    const int r = row0 + tid;
    float x[kMlpIn] = {};
    if (r < rows) {
      if (src.in) {
        for (int i = 0; i < kMlpIn; ++i) x[i] = src.in[(long long)r * kMlpIn + i];
      } else {
        const long long entries = (long long)src.P.nS[0] * src.P.nS[1] * src.P.nS[2] * src.P.nS[3];
        const uint64_t hash = splitmix64(src.seed ^ splitmix64(((uint64_t)src.step << 32) | (uint64_t)r));
        const int atm = (int)(hash % (uint64_t)src.natm);
        const long long entry = (long long)((hash >> 16) % (uint64_t)entries);
        entry_coords(src.P, entry, x);
        for (int i = 0; i < 6; ++i) x[4 + i] = src.codes[atm].v[i];
        const float* t = src.targets + ((long long)atm * entries + entry) * kMlpUsed;
        for (int o = 0; o < kMlpOut; ++o) s_t[tid][o] = o < kMlpUsed ? t[o] : 0.f;
      }
    }
    for (int i = 0; i < kMlpIn; ++i) s_in[tid][i] = x[i];
  }
  if (src.T)
    for (int i = tid; i < kRows * kMlpOut; i += blockDim.x)
      s_t[i / kMlpOut][i % kMlpOut] = row0 + i / kMlpOut < rows ? src.T[(long long)row0 * kMlpOut + i] : 0.f;
  __syncthreads();
  // features: x, then sin / cos of 2^b pi x, zero padded; rows past the batch are zero
  for (int i = tid; i < kRows * kMlpIn * 8; i += blockDim.x) {
    const int r = i / (kMlpIn * 8), q = i - r * (kMlpIn * 8), in = q >> 3, band = q & 7;
    uint16_t* f = s_x + r * kPitchX + kMlpBands * in;
    const float v = s_in[r][in];
    float sn, cs;
    sincosf(3.14159265358979f * v * (float)(1 << band), &sn, &cs);
    const bool valid = row0 + r < rows;
    if (band == 0) f[0] = valid ? f2bf(v) : 0;
    f[1 + 2 * band] = valid ? f2bf(sn) : 0;
    f[2 + 2 * band] = valid ? f2bf(cs) : 0;
  }
  for (int i = tid; i < kRows * (kMlpFeat - kMlpBands * kMlpIn); i += blockDim.x)
    s_x[(i / (kMlpFeat - kMlpBands * kMlpIn)) * kPitchX + kMlpBands * kMlpIn + i % (kMlpFeat - kMlpBands * kMlpIn)] = 0;
  __syncthreads();
  if (out.dZ[0])  // the features' fragments for the first layer's weight gradient
    for (int i = tid; i < (kMlpFeat / 32) * (kRows / 8) * 64; i += blockDim.x) {
      const int tile = i / (4 * 64), g = (i / 64) & 3, l = i & 63;
      const uint16_t* v = s_x + (8 * g + 4 * (l >> 5)) * kPitchX + 32 * tile + (l & 31);
      *(uint2*)(out.X + ((size_t)(tile * steps + step0 + g) * 64 + l) * 4) =
          make_uint2(v[0] | (uint32_t)v[kPitchX] << 16, v[2 * kPitchX] | (uint32_t)v[3 * kPitchX] << 16);
    }
  // hidden layers: Z = A W + b, A = SiLU(Z)
  float z[3][16];
  auto activate = [&](int l, const float16_t acc, float b) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float a[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        z[l][4 * g + i] = acc[4 * g + i] + b;
        a[i] = silu(z[l][4 * g + i]);
        if (row0 + 8 * g + 4 * h + i >= rows) a[i] = 0.f;  // (of the biases alone, not of a row: may be infinite)
      }
      store_rows(a, s_a[l & 1] + (8 * g + 4 * h) * kPitchH + col, kPitchH,
                 out.A[l] + ((size_t)(wave * steps + step0 + g) * 64 + lane) * 4);
    }
    __syncthreads();
  };
  activate(0, tile_product(s_x, kPitchX, w1, lane), bias1);
  const auto w3 = load_frags<kMlpHidden / 8>(wfrag + (FragLayout::f3 + wave * (kMlpHidden / 8)) * 256, lane);
  activate(1, tile_product(s_a[0], kPitchH, w2, lane), bias2);
  const auto w4 = load_frags<kMlpHidden / 8>(wfrag + FragLayout::f4 * 256, lane);
  activate(2, tile_product(s_a[1], kPitchH, w3, lane), bias3);
  const auto v4 = load_frags<kMlpOut / 8>(wfrag + (FragLayout::b4 + wave * (kMlpOut / 8)) * 256, lane);
  const auto v3 = load_frags<kMlpHidden / 8>(wfrag + (FragLayout::b3 + wave * (kMlpHidden / 8)) * 256, lane);
  // outputs (one wavefront: 16 columns)
  if (wave == 0) {
    const float16_t acc = tile_product(s_a[0], kPitchH, w4, lane);
    if (col < kMlpOut) {
      const float b = theta[MlpLayout::b4 + col];
#pragma unroll
      for (int e = 0; e < 16; ++e) s_y[(e >> 2) * 8 + 4 * h + (e & 3)][col] = acc[e] + b;
    }
  }
  __syncthreads();
  if (out.Y)
    for (int i = tid; i < kRows * kMlpOut; i += blockDim.x)
      if (row0 + i / kMlpOut < rows) out.Y[(long long)row0 * kMlpOut + i] = s_y[i / kMlpOut][i % kMlpOut];
  if (!out.dZ[0]) return;
  // dY = mask (Y - T) / rows; loss partials 0.5 sum d^2 / rows per 256 values (16 rows)
  for (int blk = 0; blk < kRows * kMlpOut / kEw; ++blk) {
    const int i = blk * kEw + tid, r = i / kMlpOut, o = i % kMlpOut;
    const bool valid = row0 + r < rows;
    float l = 0.f, g = 0.f;
    if (valid) {
      const float d = o < kMlpUsed ? (s_y[r][o] - s_t[r][o]) : 0.f;
      l = 0.5f * d * d / rows;
      g = d / rows;
      out.dYf[(size_t)o * (8 * steps) + row0 + r] = g;
    }
    s_dy[r * kPitchY + o] = f2bf(g);
    for (int off = 32; off > 0; off >>= 1) l += __shfl_down(l, off, 64);
    if (lane == 0) s_red[wave] = l;
    __syncthreads();
    if (tid == 0 && row0 + blk * (kEw / kMlpOut) < rows) {
      float s = 0.f;
      for (int w = 0; w < kEw / 64; ++w) s += s_red[w];
      out.loss[row0 / (kEw / kMlpOut) + blk] = s;
    }
    __syncthreads();
  }
  {  // dY's fragments (columns 16..31 zero)
    const int g = wave, l = lane;
    const uint16_t* v = s_dy + (8 * g + 4 * (l >> 5)) * kPitchY + (l & 15);
    *(uint2*)(out.dY + ((size_t)(step0 + g) * 64 + l) * 4) =
        (l & 31) < kMlpOut ? make_uint2(v[0] | (uint32_t)v[kPitchY] << 16, v[2 * kPitchY] | (uint32_t)v[3 * kPitchY] << 16)
                           : make_uint2(0, 0);
  }
  // hidden layers backward: dA = dZ_next W^T, dZ = dA SiLU'(Z)
  auto backward = [&](int l, const float16_t acc) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float d[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d[i] = acc[4 * g + i] * dsilu(z[l][4 * g + i]);
        if (row0 + 8 * g + 4 * h + i >= rows) d[i] = 0.f;
      }
      *(float4*)(out.dZf[l] + (size_t)col * (8 * steps) + row0 + 8 * g + 4 * h) = make_float4(d[0], d[1], d[2], d[3]);
      store_rows(d, l > 0 ? s_a[l & 1] + (8 * g + 4 * h) * kPitchH + col : nullptr, kPitchH,
                 out.dZ[l] + ((size_t)(wave * steps + step0 + g) * 64 + lane) * 4);
    }
    __syncthreads();
  };
  backward(2, tile_product(s_dy, kPitchY, v4, lane));
  const auto v2 = load_frags<kMlpHidden / 8>(wfrag + (FragLayout::b2 + wave * (kMlpHidden / 8)) * 256, lane);
  backward(1, tile_product(s_a[0], kPitchH, v3, lane));
  backward(0, tile_product(s_a[1], kPitchH, v2, lane));
}

// Weight gradients: 60 tiles (24 of W1, 16 of W2 and of W3, 4 of W4) times the splits of the rows, one wavefront each:
// split z sums rows [z kc, min(rows, (z + 1) kc)) into partial + z MlpLayout::total (the sum over the splits follows in a
// fixed order).  The first workgroups sum the bias gradients, a column (of the transposed FP32 dZ and dY) each:
// thread t adds rows t, t + 256, ..., then the wavefronts' lanes and the wavefronts in order.
constexpr int kGradTiles = 60, kBiases = kMlpOut + 3 * kMlpHidden;

__global__ void __launch_bounds__(256) weight_gradient_kernel(const PassOutputs in, int rows, int steps, int kc, int splits,
                                                              float* __restrict__ partial, float* __restrict__ grad) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((int)blockIdx.x < kBiases) {
    __shared__ float s_red[4];
    const int b = (int)blockIdx.x - kMlpOut, l = b / kMlpHidden;
    const float* G = b < 0 ? in.dYf + (size_t)blockIdx.x * (8 * steps) : in.dZf[l] + (size_t)(b % kMlpHidden) * (8 * steps);
    float s = 0.f;
#pragma unroll 8
    for (int r = threadIdx.x; r < rows; r += 256) s += G[r];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if (lane == 0) s_red[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
      float t = 0.f;
      for (int w = 0; w < 4; ++w) t += s_red[w];
      const size_t bias = b < 0 ? MlpLayout::b4 + blockIdx.x
                                : (l == 0 ? MlpLayout::b1 : l == 1 ? MlpLayout::b2 : MlpLayout::b3) + (size_t)(b % kMlpHidden);
      grad[bias] = t;
    }
    return;
  }
  const int item = (blockIdx.x - kBiases) * 4 + wave;
  if (item >= kGradTiles * splits) return;
  const int z = item / kGradTiles;
  int t = item - z * kGradTiles, l, mt, nt;
  if (t < 24) {
    l = 0;
    mt = t / 4;
    nt = t & 3;
  } else if (t < 56) {
    l = 1 + (t - 24) / 16;
    mt = ((t - 24) & 15) / 4;
    nt = t & 3;
  } else {
    l = 3;
    mt = t - 56;
    nt = 0;
  }
  const uint16_t* a = l == 0 ? in.X : in.A[l - 1];
  const uint16_t* b = l == 3 ? in.dY : in.dZ[l];
  const int N = l == 3 ? kMlpOut : kMlpHidden;
  const size_t off = l == 0 ? MlpLayout::W1 : l == 1 ? MlpLayout::W2 : l == 2 ? MlpLayout::W3 : MlpLayout::W4;
  const int k0 = z * kc / 8, k1 = (min(rows, (z + 1) * kc) + 7) / 8;
  const short4_t* fa = (const short4_t*)a + ((size_t)mt * steps + k0) * 64 + lane;
  const short4_t* fb = (const short4_t*)b + ((size_t)nt * steps + k0) * 64 + lane;
  float16_t acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  int k = k0;
  for (; k + 8 <= k1; k += 8, fa += 8 * 64, fb += 8 * 64) {
    short4_t va[8], vb[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      va[q] = fa[q * 64];
      vb[q] = fb[q * 64];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(va[q], vb[q], acc, 0, 0, 0);
  }
  for (; k < k1; ++k, fa += 64, fb += 64) acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(*fa, *fb, acc, 0, 0, 0);
  const int n = 32 * nt + (lane & 31);
  float* c = partial + (size_t)z * MlpLayout::total + off + (size_t)(32 * mt + 4 * (lane >> 5)) * N + n;
  if (n < N)
#pragma unroll
    for (int e = 0; e < 16; ++e) c[(size_t)((e >> 2) * 8 + (e & 3)) * N] = acc[e];
}

__device__ __forceinline__ bool is_bias(long long i) {
  return (i >= (long long)MlpLayout::b1 && i < (long long)MlpLayout::W2) ||
         (i >= (long long)MlpLayout::b2 && i < (long long)MlpLayout::W3) ||
         (i >= (long long)MlpLayout::b3 && i < (long long)MlpLayout::W4) || i >= (long long)MlpLayout::b4;
}

// The gradient of parameter i: a bias's own, a weight's sum over the splits in order.
__device__ __forceinline__ float gradient(const float* __restrict__ partial, int splits, const float* __restrict__ grad,
                                          long long i) {
  if (is_bias(i)) return grad[i];
  float s = 0.f;
#pragma unroll 8
  for (int z = 0; z < splits; ++z) s += partial[(size_t)z * MlpLayout::total + i];
  return s;
}

__global__ void gradient_kernel(const float* __restrict__ partial, int splits, float* __restrict__ grad, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && !is_bias(i)) grad[i] = gradient(partial, splits, grad, i);
}

__global__ void adam_kernel(float* __restrict__ theta, const float* __restrict__ partial, int splits,
                            const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v, long long n, float lr,
                            float b1, float b2, float eps, float c1, float c2, uint16_t* __restrict__ theta_bf,
                            uint16_t* __restrict__ wfrag) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float gi = gradient(partial, splits, g, i);
  float mi = b1 * m[i] + (1.f - b1) * gi;
  float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  float t = theta[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  theta[i] = t;
  store_bf16((size_t)i, f2bf(t), theta_bf, wfrag);
}

__global__ void to_bf16_kernel(const float* __restrict__ in, uint16_t* __restrict__ out, uint16_t* __restrict__ wfrag,
                               long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) store_bf16((size_t)i, f2bf(in[i]), out, wfrag);
}

// ---- fused inference over a scatter grid ---------------------------------------------------------
// Layer 1 is linear in the features and the features of an entry split into those of its 4 grid
// coordinates and those of the 6 atmosphere inputs, which one prediction holds fixed.  So
//   Z1(entry) = b1 + W1_atm^T f(atm) + sum_c W1_c^T f(x_c(entry)),
// and the terms are tabulated once per prediction: row 0 = b1 + W1_atm^T f(atm), then one row of 128
// per value of each grid coordinate (heights, elevations, sun elevations, headings).
__global__ void layer1_tables_kernel(const DevParams P, AtmosphereCode code, const uint16_t* __restrict__ wbf,
                                     const float* __restrict__ theta, float* __restrict__ ztab) {
  const int j = threadIdx.x;  // hidden unit (blockDim.x == kMlpHidden)
  const int row = blockIdx.x;
  // the row's features, each by one thread (every thread all of them: 8 sines and cosines in a row per input, 18 us)
  __shared__ float f[6 * kMlpBands];
  int first = 0, inputs = 1;  // coordinates row: input c of the four
  float x = 0.f;
  if (row == 0) {
    first = 4;
    inputs = 6;
    if (j < 6 * kMlpBands) x = code.v[j / kMlpBands];
  } else {
    int v = row - 1;
    while (v >= P.nS[first]) v -= P.nS[first++];
    x = (float)v / (float)(P.nS[first] - 1);
  }
  if (j < inputs * kMlpBands) f[j] = bf2f(encode_feature(x, j % kMlpBands));
  __syncthreads();
  const uint16_t* W1 = wbf + MlpLayout::W1 + (size_t)(kMlpBands * first) * kMlpHidden + j;
  float acc = row == 0 ? theta[MlpLayout::b1 + j] : 0.f;
  for (int q = 0; q < inputs * kMlpBands; ++q) acc += bf2f(W1[(size_t)q * kMlpHidden]) * f[q];
  ztab[(size_t)blockIdx.x * kMlpHidden + j] = acc;
}

constexpr int kFusedWaves = 4;
constexpr int kLdsRow = kMlpHidden + 8;  // padded row (bf16) of the transposed weights in LDS, 16-byte aligned
constexpr int kFusedLds = (2 * kMlpHidden + 32) * kLdsRow * 2;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// Column order of the transposed weights in LDS: within each block of 16 input units the middle two
// groups of 4 swap places, so that the 8 units a lane half supplies to one K = 16 step (see below) are
// contiguous: one 16-byte LDS read per operand.
__device__ __forceinline__ int lds_column(int k) {
  const int g = (k >> 2) & 3;
  const int gs = g == 1 ? 2 : (g == 2 ? 1 : g);
  return (k & ~15) | (gs << 2) | (k & 3);
}

// bf16 (round to nearest even, v_cvt_pk_bf16_f32) of SiLU of 8 values.
__device__ __forceinline__ bf16x8_t silu_bf16x8(float4 lo, float4 hi) {
  bf16x8_t r;
  r[0] = (__bf16)silu(lo.x);
  r[1] = (__bf16)silu(lo.y);
  r[2] = (__bf16)silu(lo.z);
  r[3] = (__bf16)silu(lo.w);
  r[4] = (__bf16)silu(hi.x);
  r[5] = (__bf16)silu(hi.y);
  r[6] = (__bf16)silu(hi.z);
  r[7] = (__bf16)silu(hi.w);
  return r;
}

__device__ __forceinline__ float4 add5(float4 a, float4 b, float4 c, float4 d, float4 e) {
  return make_float4(a.x + b.x + c.x + d.x + e.x, a.y + b.y + c.y + d.y + e.y, a.z + b.z + c.z + d.z + e.z,
                     a.w + b.w + c.w + d.w + e.w);
}

// One wavefront evaluates 32 entries at a time with the hidden units as the row dimension of every
// product (Z^T = W^T A^T) on v_mfma_f32_32x32x16_bf16.  Its accumulator leaves lane l (half h = l / 32)
// with hidden units 8 g + 4 h + i (g = 0..3, i = 0..3) of each block of 32, for entry l % 32.  A K = 16
// step t over the previous layer's units 16 t .. 16 t + 15 takes from lane half h the 8 units
// 16 t + 4 h + i and 16 t + 8 + 4 h + i (the same register positions in A and B pair up, whatever unit
// they stand for), which that lane already holds: activations never leave the registers.  W2^T, W3^T and
// W4^T (padded to 32 rows, columns in lds_column order) are staged once per workgroup in LDS;
// workgroups loop over the tiles.
struct PredTables {
  float4* p[kMlpOrders];
};

__global__ void __launch_bounds__(64 * kFusedWaves, 2) fused_predict_kernel(
    const DevParams P, const uint16_t* __restrict__ wbf, const float* __restrict__ theta,
    const float* __restrict__ ztab, long long entries, const PredTables out) {
  __shared__ __align__(16) __bf16 lds[kFusedLds / 2];
  __bf16* w2t = lds;
  __bf16* w3t = w2t + kMlpHidden * kLdsRow;
  __bf16* w4t = w3t + kMlpHidden * kLdsRow;
  {
    // 16-byte loads of 8 consecutive weights W[k][n .. n + 7] (all issued before the LDS scatter),
    // transposed into W^T rows; W4 rows 16..31 of W4^T are zero
    static_assert(MlpLayout::W2 % 8 == 0 && MlpLayout::W3 % 8 == 0 && MlpLayout::W4 % 8 == 0, "16-byte rows");
    constexpr int kVec = kMlpHidden * kMlpHidden / 8 / (64 * kFusedWaves);  // loads per thread per matrix
    uint4 v2[kVec], v3[kVec];
    const uint4* s2 = (const uint4*)(wbf + MlpLayout::W2);
    const uint4* s3 = (const uint4*)(wbf + MlpLayout::W3);
    const uint4* s4 = (const uint4*)(wbf + MlpLayout::W4);
#pragma unroll
    for (int q = 0; q < kVec; ++q) {
      v2[q] = s2[threadIdx.x + q * 64 * kFusedWaves];
      v3[q] = s3[threadIdx.x + q * 64 * kFusedWaves];
    }
    const uint4 v4 = s4[threadIdx.x];  // 128 x 16 weights = 256 vectors of 8
#pragma unroll
    for (int q = 0; q < kVec; ++q) {
      const int i = 8 * (threadIdx.x + q * 64 * kFusedWaves);
      const int k = i / kMlpHidden, n = i % kMlpHidden, c = lds_column(k);
      const uint16_t* a2 = (const uint16_t*)&v2[q];
      const uint16_t* a3 = (const uint16_t*)&v3[q];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        w2t[(n + j) * kLdsRow + c] = __builtin_bit_cast(__bf16, a2[j]);
        w3t[(n + j) * kLdsRow + c] = __builtin_bit_cast(__bf16, a3[j]);
      }
    }
    {
      const int i = 8 * threadIdx.x;
      const int k = i / kMlpOut, n = i % kMlpOut, c = lds_column(k);
      const uint16_t* a4 = (const uint16_t*)&v4;
#pragma unroll
      for (int j = 0; j < 8; ++j) w4t[(n + j) * kLdsRow + c] = __builtin_bit_cast(__bf16, a4[j]);
    }
    for (int i = threadIdx.x; i < (32 - kMlpOut) * kMlpHidden; i += blockDim.x)
      w4t[(kMlpOut + i / kMlpHidden) * kLdsRow + i % kMlpHidden] = __builtin_bit_cast(__bf16, (uint16_t)0);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const float* b2 = theta + MlpLayout::b2;
  const float* b3 = theta + MlpLayout::b3;
  const float* b4 = theta + MlpLayout::b4;
  const long long tiles = (entries + 31) / 32;
  for (long long t = (long long)blockIdx.x * kFusedWaves + wave; t < tiles; t += (long long)gridDim.x * kFusedWaves) {
    const long long e = t * 32 + r;
    const unsigned ec = (unsigned)(e < entries ? e : entries - 1);  // < 2^31: the host caps the grid
    const int ia = (int)(ec % (unsigned)NA);
    unsigned q = ec / (unsigned)NA;
    const int is = (int)(q % (unsigned)NL);
    q /= (unsigned)NL;
    const int ie = (int)(q % (unsigned)NE);
    const int ih = (int)(q / (unsigned)NE);
    const float4* z0 = (const float4*)ztab;
    const float4* zh = (const float4*)(ztab + (size_t)(1 + ih) * kMlpHidden);
    const float4* ze = (const float4*)(ztab + (size_t)(1 + NH + ie) * kMlpHidden);
    const float4* zs = (const float4*)(ztab + (size_t)(1 + NH + NE + is) * kMlpHidden);
    const float4* za = (const float4*)(ztab + (size_t)(1 + NH + NE + NL + ia) * kMlpHidden);
    bf16x8_t b[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int lo = 4 * s + h, hi = 4 * s + 2 + h;  // float4 index of units 16 s + 4 h and 16 s + 8 + 4 h
      b[s] = silu_bf16x8(add5(z0[lo], zh[lo], ze[lo], zs[lo], za[lo]), add5(z0[hi], zh[hi], ze[hi], zs[hi], za[hi]));
    }
#pragma unroll 1
    for (int layer = 0; layer < 2; ++layer) {
      const __bf16* wt = layer ? w3t : w2t;
      const float* bias = layer ? b3 : b2;
      float16_t acc[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int x = 0; x < 16; ++x) acc[mt][x] = 0.f;
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
          const bf16x8_t a = *(const bf16x8_t*)(wt + (32 * mt + r) * kLdsRow + 16 * s + 8 * h);
          acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[s], acc[mt], 0, 0, 0);
        }
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int mt = s >> 1, g = 2 * (s & 1);
        const float4 bl = *(const float4*)(bias + 32 * mt + 8 * g + 4 * h);
        const float4 bh = *(const float4*)(bias + 32 * mt + 8 * (g + 1) + 4 * h);
        b[s] = silu_bf16x8(make_float4(acc[mt][4 * g] + bl.x, acc[mt][4 * g + 1] + bl.y, acc[mt][4 * g + 2] + bl.z,
                                       acc[mt][4 * g + 3] + bl.w),
                           make_float4(acc[mt][4 * g + 4] + bh.x, acc[mt][4 * g + 5] + bh.y,
                                       acc[mt][4 * g + 6] + bh.z, acc[mt][4 * g + 7] + bh.w));
      }
    }
    float16_t y;
#pragma unroll
    for (int x = 0; x < 16; ++x) y[x] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const bf16x8_t a = *(const bf16x8_t*)(w4t + r * kLdsRow + 16 * s + 8 * h);
      y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[s], y, 0, 0, 0);
    }
    // lane (r, h) holds outputs 4 h + i (y[i]) and 8 + 4 h + i (y[4 + i]) of entry r, i = 0..3
    float o[kMlpOut];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float u = __shfl(y[i], r + 32, 64), v = __shfl(y[4 + i], r + 32, 64);
      o[i] = y[i];
      o[4 + i] = u;
      o[8 + i] = y[4 + i];
      o[12 + i] = v;
    }
    if (h == 0 && e < entries) {
#pragma unroll
      for (int k = 0; k < kMlpOrders; ++k) {
        if (out.p[k]) {
          float v[3];
#pragma unroll
          for (int c = 0; c < 3; ++c) v[c] = fmaxf(expf(o[3 * k + c] + b4[3 * k + c] - kMlpShift) - kMlpEps, 0.f);
          out.p[k][e] = make_float4(v[0], v[1], v[2], 0.f);
        }
      }
    }
  }
}

inline unsigned ew_blocks(long long n) { return (unsigned)((n + kEw - 1) / kEw); }

template <typename T>
hipError_t dalloc(T** p, size_t count) {
  return hipMalloc((void**)p, count * sizeof(T) < 256 ? 256 : count * sizeof(T));
}

}  // namespace

#define SG_TRY(expr)                         \
  do {                                       \
    hipError_t e_ = (expr);                  \
    if (e_ != hipSuccess) return e_;         \
  } while (0)

static hipError_t allocate(Surrogate& s, int batch) {
  const size_t n = MlpLayout::total;
  SG_TRY(dalloc(&s.theta, n));
  SG_TRY(dalloc(&s.theta_bf, n));
  SG_TRY(dalloc(&s.adam_m, n));
  SG_TRY(dalloc(&s.adam_v, n));
  SG_TRY(dalloc(&s.grad, n));
  SG_TRY(dalloc(&s.wfrag, (size_t)kMlpFragments));
  const size_t padded = (size_t)(batch + kRows - 1) / kRows * kRows;
  SG_TRY(dalloc(&s.X, padded * kMlpFeat));
  for (int l = 0; l < 3; ++l) {
    SG_TRY(dalloc(&s.A[l], padded * kMlpHidden));
    SG_TRY(dalloc(&s.dZ[l], padded * kMlpHidden));
    SG_TRY(dalloc(&s.dZf[l], padded * kMlpHidden));
  }
  SG_TRY(dalloc(&s.Y, (size_t)batch * kMlpOut));
  SG_TRY(dalloc(&s.T, (size_t)batch * kMlpOut));
  SG_TRY(dalloc(&s.dY, padded * 32));
  SG_TRY(dalloc(&s.dYf, padded * kMlpOut));
  SG_TRY(dalloc(&s.loss, (size_t)surrogate_loss_parts(batch) * surrogate_loss_slots(batch)));
  SG_TRY(dalloc(&s.partial, (size_t)kMaxSplits * MlpLayout::total));
  s.batch_capacity = batch;
  return hipSuccess;
}

hipError_t surrogate_alloc(Surrogate& s, int batch) {
  surrogate_free(s);
  const hipError_t e = allocate(s, batch);
  if (e != hipSuccess) {
    surrogate_free(s);
    s.batch_capacity = -1;
  }
  return e;
}

void surrogate_free(Surrogate& s) {
  void* ptrs[] = {s.theta, s.theta_bf, s.wfrag, s.adam_m, s.adam_v, s.grad,   s.X,      s.A[0],   s.A[1], s.A[2], s.dZ[0],
                  s.dZ[1], s.dZ[2],    s.dZf[0], s.dZf[1], s.dZf[2], s.Y,    s.T,      s.dY,     s.dYf,  s.loss, s.ztab,
                  s.partial};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  s = Surrogate();
}

hipError_t surrogate_init(Surrogate& s, uint64_t seed, hipStream_t stream) {
  std::vector<float> h(MlpLayout::total, 0.f);
  uint64_t state = seed;
  auto uniform = [&]() {
    state = splitmix64(state);
    return (float)((state >> 11) * (1.0 / 9007199254740992.0));
  };
  auto fill = [&](size_t off, int fan_in, int fan_out, float gain) {
    float a = gain * std::sqrt(6.0f / (float)(fan_in + fan_out));
    for (size_t i = 0; i < (size_t)fan_in * fan_out; ++i) h[off + i] = (2.f * uniform() - 1.f) * a;
  };
  fill(MlpLayout::W1, kMlpFeat, kMlpHidden, 1.f);
  fill(MlpLayout::W2, kMlpHidden, kMlpHidden, 1.f);
  fill(MlpLayout::W3, kMlpHidden, kMlpHidden, 1.f);
  fill(MlpLayout::W4, kMlpHidden, kMlpOut, 0.1f);
  SG_TRY(hipMemcpyAsync(s.theta, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice, stream));
  SG_TRY(hipMemsetAsync(s.adam_m, 0, h.size() * sizeof(float), stream));
  SG_TRY(hipMemsetAsync(s.adam_v, 0, h.size() * sizeof(float), stream));
  SG_TRY(hipMemsetAsync(s.wfrag, 0, kMlpFragments * sizeof(uint16_t), stream));  // columns past the outputs stay zero
  s.adam_step = 0;
  s.trained = false;
  SG_TRY(surrogate_sync_bf16(s, stream));
  return hipStreamSynchronize(stream);
}

hipError_t surrogate_sync_bf16(Surrogate& s, hipStream_t stream) {
  long long n = (long long)MlpLayout::total;
  hipLaunchKernelGGL(to_bf16_kernel, dim3(ew_blocks(n)), dim3(kEw), 0, stream, s.theta, s.theta_bf, s.wfrag, n);
  return hipGetLastError();
}

int surrogate_loss_parts(int rows) { return (rows * kMlpOut + kEw - 1) / kEw; }

int surrogate_loss_slots(int rows) { return std::max(1, std::min(256, (1 << 20) / std::max(1, surrogate_loss_parts(rows)))); }

static hipError_t launch_pass(Surrogate& s, const PassSource& src, int rows, bool backward, int loss_slot, hipStream_t stream) {
  PassOutputs o;
  std::memset(&o, 0, sizeof(o));
  o.X = s.X;
  o.dY = s.dY;
  o.dYf = s.dYf;
  o.Y = src.in ? s.Y : nullptr;
  o.loss = s.loss + (size_t)loss_slot * surrogate_loss_parts(rows);
  for (int l = 0; l < 3; ++l) {
    o.A[l] = s.A[l];
    o.dZ[l] = backward ? s.dZ[l] : nullptr;
    o.dZf[l] = s.dZf[l];
  }
  const unsigned blocks = (unsigned)((rows + kRows - 1) / kRows);
  hipLaunchKernelGGL(pass_kernel, dim3(blocks), dim3(64 * kFragWaves), 0, stream, src, rows, s.wfrag, s.theta, o);
  SG_TRY(hipGetLastError());
  if (!backward) return hipSuccess;
  int kc = (rows + kMaxSplits - 1) / kMaxSplits;
  kc = std::max((kc + 7) / 8 * 8, 64);
  s.splits = (rows + kc - 1) / kc;
  hipLaunchKernelGGL(weight_gradient_kernel, dim3((unsigned)(kBiases + (kGradTiles * s.splits + 3) / 4)), dim3(256), 0,
                     stream, o, rows, (int)blocks * (kRows / 8), kc, s.splits, s.partial, s.grad);
  return hipGetLastError();
}

hipError_t surrogate_eval_rows(Surrogate& s, const float* inputs_dev, int rows, bool backward, hipStream_t stream) {
  PassSource src;
  std::memset(&src, 0, sizeof(src));
  src.in = inputs_dev;
  src.T = backward ? s.T : nullptr;
  SG_TRY(launch_pass(s, src, rows, backward, 0, stream));
  if (!backward) return hipSuccess;
  const long long n = (long long)MlpLayout::total;
  hipLaunchKernelGGL(gradient_kernel, dim3(ew_blocks(n)), dim3(kEw), 0, stream, s.partial, s.splits, s.grad, n);
  return hipGetLastError();
}

hipError_t surrogate_train_rows(Surrogate& s, const DevParams& P, const AtmosphereCode* codes_dev, int natm,
                                const float* targets_dev, uint64_t seed, int step, int rows, int loss_slot, hipStream_t stream) {
  PassSource src;
  std::memset(&src, 0, sizeof(src));
  for (int d = 0; d < 4; ++d) src.P.nS[d] = P.nS[d];
  src.codes = codes_dev;
  src.natm = natm;
  src.targets = targets_dev;
  src.seed = seed;
  src.step = step;
  return launch_pass(s, src, rows, true, loss_slot, stream);
}

hipError_t surrogate_adam(Surrogate& s, float lr, hipStream_t stream) {
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  s.adam_step += 1;
  float c1 = 1.f - std::pow(b1, (float)s.adam_step), c2 = 1.f - std::pow(b2, (float)s.adam_step);
  long long n = (long long)MlpLayout::total;
  hipLaunchKernelGGL(adam_kernel, dim3(ew_blocks(n)), dim3(kEw), 0, stream, s.theta, s.partial, s.splits, s.grad, s.adam_m,
                     s.adam_v, n, lr, b1, b2, eps, c1, c2, s.theta_bf, s.wfrag);
  return hipGetLastError();
}

hipError_t surrogate_init_output_bias(Surrogate& s, const float* targets_dev, long long rows, hipStream_t stream) {
  hipLaunchKernelGGL(target_mean_kernel, dim3(kMlpUsed), dim3(kEw), 0, stream, targets_dev, rows,
                     s.theta + MlpLayout::b4);
  return hipGetLastError();
}

hipError_t surrogate_make_targets(const float4* const* sums, long long entries, float* targets_dev, hipStream_t stream) {
  SumTables st;
  for (int k = 0; k < kMlpOrders; ++k) st.p[k] = sums[k];
  hipLaunchKernelGGL(targets_kernel, dim3(ew_blocks(entries)), dim3(kEw), 0, stream, st, entries, targets_dev);
  return hipGetLastError();
}

hipError_t surrogate_reserve_tables(Surrogate& s, const DevParams& P) {
  const int rows = 1 + P.nS[0] + P.nS[1] + P.nS[2] + P.nS[3];
  if ((size_t)rows * kMlpHidden > s.ztab_capacity) {
    if (s.ztab) SG_TRY(hipFree(s.ztab));
    s.ztab = nullptr;
    s.ztab_capacity = 0;
    SG_TRY(dalloc(&s.ztab, (size_t)rows * kMlpHidden));
    s.ztab_capacity = (size_t)rows * kMlpHidden;
  }
  return hipSuccess;
}

hipError_t surrogate_predict_tables(Surrogate& s, const DevParams& P, const AtmosphereCode& code, float4* const* out,
                                    hipStream_t stream) {
  const long long entries = (long long)P.nS[0] * P.nS[1] * P.nS[2] * P.nS[3];
  const int rows = 1 + P.nS[0] + P.nS[1] + P.nS[2] + P.nS[3];
  SG_TRY(surrogate_reserve_tables(s, P));
  hipLaunchKernelGGL(layer1_tables_kernel, dim3(rows), dim3(kMlpHidden), 0, stream, P, code, s.theta_bf, s.theta,
                     s.ztab);
  SG_TRY(hipGetLastError());
  const long long tiles = (entries + 31) / 32;
  const long long groups = (tiles + kFusedWaves - 1) / kFusedWaves;
  const unsigned grid = (unsigned)std::min<long long>(groups, 512);  // 2 resident workgroups per CU
  PredTables pt;
  for (int k = 0; k < kMlpOrders; ++k) pt.p[k] = out[k];
  hipLaunchKernelGGL(fused_predict_kernel, dim3(grid), dim3(64 * kFusedWaves), 0, stream, P, s.theta_bf,
                     s.theta, s.ztab, entries, pt);
  return hipGetLastError();
}

AtmosphereCode atmosphere_code(const double* rayleigh_base, double rayleigh_scale, double mie_base, double mie_scale,
                               double mie_g, double albedo) {
  auto unit = [](double v, double lo, double hi) { return (float)std::fmin(std::fmax((v - lo) / (hi - lo), 0.0), 1.0); };
  AtmosphereCode c;
  c.v[0] = unit(rayleigh_scale, 6000.0, 10000.0);
  c.v[1] = unit(rayleigh_base[0] / 5.8e-6, 0.5, 2.0);
  c.v[2] = unit(mie_scale, 800.0, 2000.0);
  c.v[3] = unit(mie_base, 5e-6, 5e-5);
  c.v[4] = unit(mie_g, 0.6, 0.85);
  c.v[5] = unit(albedo, 0.1, 0.5);
  return c;
}

}  // namespace sfsim
