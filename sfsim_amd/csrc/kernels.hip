// HIP kernels (gfx950) of the atmosphere lookup-table precompute.
//
// Mapping: one table entry per lane.  The 4D kernels run one workgroup per view ray
// (height index, elevation index) of the scatter grid, in XCD-aware order: the ray geometry, the
// per-sample altitudes and the view-ray transmittance T(x, p_i) depend only on the ray, so they are
// computed once per build (ray_geometry_kernel) and every lane (sun-elevation, heading entry) of that
// ray reuses them.  Quadratures follow the reference (midpoint nodes of ray.clj:19-30, latitude rings
// of sphere.clj:62-105, O(n^2) transmittance of atmosphere.clj:192-200); only loop-invariant work is
// shared, and single scattering reads each sample's sun optical depth from a table of the same node
// sums (sun_depth_kernel).  Geometry (intersections, the sun direction at each sample) is FP64; the
// extinction sums along rays are FP32 with compensated accumulation, switching to FP64 for segments
// whose lowest point is interior and below DevParams::graze_height.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>

#include "kernels.hpp"

namespace sfsim {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
// min(floor(x), hi) for a coordinate already clamped to x >= 0, as one med3 (fminf would quiet a
// signalling NaN in hi on every call)
__device__ __forceinline__ float lower_cell(float x, float hi) { return __builtin_amdgcn_fmed3f(floorf(x), hi, 0.0f); }

// top_exit_distance (geometry.hpp) for a point inside the atmosphere (h <= H), branch-free, with the
// FP64 square root and reciprocal from the FP32 hardware estimates refined by one Newton step each
// (relative error ~1e-14, against ~1e-16 for the correctly rounded library sequences that cost several
// times as many instructions).  The discriminant pd^2 + (Rt^2 - r^2) lies in [0, 1e14]; it is clamped
// below at 1e-30 (an exit distance under 1e-14 m in place of the zero it stands for) so that the FP32
// estimates stay in their normal range.
__device__ __forceinline__ double sun_exit_distance(const Geo& g, double h, double pd) {
  const double c = (g.H - h) * (2.0 * g.R + g.H + h);
  const double disc = fmax(fma(pd, pd, c), 1e-30);
  double y = (double)__builtin_amdgcn_rsqf((float)disc);
  y = y * fma(-0.5 * disc * y, y, 1.5);
  const double l2 = disc * y;
  double z = (double)__builtin_amdgcn_rcpf((float)(pd + l2));
  z = z * fma(-(pd + l2), z, 2.0);
  return pd > 0.0 ? c * z : l2 - pd;
}

__device__ __forceinline__ void kahan_add(float& sum, float& comp, float x) {
  float y = x - comp;
  float t = sum + y;
  comp = (t - sum) - y;
  sum = t;
}

// atmosphere.clj:56-61 in FP32
__device__ __forceinline__ float phase_f(float g, float mu) {
  float g2 = g * g;
  float x = (1.0f + g2) - 2.0f * g * mu;
  return (3.0f * (1.0f - g2) * (1.0f + mu * mu)) / (8.0f * 3.14159265358979f * (2.0f + g2) * (x * sqrtf(x)));
}

// Altitude along a ray, centred on the segment's lowest point.  With u(t) = r(t)^2 - R^2 =
// h0 (2R + h0) + t (2 pd0 + t) and any shift t = s + ts:  u = u(ts) + s (b' + s), b' = 2 pd0 + 2 ts.
// Taking ts = clamp(-pd0, 0, D) (the point of the segment closest to the planet centre) leaves no
// cancellation: near ts, where the density is largest, u ~ u(ts) is exact, and elsewhere s and
// b' + s have the same sign.  h = u / (R + sqrt(R^2 + u)).
struct Segment {
  float c0, b, s0, dt;  // FP32 node constants in units of R: x_j = c0 + s_j (b + s_j), s_j = j dt + s0
  double c0d, bd, s0d, dtd;  // the same in metres (u_j = c0d + s_j (bd + s_j)) for the FP64 sums
  bool graze;           // lowest point interior and below the FP64 altitude threshold
};

// The midpoint nodes of a segment of length D in P.ray_steps steps (every segment of the path has that many).
__device__ __forceinline__ Segment make_segment(const DevParams& P, double h0, double pd0, double D) {
  Segment g;
  double ts = fmin(fmax(-pd0, 0.0), D);
  g.c0d = h0 * (2.0 * P.g.R + h0) + ts * (2.0 * pd0 + ts);
  g.bd = 2.0 * pd0 + 2.0 * ts;
  g.dtd = D * P.inv_steps;
  g.s0d = 0.5 * g.dtd - ts;
  g.c0 = (float)(g.c0d * P.inv_R * P.inv_R);
  g.b = (float)(g.bd * P.inv_R);
  g.s0 = (float)(g.s0d * P.inv_R);
  g.dt = (float)(g.dtd * P.inv_R);
  g.graze = (-pd0 > 0.0) && (-pd0 < D) && (g.c0d < P.graze_u);
  return g;
}

// A uniform value held in a vector register.  A multiply-add of vector registers alone issues every 2 clocks
// beside another wavefront's instruction, one that reads a scalar register every 4.
__device__ __forceinline__ float in_vgpr(float x) {
  asm("" : "+v"(x));
  return x;
}

// A value that is the same in all lanes, in scalar registers.
__device__ __forceinline__ float uniform(float x) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}
__device__ __forceinline__ double uniform(double x) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)), __builtin_amdgcn_readfirstlane(__double2loint(x)));
}

// Sums over the n midpoint nodes of exp(-h / H_mie) and exp(-h / H_rayleigh) with FP32 altitudes;
// 8-node partial sums, Kahan-compensated across them.  Node j sits at s_j = s0 + j dt (units of R,
// measured from the segment's lowest point), x_j = c0 + s_j (b + s_j) = (r_j^2 - R^2) / R^2, and the
// Mie exponent log2(exp(-h_j / H_mie)) is x_j times a polynomial of degree DEG in x_j
// (DevParams::alt_poly, alt_deg), so a node costs DEG + 3 FMAs, two multiplies, an add and the two
// exponentials.
template <int DEG>
__device__ float2 density_sums_f32_deg(const DevParams& P, const Segment& g, int n) {
  const float a0 = in_vgpr(P.alt_poly[0]), a1 = in_vgpr(P.alt_poly[1]), a2 = in_vgpr(P.alt_poly[2]), a3 = in_vgpr(P.alt_poly[3]);
  const float rho = in_vgpr(P.ray_over_mie);
  auto exponent = [&](float x) {
    const float p = DEG == 3 ? fmaf(fmaf(fmaf(a3, x, a2), x, a1), x, a0) : fmaf(fmaf(a2, x, a1), x, a0);
    return x * p;
  };
  float sm = 0.f, sr = 0.f, cm = 0.f, cr = 0.f;
  int j = 0;
  for (; j + 8 <= n; j += 8) {
    const float base = fmaf((float)j, g.dt, g.s0);
    float m[8], r[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float s = fmaf((float)q, g.dt, base);
      m[q] = exponent(fmaf(s, s + g.b, g.c0));
      r[q] = m[q] * rho;
    }
    __builtin_amdgcn_sched_barrier(0);  // 16 exponentials in a row: between them the additions would not issue in pairs
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      m[q] = fexp2(m[q]);
      r[q] = fexp2(r[q]);
    }
    __builtin_amdgcn_sched_barrier(0);
    float pm = m[0], pr = r[0];
#pragma unroll
    for (int q = 1; q < 8; ++q) {
      pm += m[q];
      pr += r[q];
    }
    kahan_add(sm, cm, pm);
    kahan_add(sr, cr, pr);
  }
  if (j < n) {
    float pm = 0.f, pr = 0.f;
    for (; j < n; ++j) {
      const float s = fmaf((float)j, g.dt, g.s0);
      const float em = exponent(fmaf(s, s + g.b, g.c0));
      pm += fexp2(em);
      pr += fexp2(em * rho);
    }
    kahan_add(sm, cm, pm);
    kahan_add(sr, cr, pr);
  }
  return make_float2(sm, sr);
}

__device__ __forceinline__ float2 density_sums_f32(const DevParams& P, const Segment& g, int n) {
  return P.alt_deg == 2 ? density_sums_f32_deg<2>(P, g, n) : density_sums_f32_deg<3>(P, g, n);
}

// Same sums with FP64 node positions, altitude exponents and accumulation (near-horizon and grazing
// segments): x_j = u_j / R^2 from the metre-valued constants and the FP64 cubic of DevParams; the
// exponentials are FP32 (their argument is rounded to FP32, a relative 6e-8).
__device__ double2 density_sums_f64(const DevParams& P, const Segment& g, int n) {
  const double inv_R2 = P.inv_R * P.inv_R;
  const double a0 = P.alt_poly_d[0], a1 = P.alt_poly_d[1], a2 = P.alt_poly_d[2], a3 = P.alt_poly_d[3];
  const float rho = P.ray_over_mie;
  double sm = 0.0, sr = 0.0;
  for (int j = 0; j < n; ++j) {
    const double s = fma((double)j, g.dtd, g.s0d);
    const double x = fma(s, s + g.bd, g.c0d) * inv_R2;
    const float em = (float)(x * fma(fma(fma(a3, x, a2), x, a1), x, a0));
    sm += (double)fexp2(em);
    sr += (double)fexp2(em * rho);
  }
  return make_double2(sm, sr);
}

// exp(-(beta_mie * integral of the Mie density + beta_rayleigh * ...)) per channel from the two sums,
// as exp2 of the log2(e)-scaled exponent.
__device__ __forceinline__ float3 transmittance_of(const DevParams& P, float sm, float sr, double D) {
  if (!(D > 0.0)) return make_float3(1.f, 1.f, 1.f);
  return make_float3(fexp2(-fmaf(P.ext_mie_l2[0], sm, P.ext_ray_l2[0] * sr)),
                     fexp2(-fmaf(P.ext_mie_l2[1], sm, P.ext_ray_l2[1] * sr)),
                     fexp2(-fmaf(P.ext_mie_l2[2], sm, P.ext_ray_l2[2] * sr)));
}

__device__ __forceinline__ float3 segment_transmittance_f32(const DevParams& P, const Segment& g, double D, int n) {
  float2 s = density_sums_f32(P, g, n);
  const float dt = (float)g.dtd;
  return transmittance_of(P, s.x * dt, s.y * dt, D);
}

__device__ __forceinline__ float3 segment_transmittance_f64(const DevParams& P, const Segment& g, double D, int n) {
  double2 s = density_sums_f64(P, g, n);
  return transmittance_of(P, (float)(s.x * g.dtd), (float)(s.y * g.dtd), D);
}

// Transmittance of the segment of length D from altitude h0 along a unit direction with
// dot(point, direction) = pd0, n midpoint samples (atmosphere.clj:114-125).  The FP64 variant is
// chosen per wavefront (when any active lane holds a grazing segment) so that the two loops never
// diverge within a wave.
__device__ float3 segment_transmittance(const DevParams& P, double h0, double pd0, double D, int n) {
  Segment g = make_segment(P, h0, pd0, D);
  if (__any(g.graze)) return segment_transmittance_f64(P, g, D, n);
  return segment_transmittance_f32(P, g, D, n);
}

// ------------------------------------------------------------------ multilinear lookups
// interpolate.clj:75-98: per dimension i = clip(c), u = floor(i), v = clip(u + 1), s = i - u.
struct Lerp {
  int i0, i1;
  float s;
};

__device__ __forceinline__ Lerp make_lerp(float c, int N) {
  float i = fminf(fmaxf(c, 0.0f), (float)(N - 1));
  float u = floorf(i);
  Lerp L;
  L.i0 = (int)u;
  L.i1 = min(L.i0 + 1, N - 1);
  L.s = i - u;
  return L;
}

// The two corners of a lerp by index parity: idx[p], w[p] for the corner whose index has parity p
// (i0 with weight 1 - s, i1 with weight s); at the upper edge (i1 == i0, s == 0) the one node carries
// weight 1 and the other parity is empty (idx -1, weight 0).
__device__ __forceinline__ void corner_by_parity(const Lerp& L, int idx[2], float w[2]) {
  const bool odd = (L.i0 & 1) != 0;
  const int other = L.i1 != L.i0 ? L.i1 : -1;
  const float w_other = L.i1 != L.i0 ? L.s : 0.0f, w_lower = 1.0f - L.s;
  idx[0] = odd ? other : L.i0;
  w[0] = odd ? w_other : w_lower;
  idx[1] = odd ? L.i0 : other;
  w[1] = odd ? w_lower : w_other;
}

__device__ __forceinline__ float3 mix3(float3 a, float3 b, float s) {
  float r = 1.0f - s;
  return make_float3(a.x * r + b.x * s, a.y * r + b.y * s, a.z * r + b.z * s);
}

__device__ __forceinline__ float3 ld3(const float4* __restrict__ T, long long i) {
  float4 v = T[i];
  return make_float3(v.x, v.y, v.z);
}

// 2D table [N0][N1]
__device__ __forceinline__ float3 lookup2(const float4* __restrict__ T, int N1, Lerp a, Lerp b) {
  float3 u = mix3(ld3(T, (long long)a.i0 * N1 + b.i0), ld3(T, (long long)a.i0 * N1 + b.i1), b.s);
  float3 v = mix3(ld3(T, (long long)a.i1 * N1 + b.i0), ld3(T, (long long)a.i1 * N1 + b.i1), b.s);
  return mix3(u, v, a.s);
}

// lookup2 when one of the two weights may be exactly zero (a grid coordinate that is an integer):
// mix(u, v, 0) = u exactly, so the row or column that it would mix in is not read.  Same result as
// lookup2, bit for bit.
__device__ __forceinline__ float3 lookup2_skip(const float4* __restrict__ T, int N1, Lerp a, Lerp b) {
  if (a.s == 0.0f) return mix3(ld3(T, (long long)a.i0 * N1 + b.i0), ld3(T, (long long)a.i0 * N1 + b.i1), b.s);
  if (b.s == 0.0f) return mix3(ld3(T, (long long)a.i0 * N1 + b.i0), ld3(T, (long long)a.i1 * N1 + b.i0), a.s);
  return lookup2(T, N1, a, b);
}

// 4D table [N0][N1][N2][N3], nested like interpolate-value (outer dimension mixed last)
__device__ __forceinline__ float3 lookup4(const float4* __restrict__ T, int N1, int N2, int N3, Lerp a, Lerp b, Lerp c,
                                          Lerp d) {
  float3 r[2];
#pragma unroll
  for (int ia = 0; ia < 2; ++ia) {
    long long ba = (long long)(ia ? a.i1 : a.i0) * N1;
    float3 rb[2];
#pragma unroll
    for (int ib = 0; ib < 2; ++ib) {
      long long bb = (ba + (ib ? b.i1 : b.i0)) * N2;
      long long c0 = (bb + c.i0) * N3, c1 = (bb + c.i1) * N3;
      float3 u = mix3(ld3(T, c0 + d.i0), ld3(T, c0 + d.i1), d.s);
      float3 v = mix3(ld3(T, c1 + d.i0), ld3(T, c1 + d.i1), d.s);
      rb[ib] = mix3(u, v, c.s);
    }
    r[ia] = mix3(rb[0], rb[1], b.s);
  }
  return mix3(r[0], r[1], a.s);
}

// lookup4 of the texels ld(i) without the reads that a zero weight would mix in: mix3(u, v, 0) is u
// exactly, so each dimension whose weight is zero reads one side only.  Same operations in the same order
// as lookup4 where they are not skipped, so the same result bit for bit.
template <class Ld>
__device__ __forceinline__ float3 lookup4_skip(Ld ld, int N1, int N2, int N3, Lerp a, Lerp b, Lerp c, Lerp d) {
  auto row = [&](int i, int j, int k) {
    const long long base = (((long long)i * N1 + j) * N2 + k) * N3;
    const float3 u = ld(base + d.i0);
    return d.s == 0.0f ? u : mix3(u, ld(base + d.i1), d.s);
  };
  auto cell = [&](int i, int j) {
    const float3 u = row(i, j, c.i0);
    return c.s == 0.0f ? u : mix3(u, row(i, j, c.i1), c.s);
  };
  auto side = [&](int i) {
    const float3 u = cell(i, b.i0);
    return b.s == 0.0f ? u : mix3(u, cell(i, b.i1), b.s);
  };
  const float3 r0 = side(a.i0);
  return a.s == 0.0f ? r0 : mix3(r0, side(a.i1), a.s);
}

__device__ __forceinline__ void count(WorkCounters* wc, unsigned long long single, unsigned long long samples,
                                      unsigned long long l4, unsigned long long l2) {
  if (wc) {
    if (single) atomicAdd(&wc->single_samples, single);
    if (samples) atomicAdd(&wc->samples, samples);
    if (l4) atomicAdd(&wc->lookups4, l4);
    if (l2) atomicAdd(&wc->lookups2, l2);
  }
}

// XCD-aware order of the view rays: workgroups are dispatched to the 8 XCDs round robin (workgroup b
// to XCD b mod 8), each with its own L2.  Giving XCD x the contiguous range of rays
// [x rays / 8, (x + 1) rays / 8) (4 of 32 heights at the full workload) keeps the tables that a height
// range reads (dJ cells, dS rows, sun-table rows) in fewer L2s.  A bijection when rays is a
// multiple of 8; identity otherwise.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_ray(int b, int rays) {
  if (rays % kXcds != 0) return b;
  return (b % kXcds) * (rays / kXcds) + b / kXcds;
}

// ------------------------------------------------------------------------------ kernels
// T table: atmosphere_lut.clj:74 over transmittance-space (atmosphere.clj:291-319)
__device__ __forceinline__ void transmittance_body(const DevParams& P, float4* __restrict__ out,
                                                               WorkCounters* wc, unsigned blk) {
  const int NH = P.nT[0], NE = P.nT[1];
  int idx = blk * blockDim.x + threadIdx.x;
  if (idx >= NH * NE) return;
  int ih = idx / NE, ie = idx - ih * NE;
  double r0 = index_to_radius(P.g, NH, ih), h0 = index_to_altitude(P.g, NH, ih);
  double se, ce;
  bool above;
  index_to_elevation(P.g, NE, r0, ie, se, ce, above);
  double pd0 = r0 * se;
  double D = above ? top_exit_distance(P.g, h0, pd0) : ground_distance(P.g, h0, pd0);
  float3 T = segment_transmittance(P, h0, pd0, D, P.ray_steps);
  out[idx] = make_float4(T.x, T.y, T.z, 0.f);
  count(wc, 0, P.ray_steps, 0, 0);
}

__global__ void __launch_bounds__(kBlock) transmittance_kernel(const DevParams P, float4* __restrict__ out,
                                                               WorkCounters* wc) {
  transmittance_body(P, out, wc, blockIdx.x);
}

// dE0 table: surface-radiance-base (atmosphere.clj:131-137) over surface-radiance-space
__device__ __forceinline__ void surface_radiance_base_body(const DevParams& P, float4* __restrict__ out,
                                                                       WorkCounters* wc, unsigned blk) {
  const int NH = P.nE[0], NL = P.nE[1];
  int idx = blk * blockDim.x + threadIdx.x;
  if (idx >= NH * NL) return;
  int ih = idx / NL, il = idx - ih * NL;
  double r0 = index_to_radius(P.g, NH, ih), h0 = index_to_altitude(P.g, NH, ih);
  double s = index_to_sin_sun_elevation(NL, il);
  double pd0 = r0 * s;  // dot(x, l) with l = (s, c, 0)
  double D = top_exit_distance(P.g, h0, pd0);
  float3 T = segment_transmittance(P, h0, pd0, D, P.ray_steps);
  float cosf_ = (float)fmax(0.0, s);  // max(0, normal . l), normal = (1 0 0)
  out[idx] = make_float4(T.x * P.intensity[0] * cosf_, T.y * P.intensity[1] * cosf_, T.z * P.intensity[2] * cosf_, 0.f);
  count(wc, 0, P.ray_steps, 0, 0);
}

__global__ void __launch_bounds__(kBlock) surface_radiance_base_kernel(const DevParams P, float4* __restrict__ out,
                                                                       WorkCounters* wc) {
  surface_radiance_base_body(P, out, wc, blockIdx.x);
}

// Per-ray setup shared by the 4D kernels: grid point x = (r0 0 0), view v = (se ce 0), ray length D.
struct Ray {
  double r0, h0, se, ce, pd0, D;
  bool above;
};

__device__ __forceinline__ Ray make_ray(const DevParams& P, int ih, int ie) {
  Ray r;
  r.r0 = index_to_radius(P.g, P.nS[0], ih);
  r.h0 = index_to_altitude(P.g, P.nS[0], ih);
  index_to_elevation(P.g, P.nS[1], r.r0, ie, r.se, r.ce, r.above);
  r.pd0 = r.r0 * r.se;
  r.D = r.above ? top_exit_distance(P.g, r.h0, r.pd0) : ground_distance(P.g, r.h0, r.pd0);
  return r;
}

// R1 (Rayleigh with phase) and M1 (Mie strength) in one pass: atmosphere_lut.clj:70-78,
// atmosphere.clj:154-200.  One workgroup per (view ray, group of 64 (sun elevation, heading) entries); groups of high
// sun elevation (most samples lit) are launched first so that the light groups fill the end of the grid.  The ray's
// samples are processed in chunks of kSSChunk: each thread marks the samples of its quarter of the chunk where its
// entry's sun is above the horizon, the workgroup compacts the lit (entry, sample) pairs into an LDS list, and its
// wavefronts take 64 items of it at a time, the FP64 ones first, so lanes never idle on unlit samples; each entry then
// adds its results in sample order (deterministic sums).
//
// VALU issue bounds it: per item ray_steps nodes of two exponentials (8 clocks each) and ten further instructions, at
// 60 clocks a node.  With one wavefront per group (32 x 64 x 32 x 8 entries: 32 per CU) the whole grid was resident at
// once, and the CUs idled for 35% of the launch while the ones that held the most lit groups finished; four wavefronts
// per group leave a quarter of the groups resident and the rest to whichever CU is free: 1080 us -> 798, and 760 with the
// node loop's coefficients in vector registers and its exponentials in a row.
constexpr int kSSEntries = 64;
constexpr int kSSWaves = 4;
constexpr int kSSChunk = 16;

// LDS of a workgroup for n samples.
inline size_t single_scatter_shared_bytes(int n) {
  return (size_t)n * (2 * sizeof(double) + sizeof(float4)) + sizeof(float) * (size_t)((n + 3) & ~3) +
         (3 * sizeof(float) + sizeof(unsigned short)) * kSSEntries * kSSChunk + 2 * sizeof(double) * kSSEntries +
         kSSWaves * kSSEntries * sizeof(unsigned) + (2 * kSSWaves + 1) * sizeof(int);
}

__device__ __forceinline__ int wave_exclusive_scan(int v, int lane) {
  int x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  return x - v;
}

__global__ void __launch_bounds__(kSSEntries* kSSWaves) single_scatter_kernel(const DevParams P, float4* __restrict__ R1,
                                                                              float4* __restrict__ M1, WorkCounters* wc) {
  extern __shared__ unsigned char s_raw[];
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const int NLA = NL * NA;
  const int n = P.ray_steps;
  constexpr int kItems = kSSEntries * kSSChunk, kQuarter = kSSChunk / kSSWaves;
  double* s_t = (double*)s_raw;                            // [n] sample distance along the ray
  double* s_h = s_t + n;                                   // [n] sample altitude
  double* s_xl = s_h + n;                                  // [64] dot(x, l) of each entry
  double* s_vl = s_xl + kSSEntries;                        // [64] dot(v, l)
  float4* s_w = (float4*)(s_vl + kSSEntries);              // [n] T(x, p_i) rgb, w: exp(-h_i / H_mie)
  float* s_bray = (float*)(s_w + n);                       // [n] exp(-h_i / H_rayleigh)
  float* s_res = s_bray + ((n + 3) & ~3);                  // [3][chunk sample][entry] sun transmittance (r, g, b planes)
  unsigned* s_mask = (unsigned*)(s_res + 3 * kItems);      // [quarter][entry] lit samples of the chunk
  int* s_total = (int*)(s_mask + kSSWaves * kSSEntries);   // [2][quarter] items listed, FP64 and FP32
  int* s_next = s_total + 2 * kSSWaves;                    // the next 64 items
  unsigned short* s_item = (unsigned short*)(s_next + 1);  // chunk sample * 64 + entry

  const int rays = NH * NE;
  const int groups = (NLA + kSSEntries - 1) / kSSEntries;
  const unsigned block = blockIdx.y * gridDim.x + blockIdx.x;  // (a launch's x holds less than 2^32 threads)
  if (block >= (unsigned)groups * rays) return;
  const int group = groups - 1 - (int)(block / rays);
  const int rayid = (int)block - (groups - 1 - group) * rays;
  const int ih = rayid / NE, ie = rayid - ih * NE;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Ray ray = make_ray(P, ih, ie);
  const double dt = ray.D / n;
  unsigned long long samples = 0, view = 0;
  for (int i = threadIdx.x; i < n; i += kSSEntries * kSSWaves) {
    double t = (i + 0.5) * dt;
    double h = altitude_along(P.g, ray.h0, ray.pd0, t);
    s_t[i] = t;
    s_h[i] = h;
    float3 T = segment_transmittance(P, ray.h0, ray.pd0, t, n);
    s_w[i] = make_float4(T.x, T.y, T.z, (float)exp(-h * P.inv_scale_mie));
    s_bray[i] = (float)exp(-h * P.inv_scale_ray);
    view += n;
  }
  const int k = group * kSSEntries + lane;
  const bool valid = k < NLA;
  double vl = 0.0, xl = 0.0;
  if (valid) {
    int is = k / NA, ia = k - is * NA;
    double sin_s = index_to_sin_sun_elevation(NL, is);
    double l0, l1, l2;
    index_to_sun_direction(NA, ray.se, ray.ce, sin_s, ia, l0, l1, l2);
    vl = ray.se * l0 + ray.ce * l1;
    xl = ray.r0 * l0;
  }
  s_xl[lane] = xl;  // every wavefront the same
  s_vl[lane] = vl;
  __syncthreads();
  float3 accR = make_float3(0.f, 0.f, 0.f), accM = make_float3(0.f, 0.f, 0.f);
  for (int i0 = 0; i0 < n; i0 += kSSChunk) {
    const int cn = min(kSSChunk, n - i0);
    // lit samples (atmosphere.clj:154-160), split by the optical-depth path their sun segment takes:
    // FP64 when its lowest point (at distance -dot(p_i, l) when that is positive) lies below
    // graze_height, FP32 otherwise
    unsigned m32 = 0, m64 = 0;
    if (valid)
      for (int c = wave * kQuarter; c < min(cn, (wave + 1) * kQuarter); ++c) {
        const int i = i0 + c;
        const double h = s_h[i], pl = xl + s_t[i] * vl;
        if (is_above_horizon(P.g, h, pl)) {
          if (pl < 0.0 && h * (2.0 * P.g.R + h) - pl * pl < P.graze_u)
            m64 |= 1u << c;
          else
            m32 |= 1u << c;
        }
      }
    const int c32 = __popc(m32), c64 = __popc(m64);
    int o32 = wave_exclusive_scan(c32, lane), o64 = wave_exclusive_scan(c64, lane);
    s_mask[threadIdx.x] = m32 | m64;
    if (lane == 63) {
      s_total[wave] = o64 + c64;
      s_total[kSSWaves + wave] = o32 + c32;
    }
    if (threadIdx.x == 0) *s_next = 0;
    __syncthreads();
    int t32 = 0, t64 = 0;
#pragma unroll
    for (int w = 0; w < kSSWaves; ++w) {
      const int a = s_total[w], b = s_total[kSSWaves + w];
      if (w < wave) {
        o64 += a;
        o32 += b;
      }
      t64 += a;
      t32 += b;
    }
    for (unsigned m = m64; m; m &= m - 1) s_item[o64++] = (unsigned short)((__ffs(m) - 1) * kSSEntries + lane);
    for (unsigned m = m32; m; m &= m - 1) s_item[t64 + o32++] = (unsigned short)((__ffs(m) - 1) * kSSEntries + lane);
    __syncthreads();
    // sun transmittance T(p_i, l) of every listed item; the two loops never share a wavefront
    const int u64 = (t64 + 63) / 64, units = u64 + (t32 + 63) / 64;
    for (;;) {
      int u = 0;
      if (lane == 0) u = atomicAdd(s_next, 1);
      u = __builtin_amdgcn_readfirstlane(u);
      if (u >= units) break;
      const bool wide = u < u64;
      const int it = wide ? u * 64 + lane : t64 + (u - u64) * 64 + lane;
      if (it < (wide ? t64 : t64 + t32)) {
        const unsigned item = s_item[it], owner = item & (kSSEntries - 1);
        const int i = i0 + (int)(item / kSSEntries);
        const double h = s_h[i];
        const double pl = s_xl[owner] + s_t[i] * s_vl[owner];  // dot(p_i, l)
        const double Ds = sun_exit_distance(P.g, h, pl);
        const Segment g = make_segment(P, h, pl, Ds);
        const float3 Ts = wide ? segment_transmittance_f64(P, g, Ds, n) : segment_transmittance_f32(P, g, Ds, n);
        s_res[item] = Ts.x;
        s_res[item + kItems] = Ts.y;
        s_res[item + 2 * kItems] = Ts.z;
      }
    }
    samples += (unsigned long long)(c32 + c64) * n;
    __syncthreads();
    if (wave == 0) {
      // each entry adds its lit samples in sample order (deterministic sums)
      unsigned m = 0;
#pragma unroll
      for (int w = 0; w < kSSWaves; ++w) m |= s_mask[w * kSSEntries + lane];
      for (; m; m &= m - 1) {
        const int c = __ffs(m) - 1, idx = c * kSSEntries + lane;
        const float3 Ts = make_float3(s_res[idx], s_res[idx + kItems], s_res[idx + 2 * kItems]);
        const float4 w = s_w[i0 + c];
        const float br = s_bray[i0 + c];
        const float3 t3 = make_float3(w.x * Ts.x, w.y * Ts.y, w.z * Ts.z);
        accR.x += t3.x * br; accR.y += t3.y * br; accR.z += t3.z * br;
        accM.x += t3.x * w.w; accM.y += t3.y * w.w; accM.z += t3.z * w.w;
      }
    }
    __syncthreads();
  }
  if (valid && wave == 0) {
    const long long o = (long long)rayid * NLA + k;
    float a = (float)dt;
    float pr = phase_f(P.g_ray, (float)vl) * a;
    R1[o] = make_float4(accR.x * P.sca_ray[0] * P.intensity[0] * pr, accR.y * P.sca_ray[1] * P.intensity[1] * pr,
                        accR.z * P.sca_ray[2] * P.intensity[2] * pr, 0.f);
    M1[o] = make_float4(accM.x * P.sca_mie[0] * P.intensity[0] * a, accM.y * P.sca_mie[1] * P.intensity[1] * a,
                        accM.z * P.sca_mie[2] * P.intensity[2] * a, 0.f);
  }
  count(wc, samples, samples + view, 0, 0);
}

// ------------------------------------------------------------ tabulated sun optical depths
// The sun segment of a sample p (atmosphere.clj:154-160: transmittance from p toward l to the top of
// the atmosphere, ray_steps midpoint nodes) depends on p and l only through r = |p| and pl = dot(p, l),
// so its two node sums (Mie and Rayleigh density times the node spacing) are functions of two
// variables.  Rows: a = rho / rho_max, rho = sqrt(r^2 - R^2), uniform in the horizon distance (the
// altitude grid is finest at the ground); columns: b = (D - D_min) / (D_max - D_min) for the exit
// distance D, D_min = Rt - r (sun at the zenith) and D_max = rho + rho_max (sun on the horizon), which
// spans every direction in which the sun is above the horizon.  Entries hold log2 of the node sums
// (FP64 for grazing segments, compensated FP32 otherwise); interpolation is bilinear in log2
// (exponential in altitude between grid points).
__device__ __forceinline__ void sun_depth_body(const DevParams& P, unsigned blk) {
  const int rows = P.sun_rows, cols = P.sun_cols;
  const int idx = blk * blockDim.x + threadIdx.x;
  if (idx >= rows * cols) return;
  const int ia = idx / cols, ib = idx - ia * cols;
  const double rho = P.g.rho_max * ia / (rows - 1);
  const double h = rho * rho / (P.g.R + sqrt(P.g.R * P.g.R + rho * rho));
  const double c = (P.g.rho_max - rho) * (P.g.rho_max + rho);  // Rt^2 - r^2
  const double dmin = P.g.H - h, dmax = rho + P.g.rho_max;
  const double D = dmin + (dmax - dmin) * ib / (cols - 1);
  float2 out = make_float2(-256.f, -256.f);  // empty segment (the top of the atmosphere, sun at the zenith)
  if (D > 0.0) {
    const double pl = (c - D * D) / (2.0 * D);  // from D = -pl + sqrt(pl^2 + c)
    const Segment g = make_segment(P, h, pl, D);
    double sm, sr;
    if (__any(g.graze)) {  // the same FP32/FP64 choice as segment_transmittance
      const double2 sum = density_sums_f64(P, g, P.ray_steps);
      sm = sum.x * g.dtd;
      sr = sum.y * g.dtd;
    } else {
      const float2 sum = density_sums_f32(P, g, P.ray_steps);
      sm = (double)sum.x * g.dtd;
      sr = (double)sum.y * g.dtd;
    }
    out = make_float2((float)fmax(log2(sm), -256.0), (float)fmax(log2(sr), -256.0));
  }
  P.sun_depth[idx] = out;
}

__global__ void __launch_bounds__(kBlock) sun_depth_kernel(const DevParams P) {
  sun_depth_body(P, blockIdx.x);
}

// Geometry of every (view ray, sample) pair, one thread each: the sample position, T(x, p_i) over
// ray_steps midpoint nodes, the height and elevation coordinates of the dJ lookup, the terms of the
// sun-elevation coordinate and, with a sun table, the sample's row and exit-distance terms in it.
// Shared by the single-scatter kernel and the ray-scatter launches of all iterations.
__device__ __forceinline__ void ray_geometry_body(const DevParams& P, WorkCounters* wc, unsigned blk) {
  const int n = P.ray_steps, NH = P.nS[0], NE = P.nS[1];
  const long long g = (long long)blk * blockDim.x + threadIdx.x;
  if (g >= (long long)NH * NE * n) return;
  const int rayid = (int)(g / n), i = (int)(g - (long long)rayid * n);
  const int ih = rayid / NE, ie = rayid - ih * NE;
  const Ray ray = make_ray(P, ih, ie);
  const double t = (i + 0.5) * (ray.D / n);
  const double h = altitude_along(P.g, ray.h0, ray.pd0, t), r = P.g.R + h;
  const float3 T = segment_transmittance(P, ray.h0, ray.pd0, t, n);
  const RayGeoView V = ray_geo_view(P);
  const double k3 = -3.0 * 1.4426950408889634;
  V.th[g] = make_double2(t, h);
  V.T[g] = make_float4(T.x, T.y, T.z, (float)exp(-h * P.inv_scale_mie));
  const float hc = (float)altitude_to_index(P.g, NH, h);
  const float ec = (float)elevation_to_index(P.g, NE, r, ray.pd0 + t, ray.above);
  V.rs[g] = make_float4(hc, ec, (float)(k3 / r), (float)(k3 * t / r));
  {  // the fold's dJ nodes by slot: the corner with height parity ph and elevation parity pe goes to slot
     // 2 ph + pe (at the upper edge of the grid, where i1 == i0 and the weight of i1 is zero, the
     // coinciding corners share one slot and the slots of the other parity stay unused)
    const int NLA = P.nS[2] * P.nS[3];
    const Lerp Lh = make_lerp(hc, NH), Le = make_lerp(ec, NE);
    int hs[2], es[2];
    float hw[2], ew[2];
    corner_by_parity(Lh, hs, hw);
    corner_by_parity(Le, es, ew);
    auto off = [&](int ph, int pe) { return hs[ph] < 0 || es[pe] < 0 ? -1 : (hs[ph] * NE + es[pe]) * NLA; };
    auto wt = [&](int ph, int pe) { return hs[ph] < 0 || es[pe] < 0 ? 0.0f : ew[pe] * hw[ph]; };
    V.fold[g] = FoldStep{make_int4(off(0, 0), off(0, 1), off(1, 0), off(1, 1)),
                         make_float4(wt(0, 0), wt(0, 1), wt(1, 0), wt(1, 1))};
  }
  if (P.sun_rows > 0) {
    const int cols = P.sun_cols;
    // clamped like horizon_distance: the sample of a ray that grazes the ground at its tangent point (the
    // middle sample of an odd number of them) has h = 0 up to FP64 rounding, of either sign
    const double rho = sqrt(fmax(0.0, h * (2.0 * P.g.R + h)));
    const double dmin = P.g.H - h, dmax = rho + P.g.rho_max;
    V.ss[g] = make_float4((float)((P.g.H - h) * (2.0 * P.g.R + P.g.H + h)), (float)dmin,
                          (float)((cols - 1) / (dmax - dmin)), (float)exp(-h * P.inv_scale_ray));
    const float x = (float)(rho / P.g.rho_max * (P.sun_rows - 1));
    const float row = fminf(floorf(x), (float)(P.sun_rows - 2));
    V.row[g] = make_float2(x - row, __int_as_float((int)row * cols));
  }
  count(wc, 0, n, 0, 0);
}

__global__ void __launch_bounds__(kBlock) ray_geometry_kernel(const DevParams P, WorkCounters* wc) {
  ray_geometry_body(P, wc, blockIdx.x);
}

// The ray-scatter items of one view ray (DevParams::rs_items), by one workgroup: one per entry whose heading
// coordinate is integral, two (the columns beside it) otherwise, none for an entry with the sun direction of the
// heading before it (clamped to the same one: the same FP64 v . l at the same sun elevation).  In (heading, sun
// elevation) order, so that neighbouring lanes of ray_scatter_kernel read neighbouring rows of a column; with
// several groups of columns counted first and then written group after group.  s_pos: NL x NA words of LDS.
__device__ __forceinline__ void ray_items_body(const DevParams& P, int rayid, unsigned* s_pos) {
  __shared__ int s_count[kMaxRsGroups], s_start[kMaxRsGroups + 1];
  const int NL = P.nS[2], NA = P.nS[3], NLA = NL * NA, groups = P.rs_groups;
  const int capacity = P.rs_slots;
  const long long base = (long long)rayid * NLA;
  const double2* __restrict__ ss = P.sun_ss + base;
  const int lane = threadIdx.x & 63;
  if (threadIdx.x <= kMaxRsGroups) {
    s_start[threadIdx.x] = 0;
    if (threadIdx.x < kMaxRsGroups) s_count[threadIdx.x] = 0;
  }
  __syncthreads();
  for (int pass = groups == 1 ? 1 : 0; pass < 2; ++pass) {
    for (int b = threadIdx.x - lane; b < NLA; b += blockDim.x) {
      const int q = min(b + lane, NLA - 1), a = q / NL, s = q - a * NL, k = s * NA + a;
      const double2 d = ss[k];
      const Lerp L = make_lerp((float)sun_angle_to_index(NA, d.x), NA);
      const bool same = a > 0 && d.x == ss[max(k - 1, 0)].x, own = b + lane < NLA && !same;
      unsigned pos[2] = {0, 0};
      for (int g = 0; g < groups; ++g)
        for (int j = 0; j < 2; ++j) {
          const int col = j ? L.i1 : L.i0;
          const bool want = own && (j == 0 || L.s != 0.0f) && (groups == 1 || col / P.rs_cols == g);
          const unsigned long long mask = __ballot(want);
          if (mask == 0) continue;
          int first = 0;
          if (lane == 0) first = atomicAdd(&s_count[g], __popcll(mask));
          const int idx = __builtin_amdgcn_readfirstlane(first) + __popcll(mask & ((1ull << lane) - 1));
          if (want && pass == 1) {
            P.rs_items[2 * base + s_start[g] + idx] = RsItem{(float)d.x, (float)d.y, ((unsigned)col << 16) | (unsigned)k};
            pos[j] = (unsigned)(g * capacity + min(idx, capacity - 1));  // (rs_split: idx < capacity)
          }
        }
      if (b + lane < NLA && pass == 1) s_pos[k] = same ? 0xffffffffu : (pos[1] << 16) | (pos[0] & 0xffffu);
    }
    __syncthreads();
    if (pass == 0) {
      if (threadIdx.x == 0)
        for (int g = 0; g < groups; ++g) {
          s_start[g + 1] = s_start[g] + s_count[g];
          s_count[g] = 0;
        }
      __syncthreads();
    }
  }
  if ((int)threadIdx.x <= groups)
    P.rs_heads[(long long)rayid * (groups + 1) + threadIdx.x] =
        (int)threadIdx.x < groups ? s_start[threadIdx.x] : s_start[groups - 1] + s_count[groups - 1];
  for (int k = threadIdx.x; k < NLA; k += blockDim.x) {
    unsigned p = s_pos[k];
    for (int q = k; p == 0xffffffffu;) p = s_pos[--q];
    P.rs_entries[base + k] = make_uint2(p, __float_as_uint(make_lerp((float)sun_angle_to_index(NA, ss[k].x), NA).s));
  }
}

__global__ void __launch_bounds__(kBlock) ray_items_kernel(const DevParams P) {
  extern __shared__ unsigned s_pos[];
  ray_items_body(P, (int)blockIdx.x, s_pos);
}

struct __attribute__((aligned(8))) UnalignedFloat4 {
  float x, y, z, w;
  __device__ operator float4() const { return make_float4(x, y, z, w); }
};

// Single scatter with the sun segments' optical depths read from the sun_depth table: one block per
// view ray, one thread per (sun elevation, heading) entry, each adding its lit samples in sample order.
// The ray's samples (t, r^2 - R^2, T(x, p_i), sun-table terms) come from the per-build geometry through LDS.
//
// What bounds it is the table's gathers in L1 (31 accesses per 16-byte read of a wavefront: 0.7 of the clocks at
// 32 x 64 x 32 x 8, 0.9 at 64 x 128 x 64 x 16) and next to them VALU issue, 60 instructions per sample, five exponentials, a
// square root, a reciprocal and six FP64 operations among them.  With the FP64 terms of a sample formed once per ray, a
// 32-bit offset per read, coefficients in vector registers and no lit count unless one is asked for: 87.7 -> 83.6 us,
// 2200 -> 2049 us at the larger grid.
constexpr int kSSTBlock = 256;

template <bool kB>
__global__ void __launch_bounds__(kSSTBlock) single_scatter_table_kernel(
    const DevParams P0, const DevParams* __restrict__ PB, const double2* __restrict__ geo_th,
    const float4* __restrict__ geo_T, const float4* __restrict__ geo_ss, const float2* __restrict__ geo_row,
    float4* __restrict__ R1, float4* __restrict__ M1, int item_blocks, WorkCounters* wc) {
  extern __shared__ unsigned char s_raw[];
  const DevParams& P = params_of<kB>(P0, PB);
  // the rays' ray-scatter items (shared by the atmospheres of a batch) ride in the launch's first workgroups
  if ((int)blockIdx.x < item_blocks) {
    if (!kB || blockIdx.z == 0) ray_items_body(P, (int)blockIdx.x, (unsigned*)s_raw);
    return;
  }
  if constexpr (kB) {  // this atmosphere's tables and ray geometry (offsets of the restrict arguments, whose
                       // loads stay provably unclobbered and uniform: scalar loads)
    geo_th = atm_ptr<kB>(geo_th, P0);
    geo_T = atm_ptr<kB>(geo_T, P0);
    geo_ss = atm_ptr<kB>(geo_ss, P0);
    geo_row = atm_ptr<kB>(geo_row, P0);
    R1 = atm_ptr<kB>(R1, P);
    M1 = atm_ptr<kB>(M1, P);
  }
  const int NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const int NLA = NL * NA;
  const int n = P.ray_steps, cols = P.sun_cols;
  const int rayid = xcd_ray(blockIdx.x - item_blocks, P.nS[0] * NE);
  const int ih = rayid / NE, ie = rayid - ih * NE;
  const Ray ray = make_ray(P, ih, ie);
  const double dt = ray.D / n;
  // this ray's samples from the per-build geometry, staged in LDS
  double2* s_tu = (double2*)s_raw;      // [n] t_i, r_i^2 - R^2
  float4* s_w = (float4*)(s_tu + n);    // [n] T(x, p_i) rgb, w: exp(-h_i / H_mie)
  float4* s_g = s_w + n;                // [n] Rt^2 - r_i^2, D_min, (cols - 1) / (D_max - D_min), exp(-h_i / H_rayleigh)
  float2* s_r = (float2*)(s_g + n);     // [n] sun-table row fraction, byte offset of the row (bits of an unsigned)
  const long long g0 = (long long)rayid * n;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const double2 th = geo_th[g0 + i];
    const float2 r = geo_row[g0 + i];
    s_tu[i] = make_double2(th.x, radius_excess(P.g, th.y));
    s_w[i] = geo_T[g0 + i];
    s_g[i] = geo_ss[g0 + i];
    s_r[i] = make_float2(r.x, __uint_as_float((unsigned)__float_as_int(r.y) * (unsigned)sizeof(float2)));
  }
  __syncthreads();
  // two rows of the table from the sample's on: a uniform base each and one 32-bit byte offset per lane
  const char* __restrict__ row0 = (const char*)P.sun_depth;
  const char* __restrict__ row1 = (const char*)(P.sun_depth + cols);
  const float top = (float)(cols - 1), top_cell = (float)(cols - 2);
  const float em[3] = {in_vgpr(P.ext_mie_l2[0]), in_vgpr(P.ext_mie_l2[1]), in_vgpr(P.ext_mie_l2[2])};
  const float er[3] = {in_vgpr(P.ext_ray_l2[0]), in_vgpr(P.ext_ray_l2[1]), in_vgpr(P.ext_ray_l2[2])};
  unsigned long long lit = 0;
  for (int k = threadIdx.x; k < NLA; k += blockDim.x) {
    // dot(v, l) and dot(x, l) in FP64 from the per-build sun map (the same FP64 evaluation)
    const double2 vx = P.sun_ss[(long long)rayid * NLA + k];
    const double vl = vx.x, xl = vx.y;
    float3 accR = make_float3(0.f, 0.f, 0.f), accM = make_float3(0.f, 0.f, 0.f);
    // branch-free: a lane whose sun is below the horizon (atmosphere.clj:154-160) reads the table at clamped,
    // in-range coordinates and adds exactly zero, so consecutive samples' reads overlap.  (Samples that no lane of
    // the wavefront sees lit, 1-19% of them, cost less than a branch per sample or per pair of samples.)
#pragma unroll 2
    for (int i = 0; i < n; ++i) {
      const double2 tu = s_tu[i];
      const double pl = xl + tu.x * vl;  // dot(p_i, l)
      const bool sun = is_above_horizon_at(tu.y, pl);
      if (wc) lit += sun;
      const float4 gm = s_g[i];
      const float2 rr = s_r[i];
      const float plf = (float)pl;
      const float q = __builtin_amdgcn_sqrtf(fmaf(plf, plf, gm.x));
      const float D = plf > 0.f ? gm.x * __builtin_amdgcn_rcpf(plf + q) : q - plf;
      const float y = __builtin_amdgcn_fmed3f((D - gm.y) * gm.z, 0.f, top);
      const float col = fminf(floorf(y), top_cell);
      const float fy = y - col;
      const unsigned at = __float_as_uint(rr.y) + (unsigned)col * (unsigned)sizeof(float2);
      const float4 lo = *(const UnalignedFloat4*)(row0 + at), hi = *(const UnalignedFloat4*)(row1 + at);  // two columns
      const float lo_m = fmaf(fy, lo.z - lo.x, lo.x), hi_m = fmaf(fy, hi.z - hi.x, hi.x);
      const float lo_r = fmaf(fy, lo.w - lo.y, lo.y), hi_r = fmaf(fy, hi.w - hi.y, hi.y);
      const float sm = fexp2(fmaf(rr.x, hi_m - lo_m, lo_m)), sr = fexp2(fmaf(rr.x, hi_r - lo_r, lo_r));
      const float4 w = s_w[i];
      const float3 t3 = make_float3(w.x * fexp2(-fmaf(em[0], sm, er[0] * sr)), w.y * fexp2(-fmaf(em[1], sm, er[1] * sr)),
                                    w.z * fexp2(-fmaf(em[2], sm, er[2] * sr)));
      const float br = sun ? gm.w : 0.0f, bm = sun ? w.w : 0.0f;
      accR.x += t3.x * br; accR.y += t3.y * br; accR.z += t3.z * br;
      accM.x += t3.x * bm; accM.y += t3.y * bm; accM.z += t3.z * bm;
    }
    const long long o = (long long)rayid * NLA + k;
    const float a = (float)dt;
    const float pr = phase_f(P.g_ray, (float)vl) * a;
    R1[o] = make_float4(accR.x * P.sca_ray[0] * P.intensity[0] * pr, accR.y * P.sca_ray[1] * P.intensity[1] * pr,
                        accR.z * P.sca_ray[2] * P.intensity[2] * pr, 0.f);
    M1[o] = make_float4(accM.x * P.sca_mie[0] * P.intensity[0] * a, accM.y * P.sca_mie[1] * P.intensity[1] * a,
                        accM.z * P.sca_mie[2] * P.intensity[2] * a, 0.f);
  }
  count(wc, lit, 0, 0, 0);
}

// dS' = ray-scatter of an interpolated dJ table (atmosphere_lut.clj:92,94; atmosphere.clj:192-200).
//
// dJ comes packed: 3 floats per entry, each ray's slab in (heading, sun elevation) order, a "column" being
// the sun elevations of one heading.  At sample p_i the height and elevation coordinates of the lookup are the
// same for every entry of the ray, so those two dimensions are folded once per sample, and each entry then
// interpolates its own sun-elevation coordinate in the folded slab.  Its heading coordinate is constant along
// the ray: the sum over the samples is taken per column and the two columns are mixed at the end, so that a
// lookup needs one column only ("item": a column and a sun direction).  Entries whose sun direction
// index-to-sun-direction clamps to the same one share their items.
//
// One workgroup per view ray.  A wavefront owns a group of columns (TS x 64 folded texels at most) and a
// contiguous segment of the ray's samples: it folds its columns into a slab of its own in LDS and looks its
// items up there, so no barrier separates the two.  What bounds it is the LDS (busy for half of a
// launch) and the latency between a sample's writes and reads, which 4 wavefronts per SIMD cover in part (they wait for
// half of their time; a fifth wavefront spills registers, 60 us): per sample and wavefront of the
// 32 x 64 x 32 x 8 grid 4 texels written and 5 lookups of two texels each, beside 4 x 12 multiply-adds of the fold and
// 5 x 20 instructions of the lookups.  A slab therefore lies in two planes, red and green in 8 bytes at byte address A and
// blue in 4 at A / 2: a 16-byte write takes 13.4 clocks where one of 8 and one of 4 take 10.7, and the rows of a column
// then meet in a bank 32 (64) rows apart instead of 16.  57.4 -> 53.6 us; 64 x 128 x 64 x 16 with 128 samples 1385 -> 1235 us,
// 32 x 127 x 32 x 8 with 100 samples 159 -> 143 us.
//
// The sun-elevation coordinate of sun-elevation-to-index (atmosphere.clj:322-326) at p_i,
// (NL - 1) max(0, (1 - exp(-3 s - 0.6)) / (1 - exp(-3.6))) with s = dot(p_i, l) / |p_i| = (xl + t_i vl) / r_i, is
// A - A exp2(alpha_i xl + beta_i vl + c) with A = (NL - 1) / (1 - exp(-3.6)), alpha_i = -3 log2(e) / r_i,
// beta_i = alpha_i t_i, c = -0.6 log2(e), clamped to [0, NL - 1] (interpolate.clj:75-98 clips the coordinate).
// Each column of the slab ends in a zero texel, which only the coordinate NL - 1 reads, with weight zero.
struct SunCoord {
  float A, c, top;  // A, c, NL - 1
};

__device__ __forceinline__ float sun_coord(const SunCoord& sc, float2 ab, float xl, float vl) {
  const float e = fexp2(fmaf(ab.y, vl, fmaf(ab.x, xl, sc.c)));
  return __builtin_amdgcn_fmed3f(fmaf(-sc.A, e, sc.A), 0.0f, sc.top);
}

// Sun-elevation grids with fewer rows than this take the exact form below.  Their rows lie far apart in
// sun elevation, so neighbouring rows can differ by orders of magnitude (a sun below the horizon against
// one above it), and the ~1e-7 index units of rounding in sun_coord's FP32 form weight such a row by as
// much: where the true coordinate is integral (a vertical ray keeps its sun elevation) or clamped (the
// exponent cancels to 0 at sin = -0.2), the FP64 oracle gives that row no weight at all.
constexpr int kExactSunRows = 16;

// sun_coord in FP64: z = -3 dot(p_i, l) / r_i - 0.6 from the sample's t_i, h_i and the entry's dot(x, l),
// dot(v, l) (1 / r_i: the FP32 estimate and one FP64 Newton step, relative error ~1e-14), the coordinate
// (NL - 1) (1 - e^z) / (1 - e^-3.6) with 1 - e^z = -expm1(z) (no cancellation near the clamp), clamped, and
// its lower row and weight, the weight formed in FP64 before rounding (a coordinate just above a row, say
// 1 + 5e-6, would lose 1% of its weight to the FP32 spacing at 1).  A64: (NL - 1) / (1 - e^-3.6).
__device__ __forceinline__ void sun_coord_exact(const SunCoord& sc, double A64, double R, double2 th, double xl,
                                                double vl, unsigned& row, float& s) {
  const double r = R + th.y;
  double inv = (double)__builtin_amdgcn_rcpf((float)r);
  inv = fma(inv, fma(-r, inv, 1.0), inv);
  const double a = -3.0 * inv;
  const double z = fma(a * th.x, vl, fma(a, xl, -0.6));
  const double c = fmin(fmax(-expm1(z) * A64, 0.0), (double)sc.top);
  const double r0 = fmin(floor(c), (double)sc.top - 1.0);
  row = (unsigned)r0;
  s = (float)(c - r0);
}

__device__ __forceinline__ float3 lerp3(float4 a, float4 b, float s) {
  return make_float3(fmaf(s, b.x - a.x, a.x), fmaf(s, b.y - a.y, a.y), fmaf(s, b.z - a.z, a.z));
}

// The per-build fold steps of one ray, read-only while a ray-scatter launch runs.  The single-atmosphere
// kernel reads them through its restrict argument; the batched one through the constant address space,
// where the compiler cannot otherwise prove them unclobbered and would use vector loads.
typedef __attribute__((address_space(4))) const int* ConstFoldSteps;

__device__ __forceinline__ FoldStep fold_step(const FoldStep* __restrict__ fs, int i) { return fs[i]; }

__device__ __forceinline__ FoldStep fold_step(ConstFoldSteps fs, int i) {
  const ConstFoldSteps p = fs + 8 * i;  // FoldStep: 8 dwords
  FoldStep st;
  st.off = make_int4(p[0], p[1], p[2], p[3]);
  st.wt = make_float4(__int_as_float(p[4]), __int_as_float(p[5]), __int_as_float(p[6]), __int_as_float(p[7]));
  return st;
}

// A lookup's byte address base + column x pitch, formed as the bits of a denormal float (build.py: denormals are kept):
// bases and pitches are below 2^23, so the sum is exact and the column needs no conversion to an integer.  The multiply-add and the subtraction
// that finds the column issue at twice the rate of a conversion, an integer multiply-add or a clamp.
__device__ __forceinline__ unsigned lds_address(float column, unsigned pitch, unsigned base) {
  return __float_as_uint(fmaf(column, __uint_as_float(pitch), __uint_as_float(base)));
}

// LDS by address, for a kernel without static LDS, whose dynamic LDS begins at 0 (dynamic_lds_from_zero; as an offset
// from the array it would cost an addition of the array's place, 0, at each access).
typedef float Vec2 __attribute__((ext_vector_type(2)));
typedef float Vec4 __attribute__((ext_vector_type(4)));
template <class T>
__device__ __forceinline__ void lds_write(unsigned address, T v) {
  *(__attribute__((address_space(3))) T*)(uintptr_t)address = v;
}

template <class T>
__device__ __forceinline__ T lds_read(unsigned address) {
  return *(__attribute__((address_space(3))) const T*)(uintptr_t)address;
}

// Orders LDS accesses of one wavefront's lanes (the hardware keeps a wavefront's LDS accesses in order; this
// keeps the compiler from moving them across).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct Rgb {
  float x, y, z;
};

// Register slots of the fold: slot ((h & 1) << 1) | (e & 1) holds dJ at node (h, e) for the lane's texels.
// The four corners of a cell have distinct parities, so every sample's corners occupy the four slots, and a
// corner shared with the previous sample is already in its slot: a slot is re-read only when its node
// changes (about 60 node reads per ray of 64 samples).
template <int TS>
struct FoldSlots {
  Rgb v[4][TS];
};

// The group's texels of a node as a buffer of `bytes` bytes: lane l's texels lie at 12 (l + 64 j) from its start, and
// those past the group's read as zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t node_buffer(const float* __restrict__ dJ, int off, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)(dJ + 3LL * off), 0, bytes, 0x00020000);
}

// Re-reads the slots whose node differs between two samples (workgroup-uniform offsets and branches).
template <int TS>
__device__ __forceinline__ void fold_load(const float* __restrict__ dJ, const int4 was, const int4 now, int bytes,
                                          int lane, FoldSlots<TS>& f) {
  const int o[4] = {now.x, now.y, now.z, now.w}, p[4] = {was.x, was.y, was.z, was.w};
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (o[c] >= 0 && o[c] != p[c]) {
      const __amdgpu_buffer_rsrc_t node = node_buffer(dJ, o[c], bytes);
#pragma unroll
      for (int j = 0; j < TS; ++j) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(node, lane * (int)sizeof(Rgb) + j * 64 * (int)sizeof(Rgb), 0, 0);
        f.v[c][j] = Rgb{__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2])};
      }
    }
}

// Texels of a wavefront's slab for TS texels per lane, with the zero texel that ends each column (a group has at
// most 64 TS / NL columns; NL >= 16 but for the exact form, which takes NL >= 2).
template <int TS>
__host__ __device__ constexpr int rs_texels(bool exact) {
  return 64 * TS + (exact ? 32 * TS : 4 * TS);
}

// LDS of one workgroup: the wavefronts' slabs, whose place the item sums take later ([segs][3][groups x slots]).  For W
// wavefronts of N texels the 4-byte plane lies at 4 W N and the 8-byte plane at 8 W N: 16 bytes per texel, of which the
// first 4 are not used, and no offset between an address and its half.
template <int TS>
inline size_t rs_shared_bytes(int wavefronts, int slots, bool exact) {
  return wavefronts * std::max(rs_texels<TS>(exact) * sizeof(float4), (size_t)slots * 3 * sizeof(float));
}

// One wavefront's samples i0 .. i1 - 1 over NS lookup slots: acc[j] = sum over its samples of T(x, p_i) times
// the folded slab interpolated for the lane's item of slot j.
template <int TS, int NS, bool kExact, class Steps>
__device__ __forceinline__ void rs_segment(const float* __restrict__ dJ, const Steps gF, const float4* __restrict__ gT,
                                           const float4* __restrict__ gRS, const double2* __restrict__ gTH, int i0, int i1,
                                           int bytes, unsigned slab, const unsigned (&laddr)[TS],
                                           const RsItem* __restrict__ items, int nitems, const double2* __restrict__ ss,
                                           int col0, int pitch, const SunCoord& sc, double R, double A64, int lane,
                                           float* s_out, int out_pitch) {
  FoldSlots<TS> f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int j = 0; j < TS; ++j) f.v[c][j] = Rgb{0.f, 0.f, 0.f};
  FoldStep st = fold_step(gF, i0);
  fold_load<TS>(dJ, make_int4(-1, -1, -1, -1), st.off, bytes, lane, f);
  float xl[NS], vl[NS];
  double xl64[kExact ? NS : 1], vl64[kExact ? NS : 1];
  unsigned caddr[NS];
  Rgb acc[NS];
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const RsItem it = items[min(64 * j + lane, nitems - 1)];  // lanes past the last item repeat it
    vl[j] = it.vl;
    xl[j] = it.xl;
    if (kExact) {
      const double2 d = ss[it.at & 0xffff];
      vl64[j] = d.x;
      xl64[j] = d.y;
    }
    caddr[j] = slab + ((it.at >> 16) - col0) * pitch * 8u;
    acc[j] = Rgb{0.f, 0.f, 0.f};
  }
  for (int i = i0; i < i1; ++i) {
    const float4 w = st.wt;
#pragma unroll
    for (int j = 0; j < TS; ++j) {
      const Rgb a = f.v[0][j], b = f.v[1][j], c = f.v[2][j], d = f.v[3][j];
      lds_write(laddr[j], Vec2{fmaf(w.w, d.x, fmaf(w.z, c.x, fmaf(w.y, b.x, w.x * a.x))),
                               fmaf(w.w, d.y, fmaf(w.z, c.y, fmaf(w.y, b.y, w.x * a.y)))});
      lds_write(laddr[j] >> 1, fmaf(w.w, d.z, fmaf(w.z, c.z, fmaf(w.y, b.z, w.x * a.z))));
    }
    wave_fence();
    // the next sample's nodes, in flight during this sample's lookups
    const FoldStep nx = fold_step(gF, min(i + 1, i1 - 1));
    fold_load<TS>(dJ, st.off, nx.off, bytes, lane, f);
    st = nx;
    const float4 T = gT[i], g = gRS[i];  // uniform: scalar loads
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      unsigned A;
      float s;
      if (kExact) {
        unsigned row;
        sun_coord_exact(sc, A64, R, gTH[i], xl64[j], vl64[j], row, s);
        A = caddr[j] + row * 8;
      } else {
        const float c = sun_coord(sc, make_float2(g.z, g.w), xl[j], vl[j]);
        s = __builtin_amdgcn_fractf(c);
        A = lds_address(c - s, 8, caddr[j]);
      }
      const unsigned B = A >> 1;
      const Vec2 u0 = lds_read<Vec2>(A), u1 = lds_read<Vec2>(A + 8);
      const float b0 = lds_read<float>(B), b1 = lds_read<float>(B + 4);
      const float3 v = make_float3(fmaf(s, u1[0] - u0[0], u0[0]), fmaf(s, u1[1] - u0[1], u0[1]), fmaf(s, b1 - b0, b0));
      acc[j].x = fmaf(T.x, v.x, acc[j].x);
      acc[j].y = fmaf(T.y, v.y, acc[j].y);
      acc[j].z = fmaf(T.z, v.z, acc[j].z);
    }
    wave_fence();
  }
  __syncthreads();  // every wavefront has done with its slab: the sums take their place
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    s_out[64 * j + lane] = acc[j].x;
    s_out[out_pitch + 64 * j + lane] = acc[j].y;
    s_out[2 * out_pitch + 64 * j + lane] = acc[j].z;
  }
}

__device__ float3 resample4_value(const DevParams& P, const float4* __restrict__ a, const float4* __restrict__ b,
                                 long long idx, const float4* __restrict__ c = nullptr);
__device__ float3 resample4_value_lean(const DevParams& P, const float4* __restrict__ a, long long idx);
__device__ float3 resample2_value(const DevParams& P, int space, const float4* __restrict__ a,
                                 const float4* __restrict__ b, long long idx);

// An entry's result of a ray-scatter launch, and S + dS at this grid point (the running sum S of atmosphere_lut.clj:95-97).
template <bool kB>
__device__ __forceinline__ void rs_store(const DevParams& P, const RsAccum& accum, float4* __restrict__ out, long long at,
                                         float3 v, float dt) {
  const float4 d = make_float4(v.x * dt, v.y * dt, v.z * dt, 0.f);
  out[at] = d;
  if (accum.S_out) {
    const float4* S_in = atm_ptr<kB>(accum.S_in, P);
    const float3 u = accum.S_resample ? resample4_value_lean(P, S_in, at) : ld3(S_in, at);
    atm_ptr<kB>(accum.S_out, P)[at] = make_float4(u.x + d.x, u.y + d.y, u.z + d.z, 0.f);
  }
}

// The extra workgroups: E <- tab(dE + E) (atmosphere_lut.clj:95-96), an entry per thread.  (By one workgroup of the launch's
// size, 128 threads at 32 x 64 x 32 x 8, a surface-radiance table of 16 x 1024 made a launch of 53 us 180.)
inline unsigned rs_surface_blocks(const DevParams& P, const RsAccum& acc, unsigned threads) {
  return acc.E_out ? (unsigned)(((long long)P.nE[0] * P.nE[1] + threads - 1) / threads) : 0;
}

template <bool kB>
__device__ __forceinline__ void rs_surface(const DevParams& P, const RsAccum& accum, int block) {
  const long long nE = (long long)P.nE[0] * P.nE[1], i = (long long)block * blockDim.x + threadIdx.x;
  const float4* dE = atm_ptr<kB>(accum.dE, P);
  const float4* E_in = atm_ptr<kB>(accum.E_in, P);
  float4* E_out = atm_ptr<kB>(accum.E_out, P);
  if (i < nE) {
    const float3 v = resample2_value(P, 3, dE, E_in, i);
    E_out[i] = make_float4(v.x, v.y, v.z, 0.f);
  }
}

// segs: sample segments per group of columns (P.rs_groups x segs wavefronts, wavefront w working on group
// w / segs and segment w % segs).
template <int TS, bool kB, bool kExact>
__global__ void __launch_bounds__(1024) ray_scatter_kernel(
    const DevParams P0, const DevParams* __restrict__ PB, const float* __restrict__ dJ,
    const double2* __restrict__ geo_th, const float4* __restrict__ geo_T, const float4* __restrict__ geo_rs,
    const FoldStep* __restrict__ geo_fold, const RsItem* __restrict__ items, const uint2* __restrict__ entries,
    const int* __restrict__ heads, float4* __restrict__ out, const RsAccum accum, int segs, WorkCounters* wc) {
  const DevParams& P = params_of<kB>(P0, PB);
  if constexpr (kB) {  // this atmosphere's tables and ray geometry (the accumulation tables where they are used);
                       // offsets of the restrict arguments, whose loads stay provably unclobbered and uniform
    geo_th = atm_ptr<kB>(geo_th, P0);
    geo_T = atm_ptr<kB>(geo_T, P0);
    geo_rs = atm_ptr<kB>(geo_rs, P0);
    // the fold steps and the items depend only on the planet and the grid, which the atmospheres of a batch
    // share: all read atmosphere 0's copy (one copy in the caches instead of one per atmosphere)
    dJ = atm_ptr<kB>(dJ, P);
    out = atm_ptr<kB>(out, P);
  }
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const int NLA = NL * NA;
  const int n = P.ray_steps;
  if ((int)blockIdx.x >= NH * NE) {
    rs_surface<kB>(P, accum, (int)blockIdx.x - NH * NE);
    return;
  }
  extern __shared__ float4 s_mem[];
  const int groups = P.rs_groups, slots = P.rs_slots, pitch_out = groups * slots;
  // XCD-aware, in ascending impact parameter: every sample of a straight ray has the same
  // |p| sqrt(1 - mu^2), so the (height, elevation) cells that a ray folds lie along one curve, and an XCD
  // given a contiguous range of impact parameters reads a band of the dJ table
  const int ord = xcd_ray(blockIdx.x, NH * NE);
  const int rayid = P.ray_order ? P.ray_order[ord] : ord;
  const long long base = (long long)rayid * NLA, base_n = (long long)rayid * n;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave / segs, seg = wave - group * segs;
  const double2* __restrict__ ss = P.sun_ss + base;
  const FoldStep* __restrict__ gS = geo_fold + base_n;
  const auto gF = [&] {
    if constexpr (kB) return (ConstFoldSteps)gS;
    else return gS;
  }();
  const SunCoord sc = {(float)((NL - 1) * (double)P.sun_inv_den), (float)(-0.6 * 1.4426950408889634), (float)(NL - 1)};
  const double A64 = kExact ? (NL - 1) / (1.0 - exp(-3.6)) : 0.0;
  const int* __restrict__ head = heads + (long long)rayid * (groups + 1);
  const int nitems = min(head[group + 1] - head[group], slots);
  // the lane's texels in the LDS slab; those past the group's texels write zeros to the last column's zero texel
  const int col0 = group * P.rs_cols, ncols = min(P.rs_cols, NA - col0), pitch = NL + 1;
  const unsigned texels = rs_texels<TS>(kExact), slab = 8 * (texels * (unsigned)(blockDim.x >> 6) + wave * texels);
  unsigned laddr[TS];
#pragma unroll
  for (int j = 0; j < TS; ++j) {
    const unsigned t = 64 * j + lane;
    laddr[j] = (t < (unsigned)(ncols * NL) ? t + t / (unsigned)NL : (unsigned)(ncols * pitch - 1)) * 8u + slab;
  }
  for (int i = lane; i < ncols; i += 64) {
    const unsigned A = slab + (i * pitch + NL) * 8;
    lds_write(A, Vec2{0.f, 0.f});
    lds_write(A >> 1, 0.f);
  }
  const int i0 = (int)((long long)n * seg / segs), i1 = (int)((long long)n * (seg + 1) / segs);
  const RsItem* __restrict__ it = items + 2 * base + head[group];
  float* s_out = (float*)s_mem + (size_t)seg * 3 * pitch_out + group * slots;
#define SFSIM_RS_CASE(NS)                                                                                             \
  case NS:                                                                                                            \
    if constexpr (64 * NS <= (kExact ? 64 * TS + 64 : rs_items(TS)))  /* exact: texels + 2 rows, of 15 at most */     \
      rs_segment<TS, NS, kExact>(dJ + 3 * col0 * NL, gF, geo_T + base_n, geo_rs + base_n, geo_th + base_n, i0, i1,     \
                                 ncols * NL * (int)sizeof(Rgb), slab, laddr, it, nitems, ss, col0, pitch, sc, P.g.R,  \
                                 A64, lane, s_out, pitch_out);                                                        \
    break
  switch ((nitems + 63) / 64) {
    SFSIM_RS_CASE(1);
    SFSIM_RS_CASE(2);
    SFSIM_RS_CASE(3);
    SFSIM_RS_CASE(4);
    SFSIM_RS_CASE(5);
    SFSIM_RS_CASE(6);
    SFSIM_RS_CASE(7);
    SFSIM_RS_CASE(8);
    default:  // no item of this group
      __syncthreads();
  }
#undef SFSIM_RS_CASE
  __syncthreads();
  // the ray's step D / n: twice its first sample's t = 0.5 D / n (FP64, exact), from the per-build geometry
  const float dt = (float)(2.0 * geo_th[base_n].x);
  for (int kk = threadIdx.x; kk < NLA; kk += blockDim.x) {
    const uint2 e = entries[base + kk];
    auto total = [&](unsigned at) {
      const float* q = (const float*)s_mem + at;
      float3 t = make_float3(q[0], q[pitch_out], q[2 * pitch_out]);
      for (int g = 1; g < segs; ++g) {
        q += 3 * pitch_out;
        t.x += q[0];
        t.y += q[pitch_out];
        t.z += q[2 * pitch_out];
      }
      return t;
    };
    float3 v = total(e.x & 0xffffu);
    const float s = __uint_as_float(e.y);
    if (s != 0.0f) {
      const float3 u = total(e.x >> 16);
      v = make_float3(fmaf(s, u.x - v.x, v.x), fmaf(s, u.y - v.y, v.y), fmaf(s, u.z - v.z, v.z));
    }
    rs_store<kB>(P, accum, out, base + kk, v, dt);
    count(wc, 0, 0, (unsigned long long)n, 0);
  }
}

// The same in plain order: both columns mixed at every sample and the samples added one by one.  The order sums that
// training and sfsim_atmo_order_sums read come from it (a network's training amplifies the last bit of its targets, so
// their rounding stays that of this plain order), and the results on grids whose columns have too many items (rs_split).
//
// One workgroup per view ray, TS texels and entries per lane.  The lanes' dJ values lie in registers as in
// ray_scatter_kernel, the whole slab is folded into LDS, 16 bytes a texel.  With many rays (`samples` 1) all wavefronts fold
// and look up each sample, in two slabs with one barrier per sample, and a lane adds its own entries.  A grid of few rays
// waits for a sample's chain of loads and barriers: there `samples` samples are in work at once, each by wavefronts
// of its own, and the values are added in their order from LDS (16 x 32 x 16 x 8 at 32 samples 18.5 us, 32 without).  Gathering
// every lookup's 16 texels from dJ instead, sfsim_atmo_order_sums took 5.5 ms at 32 x 64 x 32 x 8 and 64 samples and 139 at
// 64 x 128 x 64 x 16 and 128; now 2.5 and 35.5.
template <int TS, bool kB, bool kExact>
__global__ void __launch_bounds__(1024) ray_scatter_ordered_kernel(
    const DevParams P0, const DevParams* __restrict__ PB, const float* __restrict__ dJ, const double2* __restrict__ geo_th, const float4* __restrict__ geo_T,
    const float4* __restrict__ geo_rs, const FoldStep* __restrict__ geo_fold, float4* __restrict__ out, const RsAccum accum,
    int samples, WorkCounters* wc) {
  const DevParams& P = params_of<kB>(P0, PB);
  if constexpr (kB) {  // as in ray_scatter_kernel
    geo_th = atm_ptr<kB>(geo_th, P0);
    geo_T = atm_ptr<kB>(geo_T, P0);
    geo_rs = atm_ptr<kB>(geo_rs, P0);
    dJ = atm_ptr<kB>(dJ, P);
    out = atm_ptr<kB>(out, P);
  }
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3], NLA = NL * NA, n = P.ray_steps;
  if ((int)blockIdx.x >= NH * NE) {
    rs_surface<kB>(P, accum, (int)blockIdx.x - NH * NE);
    return;
  }
  extern __shared__ float4 s_mem[];
  const int ord = xcd_ray(blockIdx.x, NH * NE);
  const int rayid = P.ray_order ? P.ray_order[ord] : ord;
  const long long base = (long long)rayid * NLA, base_n = (long long)rayid * n;
  const double2* __restrict__ ss = P.sun_ss + base;
  const FoldStep* __restrict__ gS = geo_fold + base_n;
  const auto gF = [&] {
    if constexpr (kB) return (ConstFoldSteps)gS;
    else return gS;
  }();
  const SunCoord sc = {(float)((NL - 1) * (double)P.sun_inv_den), (float)(-0.6 * 1.4426950408889634), (float)(NL - 1)};
  const double A64 = kExact ? (NL - 1) / (1.0 - exp(-3.6)) : 0.0;
  const int lane = threadIdx.x & 63, all = (int)blockDim.x, threads = all / samples;  // threads: of a sample
  const int mine = __builtin_amdgcn_readfirstlane((int)threadIdx.x / threads), tid = (int)threadIdx.x - mine * threads;
  const int first = __builtin_amdgcn_readfirstlane(tid >> 6) * 64 * TS;
  const int texels = max(0, min(64 * TS, NLA - first)), bytes = texels * (int)sizeof(Rgb);
  const float* __restrict__ own = dJ + 3 * first;
  float4* slabs = s_mem + mine * NLA;
  float* terms = (float*)(s_mem + samples * NLA);  // [samples][3][NLA], and the samples' T (samples > 1)
  float4* s_T = (float4*)(terms + (3 * samples * NLA + 3) / 4 * 4);
  if (samples > 1)
    for (int i = threadIdx.x; i < n; i += all) s_T[i] = geo_T[base_n + i];
  int c0[TS], c1[TS];
  float mix[TS], vl[TS], xl[TS];
  Rgb acc[TS];
  bool two = false;
  // the lane's entries, in (heading, sun elevation) order: neighbouring lanes read neighbouring rows
  auto entry = [&](int q) {
    const int a = q / NL;
    return (q - a * NL) * NA + a;
  };
#pragma unroll
  for (int e = 0; e < TS; ++e) {
    const double2 d = ss[entry(min(tid + e * threads, NLA - 1))];
    const Lerp L = make_lerp((float)sun_angle_to_index(NA, d.x), NA);
    c0[e] = L.i0 * NL;
    c1[e] = L.i1 * NL;
    mix[e] = L.s;
    two = two || L.s != 0.0f;
    vl[e] = (float)d.x;
    xl[e] = (float)d.y;
    acc[e] = Rgb{0.f, 0.f, 0.f};
  }
  two = __any(two);
  FoldSlots<TS> f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int j = 0; j < TS; ++j) f.v[c][j] = Rgb{0.f, 0.f, 0.f};
  // the next sample's nodes are in flight during a sample's lookups, and its step is read a sample before that
  FoldStep st = fold_step(gF, min(mine, n - 1)), nx = fold_step(gF, min(mine + samples, n - 1));
  float4 g = geo_rs[base_n + min(mine, n - 1)];
  fold_load<TS>(own, make_int4(-1, -1, -1, -1), st.off, bytes, lane, f);
  for (int round = 0; round < n; round += samples) {
    const int i = min(round + mine, n - 1);  // (past the last sample: the last again, not added)
    float4* slab = samples == 1 ? slabs + (round & 1) * NLA : slabs;
    const float4 w = st.wt;
#pragma unroll
    for (int j = 0; j < TS; ++j)
      if (64 * j + lane < texels) {
        const Rgb a = f.v[0][j], b = f.v[1][j], c = f.v[2][j], d = f.v[3][j];
        slab[first + 64 * j + lane] = make_float4(fmaf(w.w, d.x, fmaf(w.z, c.x, fmaf(w.y, b.x, w.x * a.x))),
                                                  fmaf(w.w, d.y, fmaf(w.z, c.y, fmaf(w.y, b.y, w.x * a.y))),
                                                  fmaf(w.w, d.z, fmaf(w.z, c.z, fmaf(w.y, b.z, w.x * a.z))), 0.f);
      }
    fold_load<TS>(own, st.off, nx.off, bytes, lane, f);
    st = nx;
    nx = fold_step(gF, min(round + 2 * samples + mine, n - 1));
    const float2 ab = make_float2(g.z, g.w);
    g = geo_rs[base_n + min(round + samples + mine, n - 1)];
    const float4 T = geo_T[base_n + i];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < TS; ++e) {
      unsigned row;
      float s;
      if (kExact) {
        const double2 d = ss[entry(min(tid + e * threads, NLA - 1))];
        sun_coord_exact(sc, A64, P.g.R, geo_th[base_n + i], d.y, d.x, row, s);
      } else {
        const float c = sun_coord(sc, ab, xl[e], vl[e]);
        row = min((unsigned)c, (unsigned)NL - 2);
        s = c - (float)row;
      }
      const float4 *p = slab + c0[e] + row, *q = slab + c1[e] + row;
      const float4 p0 = p[0], p1 = p[1];
      float3 u = make_float3(p0.x, p0.y, p0.z), v = make_float3(p1.x, p1.y, p1.z);
      if (two) {
        u = lerp3(p0, q[0], mix[e]);
        v = lerp3(p1, q[1], mix[e]);
      }
      v = make_float3(fmaf(s, v.x - u.x, u.x), fmaf(s, v.y - u.y, u.y), fmaf(s, v.z - u.z, u.z));
      if (samples == 1) {
        acc[e].x = fmaf(T.x, v.x, acc[e].x);
        acc[e].y = fmaf(T.y, v.y, acc[e].y);
        acc[e].z = fmaf(T.z, v.z, acc[e].z);
      } else if (tid + e * threads < NLA) {
        float* t = terms + 3 * mine * NLA + tid + e * threads;
        t[0] = v.x;
        t[NLA] = v.y;
        t[2 * NLA] = v.z;
      }
    }
    if (samples > 1) {
      __syncthreads();
#pragma unroll
      for (int e = 0; e < TS; ++e) {
        const int q = (int)threadIdx.x + e * all;
        if (q < NLA)
#pragma unroll 2
          for (int j = 0; j < min(samples, n - round); ++j) {
            const float4 Tj = s_T[round + j];
            const float* t = terms + 3 * j * NLA + q;
            acc[e].x = fmaf(Tj.x, t[0], acc[e].x);
            acc[e].y = fmaf(Tj.y, t[NLA], acc[e].y);
            acc[e].z = fmaf(Tj.z, t[2 * NLA], acc[e].z);
          }
      }
    }
  }
  __syncthreads();
  float* sums = (float*)s_mem;
#pragma unroll
  for (int e = 0; e < TS; ++e) {
    const int q = (int)threadIdx.x + e * all;
    if (q < NLA) {
      const int k = entry(q);
      sums[k] = acc[e].x;
      sums[NLA + k] = acc[e].y;
      sums[2 * NLA + k] = acc[e].z;
    }
  }
  __syncthreads();
  const float dt = (float)(2.0 * geo_th[base_n].x);  // as in ray_scatter_kernel
  for (int k = threadIdx.x; k < NLA; k += all) {
    rs_store<kB>(P, accum, out, base + k, make_float3(sums[k], sums[NLA + k], sums[2 * NLA + k]), dt);
    count(wc, 0, 0, (unsigned long long)n, 0);
  }
}

// dJ = point-scatter over the sphere quadrature (atmosphere_lut.clj:88,91; atmosphere.clj:203-222).
// Every grid point of a height index shares its position and quadrature frame, so the per-direction
// geometry (ray extremity P, surface flag, T(x, P), elevation coordinate of omega at x) depends only
// on (height, direction) and is computed once per build (direction_geometry_kernel).  The dS lookup
// at (x, omega, l) has a height coordinate that depends only on the height and an elevation coordinate that
// depends only on the height and the direction's latitude ring (sphere.clj:62-105: the directions of a ring share
// dot(x, omega)): point_scatter_kernel folds those two dimensions ring by ring.
struct DirGeom {
  float4 omega;   // direction xyz, w: elevation coordinate of omega at x (flag: not surface)
  float4 ground;  // T(x, P) * brightness / pi (0 for sky directions), w: 1 for surface directions
  float4 phat;    // P / |P| (w unused: P is on the ground, height row 0 of the surface-radiance table)
};

__device__ __forceinline__ void direction_geometry_body(const DevParams& P, const Dir* __restrict__ dirs,
                                                                    int ndirs, DirGeom* __restrict__ geom,
                                                                    WorkCounters* wc, unsigned blk) {
  const int NH = P.nS[0], NE = P.nS[1];
  const int n = P.ray_steps;
  int idx = blk * blockDim.x + threadIdx.x;
  bool active = idx < NH * ndirs;
  int ih = active ? idx / ndirs : 0, j = active ? idx - ih * ndirs : 0;
  const double r0 = index_to_radius(P.g, NH, ih), h0 = index_to_altitude(P.g, NH, ih);
  Dir d = dirs[j];
  double pd = r0 * d.x;  // dot(x, omega)
  bool above = is_above_horizon(P.g, h0, pd);
  double D = above ? top_exit_distance(P.g, h0, pd) : ground_distance(P.g, h0, pd);
  double hP = altitude_along(P.g, h0, pd, D);
  bool surface = 2.0 * hP < P.g.H;  // atmosphere.clj:88-92
  // every lane evaluates the transmittance (uniform control flow for the wavefront vote inside);
  // sky directions discard it
  float3 T = segment_transmittance(P, h0, pd, D, n);
  if (!active) return;
  DirGeom g;
  g.omega = make_float4((float)d.x, (float)d.y, (float)d.z, (float)elevation_to_index(P.g, NE, r0, pd, !surface));
  if (surface) {
    g.ground = make_float4(T.x * P.brightness_over_pi[0], T.y * P.brightness_over_pi[1], T.z * P.brightness_over_pi[2],
                           1.f);
    double px = r0 + d.x * D, py = d.y * D, pz = d.z * D;
    double pn = 1.0 / sqrt(px * px + py * py + pz * pz);
    g.phat = make_float4((float)(px * pn), (float)(py * pn), (float)(pz * pn), 0.f);
  } else {
    g.ground = make_float4(0.f, 0.f, 0.f, 0.f);
    g.phat = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  geom[idx] = g;
  count(wc, 0, surface ? n : 0, 0, 0);
}

__global__ void __launch_bounds__(kBlock) direction_geometry_kernel(const DevParams P, const Dir* __restrict__ dirs,
                                                                    int ndirs, DirGeom* __restrict__ geom,
                                                                    WorkCounters* wc) {
  direction_geometry_body(P, dirs, ndirs, geom, wc, blockIdx.x);
}

// Constants of the per-direction lookups of one point-scatter launch.
struct PsConst {
  float hA;            // (NA - 1) / 2: heading coordinate (NA - 1) (1 + dot(omega, l)) / 2 = hA + hA dot(omega, l)
  SunCoord se;         // sun-elevation coordinate of dE (size nE[1]): alpha = -3 log2(e), beta = 0
  float mie_k, mie_a, mie_b;  // Mie phase K (1 + mu^2) (a - b mu)^(-3/2): K = 3 (1 - g^2) / (8 pi (2 + g^2))
};

// Without contraction: the same values whatever surrounds the call (near g = 1, 1 + g^2 - 2 g mu amplifies the last
// bit of its terms).
__device__ __forceinline__ void mie_constants(float g, PsConst& pc) {
#pragma clang fp contract(off)
  const float g2 = g * g;
  pc.mie_k = 3.0f * (1.0f - g2) / (8.0f * 3.14159265358979f * (2.0f + g2));
  pc.mie_a = 1.0f + g2;
  pc.mie_b = 2.0f * g;
}

// phase_f with its constants as in mie_constants: the weights of the launch that adds the Mie term (the other
// launches take phase_f; each keeps the rounding that the surrogate's training data has been made with).
__device__ __forceinline__ float weight_phase(float g, float mu) {
  float a, k, d;
  {
#pragma clang fp contract(off)
    const float g2 = g * g;
    a = 1.0f + g2;
    k = 3.0f * (1.0f - g2);
    d = 8.0f * 3.14159265358979f * (2.0f + g2);
  }
  const float x = a - 2.0f * g * mu;
  return (k * (1.0f + mu * mu)) / (d * (x * sqrtf(x)));
}

// phase of atmosphere.clj:56-61 with the hardware reciprocal square root (x^-3/2 = rsq(x)^3)
__device__ __forceinline__ float mie_phase(const PsConst& pc, float mu) {
  const float y = __builtin_amdgcn_rsqf(fmaf(-pc.mie_b, mu, pc.mie_a));
  return pc.mie_k * fmaf(mu, mu, 1.0f) * (y * y * y);
}

template <bool kFold>
__device__ __forceinline__ void surface_radiance_entry(const DevParams& P, int ndirs, const float4* __restrict__ dS,
                                                       const float4* __restrict__ mie, float4* __restrict__ out,
                                                       WorkCounters* wc, int entry, float4* s_fold, float3* s_red);

// The split of a point-scatter launch.  A workgroup takes `rays` view rays of one height and `rows` sun elevations,
// `waves` wavefronts per ray (64 EPT entries each); eblocks x sblocks workgroups per height.  pitch: texels per
// column of its slab.  dirs: directions whose weights are in LDS at a time.  e_lds: whether dE is.  The rest: byte
// addresses of what the LDS holds (see ps_layout) and its size.
struct PsPlan {
  int rows, sblocks, rays, waves, eblocks, pitch, dirs;
  bool e_lds;
  unsigned plane8, weights, dE16, dE8, omega, bytes;
};

// LDS of a workgroup: the folded slab of one latitude ring, double-buffered (and of the Mie strength in the first
// iteration), a texel for each column and sun elevation: its colour and the difference to the next column's, six
// floats in two planes: 16 bytes (colour, first difference) at byte address A, the other 8 at A / 2.  Column NA - 1
// holds the column before it plus its difference (what the interpolation between the two gives at weight 1) and no
// difference, and a column -1 column 0's colour and no difference: a heading coordinate that rounding has left just
// outside 0 ... NA - 1 gives what the clamped one would, so a lookup clamps neither the coordinate nor the column.
// The 8-byte plane begins at its own size and the 16-byte plane at twice that (ps_layout); the weights, dE (laid
// out alike) and the directions lie below the planes where they fit and else behind them.
// Where the directions' components are read: from LDS with one entry per lane, whose few lookups do not cover the
// latency of scalar loads (19 x 45 x 20 x 7 entries, 38 directions: 17.4 us against 19.1); from scalar registers with
// two entries per lane, which read more of the LDS per direction (1408 us against 1317 at 64 x 128 x 64 x 16 with 262
// directions), and with the Mie strength (24 x 48 x 24 x 9, 134 directions: 69.2 us against 66.1).
__host__ __device__ constexpr bool ps_omega_in_lds(int ept, bool mie) { return ept == 1 && !mie; }

// One texel more than the slabs have: where a wavefront holds an entry with a weight on sun-elevation row 1, all its
// lanes read the texel behind their own, also the one that ends the last slab (they do not use it).
__host__ __device__ inline unsigned ps_texels(const PsPlan& p, int na, bool mie) {
  return 2u * (mie ? 2u : 1u) * (unsigned)p.pitch * (unsigned)(na + 1) + 1u;
}
// One texel: u and the difference to v; `last`: what interpolation at weight 1 gives, and no difference.
__device__ __forceinline__ void ps_store(float4* a, float2* b, float3 u, float3 v, bool last) {
  const float3 d = make_float3(v.x - u.x, v.y - u.y, v.z - u.z);
  *a = last ? make_float4(u.x + d.x, u.y + d.y, u.z + d.z, 0.f) : make_float4(u.x, u.y, u.z, d.x);
  *b = last ? make_float2(0.f, 0.f) : make_float2(d.y, d.z);
}

// Latitude rings of the sphere quadrature: ring i holds directions start[i] .. start[i + 1] - 1.
struct PsRings {
  int count;
  unsigned short start[kMaxRings + 1];
};

// What bounds it is VALU issue and, close behind, the LDS: 13 instructions per (entry, sky direction), 3 of them of the
// kinds that issue at half rate, and some 32 per ground direction, beside 24 bytes of LDS reads per lookup (at
// 64 x 128 x 64 x 16 and 262 directions the LDS is busy for 3/4 of the launch).  Lookup addresses formed as floats and
// columns that need no clamp took that launch from 1370 to 1317 us, and 19 x 45 x 20 x 7 with 38 directions from 18.9 to
// 17.4 us together with directions read from LDS.  The slab of a ring is shared by the ring's directions and by the
// rays of a height, so it is folded in the kernel itself (nine times fewer texels than one slab per direction, and no
// launch, table or gather from L2 for them); lanes run over the sun elevations of a column, so that their reads of a
// slab's columns are contiguous whatever columns they need.
//
// kELds: the previous order's dE at the ground (height row 0) is staged in LDS.  P, the ground point of a surface
// direction, is the ray's intersection with the planet's sphere (atmosphere.clj:80-85, 213-221), so its height is
// 0: its FP64 |P| - R is rounding noise of ~1e-9 m, whose height coordinate (through the square root of the
// horizon distance, ~1.5e-6 for 16 rows and 100 km) would weight height row 1 by as much.
//
// The iteration's surface radiance (it reads the same dS and Mie strength) rides in the launch: the sr.count
// workgroups after the rays' compute its entries with the LDS-folded kernel body.
template <int EPT, bool kMie, bool kELds, bool kB, bool kBatches>
__global__ void __launch_bounds__(kBlock) point_scatter_kernel(
    const DevParams P0, const DevParams* __restrict__ PB, const Dir* __restrict__ dirs, const DirGeom* __restrict__ geom,
    int ndirs, const PsRings rings, const float4* __restrict__ dS, const float4* __restrict__ mie,
    const float4* __restrict__ dE, float* __restrict__ out, const SrJob sr, const PsPlan plan, WorkCounters* wc) {
  extern __shared__ float4 s_mem[];
  char* const lds = (char*)s_mem;
  const DevParams& P = params_of<kB>(P0, PB);
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const int NLA = NL * NA, blocks = NH * plan.eblocks * plan.sblocks;
  if ((int)blockIdx.x >= blocks) {
    float3* s_red = (float3*)s_mem;  // one per wavefront
    surface_radiance_entry<true>(P, sr.ndirs, atm_ptr<kB>(sr.dS, P), atm_ptr<kB>(sr.mie, P), atm_ptr<kB>(sr.out, P),
                                 wc, (int)blockIdx.x - blocks, s_mem + 4, s_red);
    return;
  }
  geom = atm_ptr<kB>(geom, P);
  dS = atm_ptr<kB>(dS, P);
  mie = atm_ptr<kB>(mie, P);
  dE = atm_ptr<kB>(dE, P);
  out = atm_ptr<kB>(out, P);
  const int b = xcd_ray(blockIdx.x, blocks), hb = b / plan.sblocks, ih = hb / plan.eblocks;
  const int s0 = (b - hb * plan.sblocks) * plan.rows, rows = min(plan.rows, NL - s0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = wave / plan.waves, part = wave - r * plan.waves;
  const int ie = (hb - ih * plan.eblocks) * plan.rays + r;
  const bool active = r < plan.rays && ie < NE;  // whole wavefronts; the others help to fold
  const int nE1 = P.nE[1];
  float4* s_w = (float4*)(lds + plan.weights) + r * plan.dirs;  // [rays][dirs] rgb quadrature weight times in-scattering
  float4* s_ea = (float4*)(lds + plan.dE16);                    // dE at the ground and the differences to the next
  float2* s_eb = (float2*)(lds + plan.dE8);                     // entry's, as the slabs' texels
  float2* s_om = (float2*)(lds + plan.omega);                   // [dirs] omega's y and z
  constexpr bool kOmLds = ps_omega_in_lds(EPT, kMie);
  const double r0 = index_to_radius(P.g, NH, ih), h0 = index_to_altitude(P.g, NH, ih);
  const DirGeom* __restrict__ gh = geom + (long long)ih * ndirs;

  // Slab of one ring, columns fastest (coalesced reads).
  const int fold_rows = min(plan.pitch, NL - s0), fold_n = NA * fold_rows;
  const unsigned half = plan.plane8, slab_texels = (unsigned)(plan.pitch * (NA + 1));
  const Lerp Lh = make_lerp((float)height_to_index(P.g, NH, r0), NH);
  const long long sh = (long long)NE * NLA;
  auto fold = [&](int ring, unsigned buffer) {
    const Lerp Le = make_lerp(gh[rings.start[ring]].omega.w, NE);
    auto texel = [&](const float4* __restrict__ t, long long k) {
      const float3 u = mix3(ld3(t, Lh.i0 * sh + (long long)Le.i0 * NLA + k), ld3(t, Lh.i0 * sh + (long long)Le.i1 * NLA + k), Le.s);
      if (Lh.s == 0.0f) return u;  // mix3(u, v, 0) is u exactly
      return mix3(u, mix3(ld3(t, Lh.i1 * sh + (long long)Le.i0 * NLA + k), ld3(t, Lh.i1 * sh + (long long)Le.i1 * NLA + k), Le.s), Lh.s);
    };
    for (int i = threadIdx.x; i < fold_n; i += blockDim.x) {
      const int row = i / NA, col = i - row * NA;
      const bool last = col == NA - 1;
      const long long k = (long long)(s0 + row) * NA + col - last;
      const unsigned t = buffer * (kMie ? 2u : 1u) * slab_texels + (unsigned)((col + 1) * plan.pitch + row);
#pragma unroll
      for (int m = 0; m < (kMie ? 2 : 1); ++m) {
        const float4* __restrict__ tab = m ? mie : dS;
        const unsigned A = 2 * half + 16 * (t + m * slab_texels);
        const float3 u = texel(tab, k);
        ps_store((float4*)(lds + A), (float2*)(lds + (A >> 1)), u, texel(tab, k + 1), last);
        if (col == 0) {
          const unsigned B = A - 16 * plan.pitch;
          *(float4*)(lds + B) = make_float4(u.x, u.y, u.z, 0.f);
          *(float2*)(lds + (B >> 1)) = make_float2(0.f, 0.f);
        }
      }
    }
  };

  if (kELds)
    for (int i = threadIdx.x; i < nE1; i += blockDim.x) {
      const int k = min(i, nE1 - 2);
      ps_store(s_ea + i, s_eb + i, ld3(dE, k), ld3(dE, k + 1), k != i);
    }
  double se = 0.0, ce = 0.0;
  float bm = 0.f, br = 0.f;
  if (active) {
    bool above_unused;
    index_to_elevation(P.g, NE, r0, ie, se, ce, above_unused);
    bm = (float)exp(-h0 * P.inv_scale_mie);
    br = (float)exp(-h0 * P.inv_scale_ray);
  }
  if (kBatches) {
    se = uniform(se);
    ce = uniform(ce);
    bm = uniform(bm);
    br = uniform(br);
  }
  // The weights of directions j0 .. j1 - 1.
  auto weigh = [&](int j0, int j1) {
    if (kOmLds)
      for (int j = j0 + threadIdx.x; j < j1; j += blockDim.x) s_om[j - j0] = make_float2(gh[j].omega.y, gh[j].omega.z);
    if (!active) return;
    float g_mie = P.g_mie, g_ray = P.g_ray;
    if (kBatches) asm volatile("" : "+s"(g_mie), "+s"(g_ray));  // the phases' terms are not kept in registers between batches
    for (int j = j0 + part * 64 + lane; j < j1; j += 64 * plan.waves) {
      const Dir d = dirs[j];
      const float vw = (float)(se * d.x + ce * d.y);
      const float pm = (kMie ? weight_phase(g_mie, vw) : phase_f(g_mie, vw)) * bm;
      const float pr = (kMie ? weight_phase(g_ray, vw) : phase_f(g_ray, vw)) * br;
      const float w = (float)d.w;
      s_w[j - j0] = make_float4((P.sca_mie[0] * pm + P.sca_ray[0] * pr) * w, (P.sca_mie[1] * pm + P.sca_ray[1] * pr) * w,
                                (P.sca_mie[2] * pm + P.sca_ray[2] * pr) * w, 0.f);
    }
  };
  if (!kBatches) weigh(0, ndirs);
  PsConst pc;
  pc.hA = 0.5f * (float)(NA - 1);
  pc.se = SunCoord{(float)((nE1 - 1) * (double)P.sun_inv_den), (float)(-0.6 * 1.4426950408889634), (float)(nE1 - 1)};
  mie_constants(P.g_mie, pc);

  // The lane's entries, EPT slots of 64 in (heading, sun elevation) order.  A grid entry's own sun-elevation
  // coordinate is its row: index-to-sin-sun-elevation and back in FP64 is off by ~1e-13, which the rounding to FP32
  // takes away but at row 0, where it may leave a weight of that order on row 1.
  const int count_e = rows * NA;
  const long long base = ((long long)ih * NE + (active ? ie : 0)) * NLA;
  int at[EPT];
  float lx[EPT], ly[EPT], lz[EPT], s_up[EPT];
  unsigned row_bytes[EPT];
  float3 acc[EPT];
  bool two = false;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int q = min((part * EPT + e) * 64 + lane, count_e - 1), a = q / rows, is = q - a * rows;
    at[e] = a * NL + s0 + is;
    const float4 m = P.sun_ps[base + at[e]];  // l and the sun-elevation coordinate, rounded once from FP64
    lx[e] = m.x;
    ly[e] = m.y;
    lz[e] = m.z;
    s_up[e] = s0 + is == 0 ? make_lerp(m.w, NL).s : 0.0f;
    two = two || s_up[e] != 0.0f;
    row_bytes[e] = 2 * half + 16 * (plan.pitch + is);
    acc[e] = make_float3(0.f, 0.f, 0.f);
  }
  two = __any(two);
  fold(0, 0);
  if (!kBatches) __syncthreads();
  const unsigned pitch_bytes = 16 * plan.pitch, ea_bytes = plan.dE16, eb_bytes = plan.dE8;
  int jb = 0, weighed = 0;  // the first direction of the weights in LDS, the first ring past them
  for (int ring = 0; ring < rings.count; ++ring) {
    if (kBatches && ring == weighed) {  // as many rings as fit
      jb = rings.start[ring];
      for (weighed = ring + 1; weighed < rings.count && rings.start[weighed + 1] - jb <= plan.dirs;) ++weighed;
      weigh(jb, rings.start[weighed]);
      __syncthreads();
    }
    if (ring + 1 < rings.count) fold(ring + 1, (ring + 1) & 1);
    if (active) {
      const int j0 = rings.start[ring], j1 = rings.start[ring + 1];
      const bool to_ground = gh[j0].ground.w != 0.f;  // the ring's directions meet the ground
      const unsigned buffer_bytes = (ring & 1) * (kMie ? 32u : 16u) * slab_texels;
      // one lookup of the slab at byte address A: colour + s x difference
      auto lerp_at = [&](unsigned A, float s) {
        const Vec4 u = lds_read<Vec4>(A);
        const Vec2 d = lds_read<Vec2>(A >> 1);
        return make_float3(fmaf(s, u.w, u.x), fmaf(s, d.x, u.y), fmaf(s, d.y, u.z));
      };
      auto lookup = [&](unsigned A, float sa, int e, bool second) {
        float3 v = lerp_at(A, sa);
        if (second) {
          const float3 u = lerp_at(A + 16, sa);
          const float s = s_up[e];
          if (s != 0.0f) v = make_float3(fmaf(s, u.x - v.x, v.x), fmaf(s, u.y - v.y, v.y), fmaf(s, u.z - v.z, v.z));
        }
        return v;
      };
      auto directions = [&](auto ground_ring, bool second) {
        // dot(x, omega) is the ring's
        float x0[EPT];
        unsigned rb[EPT];
#pragma unroll
        for (int e = 0; e < EPT; ++e) {
          x0[e] = gh[j0].omega.x * lx[e];
          rb[e] = row_bytes[e] + buffer_bytes;
        }
#pragma unroll 2
        for (int j = j0; j < j1; ++j) {
          const float4 w = s_w[j - jb];
          const float2 om = kOmLds ? s_om[j - jb] : make_float2(gh[j].omega.y, gh[j].omega.z);
#pragma unroll
          for (int e = 0; e < EPT; ++e) {
            const float ol = fmaf(om.y, lz[e], fmaf(om.x, ly[e], x0[e]));
            const float hc = fmaf(pc.hA, ol, pc.hA), sa = __builtin_amdgcn_fractf(hc);
            const unsigned A = lds_address(hc - sa, pitch_bytes, rb[e]);
            float3 v = lookup(A, sa, e, second);
            if (kMie) {
              const float3 m = lookup(A + 16 * slab_texels, sa, e, second);
              const float ph = mie_phase(pc, ol);
              v.x = fmaf(m.x, ph, v.x);
              v.y = fmaf(m.y, ph, v.y);
              v.z = fmaf(m.z, ph, v.z);
            }
            if (ground_ring) {
              const float4 ph = gh[j].phat, ground = gh[j].ground;  // ground: T(x, P) brightness / pi
              const float spl = fmaf(ph.z, lz[e], fmaf(ph.y, ly[e], ph.x * lx[e]));
              const float ce = __builtin_amdgcn_fmed3f(
                  fmaf(-pc.se.A, fexp2(fmaf(-3.0f * 1.4426950408889634f, spl, pc.se.c)), pc.se.A), 0.0f, pc.se.top);
              float3 u;  // of height row 0: P is on the ground
              if (kELds) {
                const float s = __builtin_amdgcn_fractf(ce), i = ce - s;
                const Vec4 c = lds_read<Vec4>(lds_address(i, 16, ea_bytes));
                const Vec2 d = lds_read<Vec2>(lds_address(i, 8, eb_bytes));
                u = make_float3(fmaf(s, c.w, c.x), fmaf(s, d.x, c.y), fmaf(s, d.y, c.z));
              } else {
                const float ecol = lower_cell(ce, pc.se.top - 1.0f);
                u = lerp3(dE[(int)ecol], dE[(int)ecol + 1], ce - ecol);
              }
              v.x = fmaf(ground.x, u.x, v.x);
              v.y = fmaf(ground.y, u.y, v.y);
              v.z = fmaf(ground.z, u.z, v.z);
            }
            acc[e].x = fmaf(w.x, v.x, acc[e].x);
            acc[e].y = fmaf(w.y, v.y, acc[e].y);
            acc[e].z = fmaf(w.z, v.z, acc[e].z);
          }
        }
      };
      if (two) {
        if (to_ground) directions(std::true_type(), true);
        else directions(std::false_type(), true);
      } else {
        if (to_ground) directions(std::true_type(), false);
        else directions(std::false_type(), false);
      }
    }
    __syncthreads();
  }
  unsigned long long l4 = 0, l2 = 0;
#pragma unroll
  for (int e = 0; e < EPT; ++e)
    if (active && (part * EPT + e) * 64 + lane < count_e) {
      *(Rgb*)(out + 3 * (base + at[e])) = Rgb{acc[e].x, acc[e].y, acc[e].z};  // packed, (heading, sun elevation) order
      l4 += (unsigned long long)ndirs * (kMie ? 2 : 1);
      if (wc)
        for (int j = 0; j < ndirs; ++j) l2 += gh[j].ground.w != 0.f;
    }
  count(wc, 0, 0, l4, l2);
}

// dE' = surface-radiance of dS (atmosphere_lut.clj:89,93; atmosphere.clj:225-230): one workgroup per
// entry of the surface-radiance table, lanes over half-sphere directions, workgroup reduction.
// The half-sphere directions' geometry at every surface-radiance height (once per build).
__device__ __forceinline__ void surface_geometry_body(const DevParams& P, const Dir* __restrict__ dirs,
                                                                  int ndirs, unsigned blk) {
  const int idx = blk * blockDim.x + threadIdx.x;
  if (idx >= P.nE[0] * ndirs) return;
  const int ih = idx / ndirs, j = idx - ih * ndirs;
  const double r0 = index_to_radius(P.g, P.nE[0], ih);
  const Dir d = dirs[j];
  P.sgeo[idx] = make_float4((float)d.x, (float)d.y, (float)elevation_to_index(P.g, P.nS[1], r0, r0 * d.x, true),
                            (float)(d.x * d.w));  // (omega . normal) * quadrature weight, normal = (1 0 0)
}

__global__ void __launch_bounds__(kBlock) surface_geometry_kernel(const DevParams P, const Dir* __restrict__ dirs,
                                                                  int ndirs) {
  surface_geometry_body(P, dirs, ndirs, blockIdx.x);
}

// kFold: the entry's height and sun-elevation coordinates are the same for every direction, so the
// workgroup first folds those two dimensions of dS (and of the Mie strength) into an (elevation,
// heading) slab in LDS, NE x NA float4, and each direction interpolates the other two in it.
// One workgroup computes entry `entry` of the table; s_fold: kFold's LDS slab, s_red: one float3 per
// wavefront.
template <bool kFold>
__device__ __forceinline__ void surface_radiance_entry(const DevParams& P, int ndirs, const float4* __restrict__ dS,
                                                       const float4* __restrict__ mie, float4* __restrict__ out,
                                                       WorkCounters* wc, int entry, float4* s_fold, float3* s_red) {
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const int ih = entry / P.nE[1], il = entry - ih * P.nE[1];
  const double r0 = index_to_radius(P.g, P.nE[0], ih);
  const double s = index_to_sin_sun_elevation(P.nE[1], il);
  const double c = sqrt(fmax(0.0, 1 - s * s));
  const float lx = (float)s, ly = (float)c;
  const Lerp Lh = make_lerp((float)height_to_index(P.g, NH, r0), NH);
  const Lerp Ls = make_lerp((float)sun_elevation_to_index(NL, (r0 * s) / r0), NL);
  const float gm = P.g_mie;
  const float mk = 3.0f * (1.0f - gm * gm) / (8.0f * 3.14159265358979f * (2.0f + gm * gm)), ma = 1.0f + gm * gm,
              mb = 2.0f * gm;
  const float4* __restrict__ geo = P.sgeo + ih * ndirs;
  const int NEA = NE * NA;
  float4* s_m = s_fold + NEA;
  if (kFold) {
    const long long h0 = (long long)Lh.i0 * NE * NL * NA, h1 = (long long)Lh.i1 * NE * NL * NA;
    const int s0 = Ls.i0 * NA, s1 = Ls.i1 * NA;
    for (int c = threadIdx.x; c < NEA; c += blockDim.x) {
      const int e = c / NA, a = c - e * NA;
      const long long eo = (long long)e * NL * NA + a;
      const float3 u = mix3(mix3(ld3(dS, h0 + eo + s0), ld3(dS, h0 + eo + s1), Ls.s),
                            mix3(ld3(dS, h1 + eo + s0), ld3(dS, h1 + eo + s1), Ls.s), Lh.s);
      s_fold[c] = make_float4(u.x, u.y, u.z, 0.f);
      if (mie) {
        const float3 m = mix3(mix3(ld3(mie, h0 + eo + s0), ld3(mie, h0 + eo + s1), Ls.s),
                              mix3(ld3(mie, h1 + eo + s0), ld3(mie, h1 + eo + s1), Ls.s), Lh.s);
        s_m[c] = make_float4(m.x, m.y, m.z, 0.f);
      }
    }
    __syncthreads();
  }
  float3 acc = make_float3(0.f, 0.f, 0.f);
  for (int j = threadIdx.x; j < ndirs; j += blockDim.x) {
    const float4 g = geo[j];
    const float ol = fmaf(g.x, lx, g.y * ly);
    const Lerp Le = make_lerp(g.z, NE);
    const Lerp La = make_lerp((NA - 1) * ((1.0f + ol) * 0.5f), NA);
    float3 v = kFold ? lookup2(s_fold, NA, Le, La) : lookup4(dS, NE, NL, NA, Lh, Le, Ls, La);
    if (mie) {
      const float3 m = kFold ? lookup2(s_m, NA, Le, La) : lookup4(mie, NE, NL, NA, Lh, Le, Ls, La);
      const float y = __builtin_amdgcn_rsqf(fmaf(-mb, ol, ma));  // phase (atmosphere.clj:56-61), x^-3/2 = rsq(x)^3
      const float ph = mk * fmaf(ol, ol, 1.0f) * (y * y * y);
      v.x = fmaf(m.x, ph, v.x);
      v.y = fmaf(m.y, ph, v.y);
      v.z = fmaf(m.z, ph, v.z);
    }
    acc.x = fmaf(v.x, g.w, acc.x);
    acc.y = fmaf(v.y, g.w, acc.y);
    acc.z = fmaf(v.z, g.w, acc.z);
  }
  // wavefront reduction, then across the workgroup's wavefronts
  for (int off = 32; off > 0; off >>= 1) {
    acc.x += __shfl_down(acc.x, off, 64);
    acc.y += __shfl_down(acc.y, off, 64);
    acc.z += __shfl_down(acc.z, off, 64);
  }
  int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) s_red[wave] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float3 t = s_red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
      t.x += s_red[w].x; t.y += s_red[w].y; t.z += s_red[w].z;
    }
    out[entry] = make_float4(t.x, t.y, t.z, 0.f);
  }
  if (threadIdx.x == 0) count(wc, 0, 0, (unsigned long long)ndirs * (mie ? 2 : 1), 0);
}

template <bool kFold, bool kB>
__global__ void __launch_bounds__(kBlock) surface_radiance_kernel(const DevParams P0, const DevParams* __restrict__ PB,
                                                                  int ndirs, const float4* __restrict__ dS,
                                                                  const float4* __restrict__ mie,
                                                                  float4* __restrict__ out, WorkCounters* wc) {
  __shared__ float3 s_red[kBlock / 64];
  extern __shared__ float4 s_fold[];  // kFold: [NE x NA] dS, then [NE x NA] Mie strength
  const DevParams& P = params_of<kB>(P0, PB);
  surface_radiance_entry<kFold>(P, ndirs, atm_ptr<kB>(dS, P), atm_ptr<kB>(mie, P), atm_ptr<kB>(out, P), wc,
                                blockIdx.x, s_fold, s_red);
}

// f(backward(i)) re-sampling of interpolated tables (interpolate.clj:54-72 with interpolation-table).
// Lerps of forward(backward(i)) for 4D entry i = ((ih NE + ie) NL + is) NA + ia (atmosphere.clj:233-422).
// With ps / ss (nullable) also the entry's sun terms that the scatter kernels use (DevParams::sun_ps, sun_ss),
// from the same FP64 values.
__device__ __forceinline__ void resample4_lerps(const DevParams& P, int ih, int ie, int is, int ia, Lerp& Lh, Lerp& Le,
                                                Lerp& Ls, Lerp& La, float4* ps = nullptr, double2* ss = nullptr) {
  SFSIM_EXACT  // the reference's rounding (see geometry.hpp)
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  double r0 = index_to_radius(P.g, NH, ih);
  double se, ce;
  bool above;
  index_to_elevation(P.g, NE, r0, ie, se, ce, above);
  double sin_s = index_to_sin_sun_elevation(NL, is);
  double l0, l1, l2;
  index_to_sun_direction(NA, se, ce, sin_s, ia, l0, l1, l2);
  const double cs = sun_elevation_to_index(NL, (r0 * l0) / r0), vl = se * l0 + ce * l1;
  const double ca = sun_angle_to_index(NA, vl);
  Lh = make_lerp((float)height_to_index(P.g, NH, r0), NH);
  Le = make_lerp((float)elevation_to_index(P.g, NE, r0, r0 * se, above), NE);
  Ls = make_lerp((float)cs, NL);
  La = make_lerp((float)ca, NA);
  if (ps) *ps = make_float4((float)l0, (float)l1, (float)l2, (float)cs);
  if (ss) *ss = make_double2(vl, r0 * l0);
}

__device__ __forceinline__ Lerp lerp_of(int i0, float s, int N) {
  Lerp L;
  L.i0 = i0;
  L.i1 = min(i0 + 1, N - 1);
  L.s = s;
  return L;
}

// The 4D re-sampling lookups of a build, once (every accumulation and final table reads them).
__device__ __forceinline__ void resample_map_body(const DevParams& P, unsigned blk) {
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const long long n = (long long)NH * NE * NL * NA;
  const long long idx = (long long)blk * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const int ia = (int)(idx % NA);
  long long q = idx / NA;
  const int is = (int)(q % NL);
  q /= NL;
  const int ie = (int)(q % NE), ih = (int)(q / NE);
  Lerp Lh, Le, Ls, La;
  float4 ps;
  double2 ss;
  resample4_lerps(P, ih, ie, is, ia, Lh, Le, Ls, La, &ps, &ss);
  ((float4*)P.rmap)[idx] = make_float4(Lh.s, Le.s, Ls.s, La.s);
  if (P.sun_ps) {
    P.sun_ps[idx - (is * NA + ia) + ia * NL + is] = ps;
    P.sun_ss[idx] = ss;
  }
  ((ushort4*)(P.rmap + n * sizeof(float4)))[idx] =
      make_ushort4((unsigned short)Lh.i0, (unsigned short)Le.i0, (unsigned short)Ls.i0, (unsigned short)La.i0);
}

__global__ void __launch_bounds__(kBlock) resample_map_kernel(const DevParams P) {
  resample_map_body(P, blockIdx.x);
}

// The per-build jobs in one launch, job k over workgroups first[k] .. first[k + 1] - 1, the small
// long-running grids first so that they start at once: direction geometry, transmittance, E0, surface
// geometry, the sun table, ray geometry, the re-sampling map.  An absent job has an empty range.
struct PrologueArgs {
  PrologueJobs j;
  unsigned first[8];
};

// Batched (kB): each atmosphere's own jobs in its z slice; the shared geometry (surface geometry and the
// re-sampling and sun maps, which depend only on the planet and the grid) once, in slice 0.
template <bool kB>
__global__ void __launch_bounds__(kBlock) prologue_kernel(const DevParams P0, const DevParams* __restrict__ PB,
                                                          const PrologueArgs A) {
  const DevParams& P = params_of<kB>(P0, PB);
  const unsigned b = blockIdx.x;
  const bool shared = !kB || blockIdx.z == 0;
  if (b < A.first[1])
    direction_geometry_body(P, A.j.sdirs, A.j.sphere_n, atm_ptr<kB>((DirGeom*)A.j.geom, P), A.j.wc, b - A.first[0]);
  else if (b < A.first[2])
    transmittance_body(P, atm_ptr<kB>(A.j.T, P), A.j.wc, b - A.first[1]);
  else if (b < A.first[3])
    surface_radiance_base_body(P, atm_ptr<kB>(A.j.E0, P), A.j.wc, b - A.first[2]);
  else if (b < A.first[4]) {
    if (shared) surface_geometry_body(P, A.j.hdirs, A.j.half_n, b - A.first[3]);
  } else if (b < A.first[5])
    sun_depth_body(P, b - A.first[4]);
  else if (b < A.first[6])
    ray_geometry_body(P, A.j.wc, b - A.first[5]);
  else if (shared)
    resample_map_body(P, b - A.first[6]);
}

// Value at 4D entry idx of tab(a + b) (b nullable), or of tab(a + (b - c)) with c (each texel's
// difference formed first): the multilinear lookup at forward(backward(idx)), from the per-build map
// when there is one.
__device__ float3 resample4_value(const DevParams& P, const float4* __restrict__ a, const float4* __restrict__ b,
                                 long long idx, const float4* __restrict__ c) {
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const long long n = (long long)NH * NE * NL * NA;
  Lerp Lh, Le, Ls, La;
  if (P.rmap) {
    const float4 w = ((const float4*)P.rmap)[idx];
    const ushort4 i = ((const ushort4*)(P.rmap + n * sizeof(float4)))[idx];
    Lh = lerp_of(i.x, w.x, NH);
    Le = lerp_of(i.y, w.y, NE);
    Ls = lerp_of(i.z, w.z, NL);
    La = lerp_of(i.w, w.w, NA);
  } else {
    const int ia = (int)(idx % NA);
    long long q = idx / NA;
    const int is = (int)(q % NL);
    q /= NL;
    resample4_lerps(P, (int)(q / NE), (int)(q % NE), is, ia, Lh, Le, Ls, La);
  }
  float3 v;
  if (Lh.s == 0.0f && Le.s == 0.0f && Ls.s == 0.0f && La.s == 0.0f) {
    // the entry maps onto a grid point (every weight zero): the lookup is that point's value, bit for bit
    const long long g = (((long long)Lh.i0 * NE + Le.i0) * NL + Ls.i0) * NA + La.i0;
    v = ld3(a, g);
    if (b) {
      float3 w = ld3(b, g);
      if (c) {
        const float3 m = ld3(c, g);
        w = make_float3(w.x - m.x, w.y - m.y, w.z - m.z);
      }
      v.x += w.x; v.y += w.y; v.z += w.z;
    }
  } else {
    v = lookup4_skip([&](long long j) { return ld3(a, j); }, NE, NL, NA, Lh, Le, Ls, La);
    if (b) {
      const float3 w =
          c ? lookup4_skip(
                  [&](long long j) {
                    const float3 u = ld3(b, j), m = ld3(c, j);
                    return make_float3(u.x - m.x, u.y - m.y, u.z - m.z);
                  },
                  NE, NL, NA, Lh, Le, Ls, La)
            : lookup4_skip([&](long long j) { return ld3(b, j); }, NE, NL, NA, Lh, Le, Ls, La);
      v.x += w.x; v.y += w.y; v.z += w.z;
    }
  }
  return v;
}

// resample4_value(P, a, nullptr, idx) with the per-build map, in the same order of operations, one
// (height, elevation) cell at a time, and without the reads that a zero weight would mix in: mix3(u, v, 0)
// is u exactly, so a dimension whose weight is zero is not read (same result bit for bit).  Over the
// scatter grid of the full workload two thirds of the entries map onto a grid point, a quarter have only
// a heading weight (the clamped sun directions) and the height and sun-elevation weights are always zero:
// 1.4 reads per entry instead of 6.
__device__ float3 resample4_value_lean(const DevParams& P, const float4* __restrict__ a, long long idx) {
  const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
  const long long n = (long long)NH * NE * NL * NA;
  const float4 w = ((const float4*)P.rmap)[idx];
  const ushort4 i = ((const ushort4*)(P.rmap + n * sizeof(float4)))[idx];
  const Lerp Lh = lerp_of(i.x, w.x, NH), Le = lerp_of(i.y, w.y, NE), Ls = lerp_of(i.z, w.z, NL),
             La = lerp_of(i.w, w.w, NA);
  // entry offsets in 32 bits: a 4D table has fewer than 2^29 entries (validated on the host)
  auto row = [&](int h, int e, int s) {  // mixed over the heading
    const float4* c = a + ((unsigned)((h * NE + e) * NL + s)) * (unsigned)NA;
    const float3 u = ld3(c, La.i0);
    return La.s == 0.0f ? u : mix3(u, ld3(c, La.i1), La.s);
  };
  auto cell = [&](int h, int e) {  // mixed over the sun elevation
    const float3 u = row(h, e, Ls.i0);
    const float3 r = Ls.s == 0.0f ? u : mix3(u, row(h, e, Ls.i1), Ls.s);
    __builtin_amdgcn_sched_barrier(0);
    return r;
  };
  auto side = [&](int h) {  // mixed over the elevation
    const float3 u = cell(h, Le.i0);
    return Le.s == 0.0f ? u : mix3(u, cell(h, Le.i1), Le.s);
  };
  const float3 r0 = side(Lh.i0);
  return Lh.s == 0.0f ? r0 : mix3(r0, side(Lh.i1), Lh.s);
}

// Value at 2D entry idx of tab(a + b) (b nullable) for the transmittance (space 2) or
// surface-radiance (space 3) table.
__device__ float3 resample2_value(const DevParams& P, int space, const float4* __restrict__ a,
                                 const float4* __restrict__ b, long long idx) {
  SFSIM_EXACT  // the reference's rounding (see geometry.hpp)
  const int N0 = space == 2 ? P.nT[0] : P.nE[0], N1 = space == 2 ? P.nT[1] : P.nE[1];
  int i0 = (int)(idx / N1), i1 = (int)(idx % N1);
  double r0 = index_to_radius(P.g, N0, i0);
  double c1;
  if (space == 2) {
    double se, ce;
    bool above;
    index_to_elevation(P.g, N1, r0, i1, se, ce, above);
    c1 = elevation_to_index(P.g, N1, r0, r0 * se, above);
  } else {
    double s = index_to_sin_sun_elevation(N1, i1);
    c1 = sun_elevation_to_index(N1, (r0 * s) / r0);
  }
  Lerp L0 = make_lerp((float)height_to_index(P.g, N0, r0), N0);
  Lerp L1 = make_lerp((float)c1, N1);
  float3 v = lookup2_skip(a, N1, L0, L1);
  if (b) {
    float3 w = lookup2_skip(b, N1, L0, L1);
    v.x += w.x; v.y += w.y; v.z += w.z;
  }
  return v;
}

__device__ __forceinline__ void resample_entry(const DevParams& P, int space, const float4* __restrict__ a,
                                               const float4* __restrict__ b, float4* __restrict__ out4,
                                               float* __restrict__ out_rgb, int tiled, long long idx,
                                               const float4* __restrict__ c = nullptr) {
  float3 v;
  long long dst = idx;
  if (space == 4) {
    const int NH = P.nS[0], NE = P.nS[1], NL = P.nS[2], NA = P.nS[3];
    if (idx >= (long long)NH * NE * NL * NA) return;
    v = resample4_value(P, a, b, idx, c);
    if (tiled) {  // image.clj:299-312: row h * NL + s, column e * NA + a
      const int ia = (int)(idx % NA);
      long long q = idx / NA;
      const int is = (int)(q % NL);
      q /= NL;
      const int ie = (int)(q % NE), ih = (int)(q / NE);
      dst = (long long)(ih * NL + is) * (NE * NA) + (long long)ie * NA + ia;
    }
  } else {
    const int N0 = space == 2 ? P.nT[0] : P.nE[0], N1 = space == 2 ? P.nT[1] : P.nE[1];
    if (idx >= (long long)N0 * N1) return;
    v = resample2_value(P, space, a, b, idx);
  }
  if (out4) out4[idx] = make_float4(v.x, v.y, v.z, 0.f);
  if (out_rgb) {
    out_rgb[dst * 3 + 0] = v.x;
    out_rgb[dst * 3 + 1] = v.y;
    out_rgb[dst * 3 + 2] = v.z;
  }
}

template <bool kB>
__global__ void __launch_bounds__(kBlock) resample_kernel(const DevParams P0, const DevParams* __restrict__ PB,
                                                          int space, const float4* __restrict__ a,
                                                          const float4* __restrict__ b, float4* __restrict__ out4,
                                                          float* __restrict__ out_rgb, int tiled) {
  const DevParams& P = params_of<kB>(P0, PB);
  resample_entry(P, space, atm_ptr<kB>(a, P), atm_ptr<kB>(b, P), atm_ptr<kB>(out4, P), atm_ptr<kB>(out_rgb, P), tiled,
                 (long long)blockIdx.x * blockDim.x + threadIdx.x);
}

// Several independent re-samplings in one launch: job k takes workgroups first[k] .. first[k + 1] - 1.
struct ResampleJobs {
  ResampleJob job[kMaxResampleJobs];
  unsigned first[kMaxResampleJobs + 1];
  int count;
};

template <bool kB>
__global__ void __launch_bounds__(kBlock) resample_jobs_kernel(const DevParams P0, const DevParams* __restrict__ PB,
                                                               const ResampleJobs J) {
  const DevParams& P = params_of<kB>(P0, PB);
  int k = 0;
  while (k + 1 < J.count && blockIdx.x >= J.first[k + 1]) ++k;
  const ResampleJob& j = J.job[k];
  resample_entry(P, j.space, atm_ptr<kB>(j.a, P), atm_ptr<kB>(j.b, P), atm_ptr<kB>(j.out4, P),
                 atm_ptr<kB>(j.out_rgb, P), j.tiled, (long long)(blockIdx.x - J.first[k]) * blockDim.x + threadIdx.x,
                 atm_ptr<kB>(j.c, P));
}

__global__ void pack_rgb_kernel(const float4* __restrict__ in, float* __restrict__ out, long long count) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  float4 v = in[i];
  out[i * 3] = v.x;
  out[i * 3 + 1] = v.y;
  out[i * 3 + 2] = v.z;
}

__global__ void unpack_rgb_kernel(const float* __restrict__ in, float4* __restrict__ out, long long count) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  out[i] = make_float4(in[i * 3], in[i * 3 + 1], in[i * 3 + 2], 0.f);
}

// Packed RGB entries of [blocks][d0][d1] order in [blocks][d1][d0] order.
__global__ void transpose_rgb_kernel(const float* __restrict__ in, float* __restrict__ out, long long count, int d0,
                                     int d1) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;  // output entry
  if (i >= count) return;
  const long long q = i / d0, b = q / d1;
  const float* v = in + 3 * ((b * d0 + (i - q * d0)) * d1 + (q - b * d1));
  out[i * 3] = v[0];
  out[i * 3 + 1] = v[1];
  out[i * 3 + 2] = v[2];
}

__global__ void add4_kernel(const float4* __restrict__ a, const float4* __restrict__ b, float4* __restrict__ c,
                            long long count) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  float4 x = a[i], y = b[i];
  c[i] = make_float4(x.x + y.x, x.y + y.y, x.z + y.z, 0.f);
}

// Block maxima of |a + x| per channel: partial[block] (x, y, z).  Two passes without atomics (the
// second is one block over the partials), deterministic and free of memsets.
__device__ __forceinline__ float3 block_max3(float3 m, float3* red) {
  for (int off = 32; off > 0; off >>= 1) {
    m.x = fmaxf(m.x, __shfl_down(m.x, off, 64));
    m.y = fmaxf(m.y, __shfl_down(m.y, off, 64));
    m.z = fmaxf(m.z, __shfl_down(m.z, off, 64));
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
      m = make_float3(fmaxf(m.x, red[w].x), fmaxf(m.y, red[w].y), fmaxf(m.z, red[w].z));
  return m;  // valid in thread 0
}

__global__ void __launch_bounds__(kBlock) channel_max_kernel(const float4* __restrict__ a, const float4* __restrict__ b,
                                                             long long count, float4* __restrict__ partial) {
  __shared__ float3 red[kBlock / 64];
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  float3 m = make_float3(0.f, 0.f, 0.f);
  if (i < count) {
    float4 x = a[i], y = b[i];
    m = make_float3(fabsf(x.x + y.x), fabsf(x.y + y.y), fabsf(x.z + y.z));
  }
  m = block_max3(m, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = make_float4(m.x, m.y, m.z, 0.f);
}

// out[0] = maximum over the n partials (one block).
__global__ void __launch_bounds__(kBlock) max_partials_kernel(const float4* __restrict__ partial, int n,
                                                              float4* __restrict__ out) {
  __shared__ float3 red[kBlock / 64];
  float3 m = make_float3(0.f, 0.f, 0.f);
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    float4 v = partial[i];
    m = make_float3(fmaxf(m.x, v.x), fmaxf(m.y, v.y), fmaxf(m.z, v.z));
  }
  m = block_max3(m, red);
  if (threadIdx.x == 0) out[0] = make_float4(m.x, m.y, m.z, 0.f);
}

// Block maxima over entries and channels of |x - y| / max(|a + x|, floor_c), floor_c = fraction *
// channel max (cmax), in partial[block].x.
__global__ void __launch_bounds__(kBlock) residual_kernel(const float4* __restrict__ a, const float4* __restrict__ x,
                                                          const float4* __restrict__ y, long long count,
                                                          const float4* __restrict__ cmax, float fraction,
                                                          float4* __restrict__ partial) {
  __shared__ float3 red[kBlock / 64];
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  float r = 0.f;
  if (i < count) {
    const float4 c = cmax[0];
    float4 av = a[i], xv = x[i], yv = y[i];
    float f0 = fraction * c.x, f1 = fraction * c.y, f2 = fraction * c.z;
    r = fmaxf(fabsf(xv.x - yv.x) / fmaxf(fabsf(av.x + xv.x), fmaxf(f0, 1e-30f)),
              fmaxf(fabsf(xv.y - yv.y) / fmaxf(fabsf(av.y + xv.y), fmaxf(f1, 1e-30f)),
                    fabsf(xv.z - yv.z) / fmaxf(fabsf(av.z + xv.z), fmaxf(f2, 1e-30f))));
  }
  float3 m = block_max3(make_float3(r, r, r), red);
  if (threadIdx.x == 0) partial[blockIdx.x] = make_float4(m.x, 0.f, 0.f, 0.f);
}

__global__ void fill_zero_kernel(float* __restrict__ p, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

// Whether kernel K has no static LDS, so that its dynamic LDS begins at 0 as lds_read and lds_write take it; once per kernel.
template <auto K>
bool dynamic_lds_from_zero() {
  static std::atomic<bool> seen{false};
  if (seen.load()) return true;
  hipFuncAttributes a;
  if (hipFuncGetAttributes(&a, (const void*)K) != hipSuccess || a.sharedSizeBytes != 0) return false;
  seen.store(true);
  return true;
}

inline unsigned blocks_for(long long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

hipError_t launch_transmittance(const DevParams& P, float4* out, WorkCounters* wc, hipStream_t stream) {
  if (P.batch > 0) return hipErrorInvalidValue;  // batches run these jobs in launch_prologue
  long long n = (long long)P.nT[0] * P.nT[1];
  hipLaunchKernelGGL(transmittance_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, stream, P, out, wc);
  return hipGetLastError();
}

hipError_t launch_surface_radiance_base(const DevParams& P, float4* out, WorkCounters* wc, hipStream_t stream) {
  if (P.batch > 0) return hipErrorInvalidValue;  // batches run these jobs in launch_prologue
  long long n = (long long)P.nE[0] * P.nE[1];
  hipLaunchKernelGGL(surface_radiance_base_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, stream, P, out, wc);
  return hipGetLastError();
}

hipError_t launch_ray_geometry(const DevParams& P, WorkCounters* wc, hipStream_t stream) {
  if (P.batch > 0) return hipErrorInvalidValue;  // batches run these jobs in launch_prologue
  if (!P.ray_geo) return hipErrorInvalidValue;
  hipLaunchKernelGGL(ray_geometry_kernel, dim3(blocks_for((long long)ray_geo_samples(P))), dim3(kBlock), 0, stream, P,
                     wc);
  return hipGetLastError();
}

hipError_t launch_ray_items(const DevParams& P, hipStream_t stream) {
  if (P.batch > 0) return hipErrorInvalidValue;  // batches make them in launch_single_scatter
  if (!P.rs_items || !P.sun_ss || P.rs_groups > kMaxRsGroups) return hipErrorInvalidValue;
  if (P.rs_ts == 0) return hipSuccess;  // ray_scatter_ordered_kernel reads none
  hipLaunchKernelGGL(ray_items_kernel, dim3((unsigned)(P.nS[0] * P.nS[1])), dim3(kBlock),
                     sizeof(unsigned) * (size_t)P.nS[2] * P.nS[3], stream, P);
  return hipGetLastError();
}

RayItems ray_items_most(const int* nS, double radius, double height) {
  DevParams P{};
  for (int d = 0; d < 4; ++d) P.nS[d] = nS[d];
  P.g.R = radius;
  P.g.H = height;
  P.g.Rt = radius + height;
  P.g.rho_max = std::sqrt(sqr(P.g.Rt) - sqr(P.g.R));
  rs_split(P);
  const int NL = nS[2], NA = nS[3];
  RayItems r{0, P.rs_ts > 0 ? P.rs_slots : 0};
  for (int ray = 0; ray < nS[0] * nS[1]; ++ray) {
    double se, ce;
    bool above;
    index_to_elevation(P.g, nS[1], index_to_radius(P.g, nS[0], ray / nS[1]), ray % nS[1], se, ce, above);
    int count[kMaxRsGroups] = {};
    for (int is = 0; is < NL; ++is) {
      double last = 2.0, l0, l1, l2;
      for (int ia = 0; ia < NA; ++ia) {
        index_to_sun_direction(NA, se, ce, index_to_sin_sun_elevation(NL, is), ia, l0, l1, l2);
        const double vl = se * l0 + ce * l1;
        if (vl != last) {
          const float c = std::min(std::max((float)sun_angle_to_index(NA, vl), 0.0f), (float)(NA - 1));
          ++count[(int)c / P.rs_cols];
          if (c != (float)(int)c) ++count[((int)c + 1) / P.rs_cols];
        }
        last = vl;
      }
    }
    for (int g = 0; g < P.rs_groups; ++g) r.most = std::max(r.most, count[g]);
  }
  return r;
}

hipError_t launch_single_scatter(const DevParams& P, float4* rayleigh, float4* mie, WorkCounters* wc,
                                 hipStream_t stream, bool sun_table_built, bool ray_items) {
  unsigned rays = (unsigned)(P.nS[0] * P.nS[1]);
  // a batch runs the table path with the tables built by its prologue
  if (P.batch > 0 && (P.sun_rows <= 0 || !sun_table_built)) return hipErrorInvalidValue;
  if (P.sun_rows > 0) {
    if (!P.sun_depth || !P.ray_geo || !P.sun_ss || P.sun_rows < 2 || P.sun_cols < 2) return hipErrorInvalidValue;
    if (!sun_table_built)
      hipLaunchKernelGGL(sun_depth_kernel, dim3(blocks_for((long long)P.sun_rows * P.sun_cols)), dim3(kBlock), 0, stream,
                         P);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const RayGeoView V = ray_geo_view(P);
    const unsigned extra = ray_items && P.rs_ts > 0 ? rays : 0;
    const size_t shmem = std::max((size_t)P.ray_steps * (sizeof(double2) + 2 * sizeof(float4) + sizeof(float2)),
                                  extra ? (size_t)P.nS[2] * P.nS[3] * sizeof(unsigned) : 0);
    if (P.batch > 0)
      hipLaunchKernelGGL(single_scatter_table_kernel<true>, dim3(rays + extra, 1, P.batch), dim3(kSSTBlock), shmem, stream, P,
                         P.batch_params, V.th, V.T, V.ss, V.row, rayleigh, mie, (int)extra, wc);
    else
      hipLaunchKernelGGL(single_scatter_table_kernel<false>, dim3(rays + extra), dim3(kSSTBlock), shmem, stream, P,
                         P.batch_params, V.th, V.T, V.ss, V.row, rayleigh, mie, (int)extra, wc);
    return hipGetLastError();
  }
  if (ray_items) {
    const hipError_t e = launch_ray_items(P, stream);
    if (e != hipSuccess) return e;
  }
  const unsigned groups = (unsigned)((P.nS[2] * P.nS[3] + kSSEntries - 1) / kSSEntries);
  const unsigned most = 1u << 22, blocks = rays * groups;
  hipLaunchKernelGGL(single_scatter_kernel, dim3(std::min(blocks, most), (blocks + most - 1) / most), dim3(kSSEntries * kSSWaves),
                     single_scatter_shared_bytes(P.ray_steps), stream, P, rayleigh, mie, wc);
  return hipGetLastError();
}

hipError_t launch_direction_geometry(const DevParams& P, const Dir* dirs, int ndirs, void* geom, WorkCounters* wc,
                                    hipStream_t stream) {
  if (P.batch > 0) return hipErrorInvalidValue;  // batches run these jobs in launch_prologue
  long long n = (long long)P.nS[0] * ndirs;
  hipLaunchKernelGGL(direction_geometry_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, stream, P, dirs, ndirs,
                     (DirGeom*)geom, wc);
  return hipGetLastError();
}

size_t direction_geometry_bytes(const DevParams& P, int ndirs) { return sizeof(DirGeom) * (size_t)P.nS[0] * ndirs; }

// The split of a point-scatter launch.  Sun elevations in equal blocks of about 16 rows (a wavefront's 16-lane LDS
// phases then stay within a column: blocks of 8 or 32 rows took 4-30% longer), of at most 512 texels per slab;
// two entries per lane where that leaves 4 wavefronts per SIMD, one on smaller grids: 32 x 64 x 32 x 8 with 66
// directions 39 us with two and 48 with one, 19 x 45 x 20 x 7 with 38 directions 19.6 us with one and 20.3 with two.
//
// Weights and dE take LDS that the slabs leave of a quarter of a CU's 160 KiB (four wavefronts per SIMD).  dE stays in
// memory where it and the fewest weights leave fewer than four workgroups per CU (64 x 128 x 64 x 16, 66 directions, mean
// of the launches with and without the Mie strength: 768 columns, for which only the launch without it has room, 685 us,
// 727 with dE in LDS in both; 1024 columns, in memory in both, 884 against 957).  The weights of all directions where they
// fit, else those of as many latitude rings at a time as do, but at least of 64 directions and of the largest ring (a ring
// never lies in two batches).  32 x 64 x 32 x 8 with 808 directions: 342 us; 996 with the weights of all of them in LDS.
constexpr unsigned kCuLds = 163840;
constexpr int kPsWorkgroups = 4;

// The planes and, below or behind them, the other arrays: the weights of `dirs` directions, dE and omega.
static void ps_layout(PsPlan& p, int na, bool mie, bool omega, int nE1, int dirs) {
  const unsigned texels = ps_texels(p, na, mie);
  p.dirs = dirs;
  p.plane8 = (8 * texels + 15) & ~15u;
  unsigned below = 0;
  p.bytes = 2 * p.plane8 + 16 * texels;
  auto place = [&](unsigned size) {
    unsigned& at = below + size <= p.plane8 ? below : p.bytes;
    const unsigned place = at;
    at += (size + 15) & ~15u;
    return place;
  };
  p.weights = place(16u * p.rays * dirs);
  p.dE16 = place(p.e_lds ? 16u * nE1 : 0u);
  p.dE8 = place(p.e_lds ? 8u * nE1 : 0u);
  p.omega = place(omega ? 8u * dirs : 0u);
}

template <bool kMie>
static PsPlan point_scatter_plan(const DevParams& P, int ndirs, int sphere_steps, int& ept) {
  const int NL = P.nS[2], NA = P.nS[3], most = std::max(1, 512 / ((kMie ? 2 : 1) * NA));
  PsPlan p;
  p.sblocks = std::max({1, (NL + 8) / 16, (NL + most - 1) / most});
  p.rows = (NL + p.sblocks - 1) / p.sblocks;
  p.sblocks = (NL + p.rows - 1) / p.rows;
  p.pitch = std::max(2, p.rows);
  const int slots = (p.rows * NA + 63) / 64;  // at most 8
  const long long tiles = (long long)P.nS[0] * P.nS[1] * std::max(1, P.batch) * p.sblocks;
  ept = slots > 4 || (slots > 1 && tiles * ((slots + 1) / 2) >= 4096) ? 2 : 1;
  p.waves = (slots + ept - 1) / ept;
  p.rays = 4 / p.waves;
  p.eblocks = (P.nS[1] + p.rays - 1) / p.rays;
  const bool omega = ps_omega_in_lds(ept, kMie);
  const int least = std::min(ndirs, std::max(64, sphere_steps));
  auto fits = [&](int dirs, int workgroups) {
    ps_layout(p, NA, kMie, omega, P.nE[1], dirs);
    return p.bytes <= kCuLds / workgroups;
  };
  p.e_lds = true;
  p.e_lds = P.nE[1] <= 1024 && fits(least, kPsWorkgroups);
  int workgroups = kPsWorkgroups;
  while (workgroups > 1 && !fits(least, workgroups)) --workgroups;
  int dirs = ndirs;
  while (dirs > least && !fits(dirs, workgroups)) dirs = std::max(dirs - 16, least);
  ps_layout(p, NA, kMie, omega, P.nE[1], dirs);
  return p;
}

PointScatterLds point_scatter_lds(const int* nS, int nE1, int sphere_steps, int batch, bool mie) {
  DevParams P{};
  for (int d = 0; d < 4; ++d) P.nS[d] = nS[d];
  P.nE[1] = nE1;
  P.batch = batch;
  int ndirs = 0, ept = 1;
  for (int i = 0; i < sphere_steps >> 1; ++i) ndirs += sphere_ring_directions(0, sphere_steps, i);
  const PsPlan p = mie ? point_scatter_plan<true>(P, ndirs, sphere_steps, ept) : point_scatter_plan<false>(P, ndirs, sphere_steps, ept);
  PointScatterLds l;
  l.bytes = p.bytes;
  l.plane8 = p.plane8;
  l.plane16 = 2 * p.plane8;
  l.pitch = (unsigned)p.pitch;
  l.dirs = (unsigned)p.dirs;
  const unsigned at[4] = {p.weights, p.dE16, p.dE8, p.omega}, e = p.e_lds ? (unsigned)nE1 : 0u;
  const unsigned size[4] = {16u * p.rays * p.dirs, 16 * e, 8 * e, ps_omega_in_lds(ept, mie) ? 8u * p.dirs : 0u};
  for (int i = 0; i < 4; ++i) {
    l.at[i] = at[i];
    l.size[i] = size[i];
  }
  return l;
}

template <int EPT, bool kMie, bool kELds, bool kBatches>
static hipError_t point_scatter_as(const DevParams& P, const Dir* dirs, int ndirs, const PsRings& rings, const DirGeom* geom,
                                   const float4* dS, const float4* mie, const float4* dE, float* out, WorkCounters* wc,
                                   hipStream_t stream, const SrJob& sr, const PsPlan& plan) {
  const unsigned blocks = (unsigned)(P.nS[0] * plan.eblocks * plan.sblocks + sr.count);
  size_t shmem = plan.bytes;
  if (sr.count > 0) shmem = std::max(shmem, 4 * sizeof(float4) + sr_fold_bytes(P, sr.mie != nullptr));
  auto as = [&](auto kB) {
    constexpr auto kernel = point_scatter_kernel<EPT, kMie, kELds, decltype(kB)::value, kBatches>;
    if (!dynamic_lds_from_zero<kernel>()) return hipErrorInvalidKernelFile;
    hipLaunchKernelGGL(kernel, dim3(blocks, 1, std::max(P.batch, 1)), dim3(kBlock), shmem, stream, P, P.batch_params, dirs, geom,
                       ndirs, rings, dS, mie, dE, out, sr, plan, wc);
    return hipGetLastError();
  };
  return P.batch > 0 ? as(std::true_type()) : as(std::false_type());
}

template <bool kMie>
static hipError_t launch_point_scatter_as(const DevParams& P, const Dir* dirs, int ndirs, int sphere_steps, const PsRings& rings,
                                          const DirGeom* geom, const float4* dS, const float4* mie, const float4* dE,
                                          float* out, WorkCounters* wc, hipStream_t stream, const SrJob& sr) {
  int ept = 1;
  const PsPlan plan = point_scatter_plan<kMie>(P, ndirs, sphere_steps, ept);
  if (plan.bytes > kCuLds) return hipErrorInvalidValue;  // (no accepted shape)
  auto as = [&](auto entries, auto e_lds, auto batches) {
    return point_scatter_as<decltype(entries)::value, kMie, decltype(e_lds)::value, decltype(batches)::value>(
        P, dirs, ndirs, rings, geom, dS, mie, dE, out, wc, stream, sr, plan);
  };
  auto with_dE = [&](auto entries, auto batches) {
    return plan.e_lds ? as(entries, std::true_type(), batches) : as(entries, std::false_type(), batches);
  };
  auto with_entries = [&](auto batches) {
    return ept == 1 ? with_dE(std::integral_constant<int, 1>(), batches) : with_dE(std::integral_constant<int, 2>(), batches);
  };
  return plan.dirs < ndirs ? with_entries(std::true_type()) : with_entries(std::false_type());
}

hipError_t launch_point_scatter(const DevParams& P, const Dir* dirs, int ndirs, int sphere_steps, const void* geom,
                                const float4* dS, const float4* mie, const float4* dE, float* out, WorkCounters* wc,
                                hipStream_t stream, const SrJob* sr) {
  if (!P.sun_ps) return hipErrorInvalidValue;
  PsRings rings;
  rings.count = sphere_steps >> 1;
  if (rings.count < 1 || rings.count > kMaxRings) return hipErrorInvalidValue;
  rings.start[0] = 0;
  for (int i = 0; i < rings.count; ++i)
    rings.start[i + 1] = (unsigned short)(rings.start[i] + sphere_ring_directions(0, sphere_steps, i));
  if (rings.start[rings.count] != ndirs) return hipErrorInvalidValue;
  SrJob job{};
  if (sr) {
    if (!P.sgeo || !sr->out || !sr_fits_point_scatter(P, sr->mie != nullptr)) return hipErrorInvalidValue;
    job = *sr;
    job.count = P.nE[0] * P.nE[1];
  }
  if (mie)
    return launch_point_scatter_as<true>(P, dirs, ndirs, sphere_steps, rings, (const DirGeom*)geom, dS, mie, dE, out, wc, stream, job);
  return launch_point_scatter_as<false>(P, dirs, ndirs, sphere_steps, rings, (const DirGeom*)geom, dS, mie, dE, out, wc, stream, job);
}

// Sample segments per ray and group of columns: as many as let the workgroups of all rays be resident at once (four
// wavefronts per SIMD, 16 per CU of 256, which is what the kernel's registers allow), down to two samples each and
// within 64 KiB of LDS.  The 32 x 64 x 32 x 8 grid at 64 steps: 59 us with 2 segments, 76 with 1, 60 with 4 (two
// rounds); 19 x 45 x 20 x 7 at 51 steps: 24 us with 4, 38 with 5 (a second round of few), 30 with 2, 48 with 1.
// Workgroups of five wavefronts do not share a CU's four SIMDs out (24 x 25 x 32 x 8 at 64 steps: 35 us with 5, 25 with 4).
template <int TS, bool kExact>
static hipError_t launch_ray_scatter_as(const DevParams& P, const float* dJ, float4* out, WorkCounters* wc, hipStream_t stream,
                                        const RsAccum& acc) {
  const int groups = P.rs_groups;
  const long long rays = (long long)P.nS[0] * P.nS[1];
  int segs = (int)(16 / ((rays + 255) / 256)) / groups;
  segs = std::max(1, std::min(segs, P.ray_steps / 2));
  if (groups * segs == 5) --segs;
  while (segs > 1 && rs_shared_bytes<TS>(groups * segs, P.rs_slots, kExact) > 65536) --segs;
  const size_t shmem = rs_shared_bytes<TS>(groups * segs, P.rs_slots, kExact);
  const RayGeoView V = ray_geo_view(P);
  const dim3 block(64u * groups * segs);
  const dim3 grid((unsigned)rays + rs_surface_blocks(P, acc, block.x), 1, P.batch > 0 ? (unsigned)P.batch : 1u);
  auto as = [&](auto kB) {
    constexpr auto kernel = ray_scatter_kernel<TS, decltype(kB)::value, kExact>;
    if (!dynamic_lds_from_zero<kernel>()) return hipErrorInvalidKernelFile;
    hipLaunchKernelGGL(kernel, grid, block, shmem, stream, P, P.batch_params, dJ, V.th, V.T, V.rs, V.fold, P.rs_items, P.rs_entries,
                       P.rs_heads, out, acc, segs, wc);
    return hipGetLastError();
  };
  return P.batch > 0 ? as(std::true_type()) : as(std::false_type());
}

// In plain order: the fewest texels per lane (1, 2 or 4) with which the workgroups of all rays are resident at once, and as
// many samples at once as the wavefronts that are then left allow, within 64 KiB of LDS (28 bytes per texel and sample, and
// the ray's T).
template <bool kExact>
static hipError_t launch_ray_scatter_ordered(const DevParams& P, const float* dJ, float4* out, WorkCounters* wc,
                                             hipStream_t stream, const RsAccum& acc) {
  const long long rays = (long long)P.nS[0] * P.nS[1];
  const int NLA = P.nS[2] * P.nS[3], tiles = (NLA + 63) / 64, waves = std::max(1, (int)(16 / ((rays + 255) / 256)));
  int ts = 1;
  while (ts < 4 && (tiles + ts - 1) / ts > waves) ts *= 2;
  const int own = (tiles + ts - 1) / ts;  // wavefronts per sample
  const int samples = std::max(1, std::min({waves / own, (P.ray_steps + 1) / 2, 61440 / (28 * NLA)}));
  const size_t shmem = samples == 1 ? 2 * sizeof(float4) * (size_t)NLA
                                    : ((28 * (size_t)samples * NLA + 15) & ~(size_t)15) + sizeof(float4) * P.ray_steps;
  const RayGeoView V = ray_geo_view(P);
  const dim3 block(64u * own * samples);
  const dim3 grid((unsigned)rays + rs_surface_blocks(P, acc, block.x), 1, P.batch > 0 ? (unsigned)P.batch : 1u);
  auto as = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, shmem, stream, P, P.batch_params, dJ, V.th, V.T, V.rs, V.fold, out, acc, samples, wc);
  };
  auto with = [&](auto kB) {
    constexpr bool b = decltype(kB)::value;
    if (ts == 1) as(ray_scatter_ordered_kernel<1, b, kExact>);
    else if (ts == 2) as(ray_scatter_ordered_kernel<2, b, kExact>);
    else as(ray_scatter_ordered_kernel<4, b, kExact>);
  };
  P.batch > 0 ? with(std::true_type()) : with(std::false_type());
  return hipGetLastError();
}

hipError_t launch_ray_scatter(const DevParams& P, const float* dJ, float4* out, WorkCounters* wc, hipStream_t stream,
                              const RsAccum& acc, bool ordered) {
  if ((acc.S_in == nullptr) != (acc.S_out == nullptr) || (acc.E_out && !acc.dE)) return hipErrorInvalidValue;
  if (!P.ray_geo || !P.sun_ss || !P.rs_items || P.rs_groups < 1 || P.rs_groups > kMaxRsGroups) return hipErrorInvalidValue;
  const bool exact = P.nS[2] < kExactSunRows;
  if (ordered || P.rs_ts == 0)
    return exact ? launch_ray_scatter_ordered<true>(P, dJ, out, wc, stream, acc)
                 : launch_ray_scatter_ordered<false>(P, dJ, out, wc, stream, acc);
  auto as = [&](auto ts) {
    constexpr int TS = decltype(ts)::value;
    return exact ? launch_ray_scatter_as<TS, true>(P, dJ, out, wc, stream, acc)
                 : launch_ray_scatter_as<TS, false>(P, dJ, out, wc, stream, acc);
  };
  switch (P.rs_ts) {
    case 1: return as(std::integral_constant<int, 1>());
    case 2: return as(std::integral_constant<int, 2>());
    case 4: return as(std::integral_constant<int, 4>());
  }
  return hipErrorInvalidValue;
}

hipError_t launch_surface_geometry(const DevParams& P, const Dir* dirs, int ndirs, hipStream_t stream) {
  if (P.batch > 0) return hipErrorInvalidValue;  // batches run these jobs in launch_prologue
  if (!P.sgeo) return hipErrorInvalidValue;
  hipLaunchKernelGGL(surface_geometry_kernel, dim3(blocks_for((long long)P.nE[0] * ndirs)), dim3(kBlock), 0, stream, P,
                     dirs, ndirs);
  return hipGetLastError();
}

size_t sr_fold_bytes(const DevParams& P, bool mie) { return sizeof(float4) * (size_t)P.nS[1] * P.nS[3] * (mie ? 2 : 1); }

bool sr_fits_point_scatter(const DevParams& P, bool mie) { return sr_fold_bytes(P, mie) <= 16384; }

hipError_t launch_surface_radiance(const DevParams& P, int ndirs, const float4* dS, const float4* mie, float4* out,
                                   WorkCounters* wc, hipStream_t stream) {
  if (!P.sgeo) return hipErrorInvalidValue;
  unsigned entries = (unsigned)(P.nE[0] * P.nE[1]);
  const size_t fold = sr_fold_bytes(P, mie != nullptr);
  const dim3 grid(entries, 1, P.batch > 0 ? (unsigned)P.batch : 1u);
  const DevParams* PB = P.batch_params;
  if (P.batch > 0) {
    if (fold <= 65536)
      hipLaunchKernelGGL((surface_radiance_kernel<true, true>), grid, dim3(kBlock), fold, stream, P, PB, ndirs, dS, mie,
                         out, wc);
    else
      hipLaunchKernelGGL((surface_radiance_kernel<false, true>), grid, dim3(kBlock), 0, stream, P, PB, ndirs, dS, mie,
                         out, wc);
  } else {
    if (fold <= 65536)
      hipLaunchKernelGGL((surface_radiance_kernel<true, false>), grid, dim3(kBlock), fold, stream, P, PB, ndirs, dS, mie,
                         out, wc);
    else
      hipLaunchKernelGGL((surface_radiance_kernel<false, false>), grid, dim3(kBlock), 0, stream, P, PB, ndirs, dS, mie,
                         out, wc);
  }
  return hipGetLastError();
}

hipError_t launch_prologue(const DevParams& P, const PrologueJobs& J, hipStream_t stream) {
  if (!P.ray_geo || !P.rmap || (P.sun_rows > 0 && !P.sun_depth)) return hipErrorInvalidValue;
  if ((J.sdirs && !J.geom) || (J.hdirs && !P.sgeo) || !J.T || !J.E0) return hipErrorInvalidValue;
  PrologueArgs A;
  A.j = J;
  const long long counts[7] = {J.sdirs ? (long long)P.nS[0] * J.sphere_n : 0,
                               (long long)P.nT[0] * P.nT[1],
                               (long long)P.nE[0] * P.nE[1],
                               J.hdirs ? (long long)P.nE[0] * J.half_n : 0,
                               P.sun_rows > 0 ? (long long)P.sun_rows * P.sun_cols : 0,
                               (long long)ray_geo_samples(P),
                               (long long)P.nS[0] * P.nS[1] * P.nS[2] * P.nS[3]};
  A.first[0] = 0;
  for (int k = 0; k < 7; ++k) A.first[k + 1] = A.first[k] + blocks_for(counts[k]);
  if (P.batch > 0)
    hipLaunchKernelGGL(prologue_kernel<true>, dim3(A.first[7], 1, P.batch), dim3(kBlock), 0, stream, P,
                       P.batch_params, A);
  else
    hipLaunchKernelGGL(prologue_kernel<false>, dim3(A.first[7]), dim3(kBlock), 0, stream, P, P.batch_params, A);
  return hipGetLastError();
}

hipError_t launch_resample_map(const DevParams& P, hipStream_t stream) {
  if (P.batch > 0) return hipErrorInvalidValue;  // batches run these jobs in launch_prologue
  if (!P.rmap) return hipErrorInvalidValue;
  const long long n = (long long)P.nS[0] * P.nS[1] * P.nS[2] * P.nS[3];
  hipLaunchKernelGGL(resample_map_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, stream, P);
  return hipGetLastError();
}

static long long resample_count(const DevParams& P, int space) {
  return space == 4   ? (long long)P.nS[0] * P.nS[1] * P.nS[2] * P.nS[3]
         : space == 2 ? (long long)P.nT[0] * P.nT[1]
                      : (long long)P.nE[0] * P.nE[1];
}

hipError_t launch_resamples(const DevParams& P, const ResampleJob* jobs, int count, hipStream_t stream) {
  if (count < 1 || count > kMaxResampleJobs) return hipErrorInvalidValue;
  ResampleJobs J;
  J.count = count;
  J.first[0] = 0;
  for (int k = 0; k < kMaxResampleJobs; ++k) {
    J.job[k] = jobs[k < count ? k : 0];
    if (k < count) {
      if (jobs[k].space < 2 || jobs[k].space > 4 || !jobs[k].a || (jobs[k].c && (jobs[k].space != 4 || !jobs[k].b)))
        return hipErrorInvalidValue;
      J.first[k + 1] = J.first[k] + blocks_for(resample_count(P, jobs[k].space));
    }
  }
  if (P.batch > 0)
    hipLaunchKernelGGL(resample_jobs_kernel<true>, dim3(J.first[count], 1, P.batch), dim3(kBlock), 0, stream, P,
                       P.batch_params, J);
  else
    hipLaunchKernelGGL(resample_jobs_kernel<false>, dim3(J.first[count]), dim3(kBlock), 0, stream, P, P.batch_params,
                       J);
  return hipGetLastError();
}

hipError_t launch_resample(const DevParams& P, int space, const float4* a, const float4* b, float4* out4,
                           float* out_rgb, int tiled, hipStream_t stream) {
  const long long n = resample_count(P, space);
  if (P.batch > 0)
    hipLaunchKernelGGL(resample_kernel<true>, dim3(blocks_for(n), 1, P.batch), dim3(kBlock), 0, stream, P,
                       P.batch_params, space, a, b, out4, out_rgb, tiled);
  else
    hipLaunchKernelGGL(resample_kernel<false>, dim3(blocks_for(n)), dim3(kBlock), 0, stream, P, P.batch_params, space,
                       a, b, out4, out_rgb, tiled);
  return hipGetLastError();
}

hipError_t launch_add4(const float4* a, const float4* b, float4* c, long long count, hipStream_t stream) {
  hipLaunchKernelGGL(add4_kernel, dim3(blocks_for(count)), dim3(kBlock), 0, stream, a, b, c, count);
  return hipGetLastError();
}

size_t residual_scratch_floats(long long count) { return 4 * (2 + (size_t)blocks_for(count)); }

hipError_t launch_residual(const float4* a, const float4* x, const float4* y, long long count, float fraction,
                           float* scratch, hipStream_t stream) {
  const unsigned nb = blocks_for(count);
  float4* s4 = (float4*)scratch;  // [0] channel maxima, [1] result, [2 ..] block partials
  hipLaunchKernelGGL(channel_max_kernel, dim3(nb), dim3(kBlock), 0, stream, a, x, count, s4 + 2);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(max_partials_kernel, dim3(1), dim3(kBlock), 0, stream, s4 + 2, (int)nb, s4);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(residual_kernel, dim3(nb), dim3(kBlock), 0, stream, a, x, y, count, s4, fraction, s4 + 2);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(max_partials_kernel, dim3(1), dim3(kBlock), 0, stream, s4 + 2, (int)nb, s4 + 1);
  return hipGetLastError();
}

hipError_t launch_fill_zero(float* p, long long n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, stream, p, n);
  return hipGetLastError();
}

hipError_t launch_pack_rgb(const float4* in, float* out, long long count, hipStream_t stream) {
  hipLaunchKernelGGL(pack_rgb_kernel, dim3(blocks_for(count)), dim3(kBlock), 0, stream, in, out, count);
  return hipGetLastError();
}

hipError_t launch_transpose_rgb(const float* in, float* out, long long count, int d0, int d1, hipStream_t stream) {
  hipLaunchKernelGGL(transpose_rgb_kernel, dim3(blocks_for(count)), dim3(kBlock), 0, stream, in, out, count, d0, d1);
  return hipGetLastError();
}

hipError_t launch_unpack_rgb(const float* in, float4* out, long long count, hipStream_t stream) {
  hipLaunchKernelGGL(unpack_rgb_kernel, dim3(blocks_for(count)), dim3(kBlock), 0, stream, in, out, count);
  return hipGetLastError();
}

}  // namespace sfsim
