// xrh_interp.hip -- line integrals with the CPU caster's other sampling options.
//
// RayCasterLineIntCPU builds one ITK interpolator per range and evaluates it at every sample
// (lib/ray_cast/xregRayCastLineIntCPU.cpp:115-147, 270-277): nearest neighbour, windowed sinc
// (radius 4, Lanczos window, constant-zero boundary) or an order-3 B-spline besides the linear
// one; with an anti-aliasing factor k >= 1 it casts k rays per pixel through jittered detector
// indices and averages them (:150-183). The rays here are the reference's own float set-up
// (setup_ray_f32) and samples advance by repeated float addition, so every sample is taken at
// the reference's continuous index.
//
// Mapping onto CDNA4: each interpolator reads a grid built once per volume from the stored
// voxels, with an apron wide enough that no tap needs a bounds test:
//   - nearest neighbour and sinc: the float voxels with a zero apron of 4 (the sinc taps reach
//     floor(x) - 3 .. floor(x) + 4; zeros are the constant boundary);
//   - B-spline: the cubic B-spline coefficients in double (mirror-boundary recursive filter run
//     on the device, one thread per grid line per axis) with an apron of 2 holding the mirrored
//     coefficients, so the 4x4x4 taps are plain loads.
// Taps are x-contiguous; the many-tap interpolators read them from LDS, where a wave loads the box of
// grid elements its next samples reach.
// Sinc and B-spline weights and sums are FP64, as ITK evaluates them, and each sample is
// rounded to float once: the sums cancel (negative sinc lobes, B-spline coefficients that
// overshoot at edges), and a faint sample beside bright tissue would otherwise lose digits
// that a maximum-intensity projection keeps. Weights are separable and the sums run row ->
// plane -> volume. Grids go through buffer resources (a stray offset reads 0, never faults).
// One lane casts one ray over the same band-major, XCD-aware tile order as the trilinear
// kernels.
#include "xrh_internal.h"
#include "xrh_ray.h"

#include <climits>
#include <cmath>
#include <mutex>

namespace xrh {
namespace {

// The value the layout stores for voxel (x, y, z) (0 <= x < X, ...), as a float: every layout
// keeps the voxel itself (FP32, or its 16-bit rounding) as the first component of the entry
// at padded index (x + 1, y + 1, z + 1).
__device__ inline float layout_voxel(const VolDesc& d, int x, int y, int z)
{
  const int64_t a = x + 1, b = y + 1, c = z + 1;
  if (d.layout == kLayoutBrick) {
    const int64_t brick = (c >> 2) * (int64_t)d.pitch_z + (b >> 2) * (int64_t)d.pitch_y + (a >> 2);
    const int64_t local = (c & 3) * (kBrickEdge + 1) * kBrickEdge + (b & 3) * (kBrickEdge + 1) + (a & 3);
    return ((const float4*)d.data)[brick * kBrickFaces + local].x;
  }
  const int64_t e = a + (int64_t)d.pitch_y * b + (int64_t)d.pitch_z * c;
  if (d.layout == kLayoutLinear) {
    if (d.storage == XRH_F32) return ((const float*)d.data)[e];
    const uint32_t bits = ((const uint16_t*)d.data)[e];
    return (d.storage == XRH_F16) ? h2f(bits) : bf2f(bits);
  }
  if (d.layout == kLayoutQuad || d.layout == kLayoutFace) return ((const float4*)d.data)[e].x;
  if (d.layout == kLayoutCoef) return ((const float4*)d.data)[2 * e].x;
  const uint32_t bits = ((const uint4*)d.data)[e].x & 0xFFFFu;  // oct: corner (0, 0, 0) in the low half
  return (d.storage == XRH_F16) ? h2f(bits) : bf2f(bits);
}

// Voxels with a zero apron of A: one thread per grid element.
__global__ void voxel_grid_kernel(VolDesc d, int A, float* __restrict__ out, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t GX = d.X + 2 * A, GY = d.Y + 2 * A;
  const int x = (int)(i % GX) - A, y = (int)((i / GX) % GY) - A, z = (int)(i / (GX * GY)) - A;
  const bool in = x >= 0 && x < d.X && y >= 0 && y < d.Y && z >= 0 && z < d.Z;
  out[i] = in ? layout_voxel(d, x, y, z) : 0.0f;
}

// The voxels in double, x fastest: the B-spline filter's input.
__global__ void voxels_to_double_kernel(VolDesc d, double* __restrict__ out, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int x = (int)(i % d.X), y = (int)((i / d.X) % d.Y), z = (int)(i / ((int64_t)d.X * d.Y));
  out[i] = (double)layout_voxel(d, x, y, z);
}

// Cubic B-spline coefficients of one grid line in place (itk::BSplineDecompositionImageFilter,
// spline order 3: one pole z = sqrt(3) - 2, mirror boundaries -- Unser, "Splines: a perfect
// fit for signal and image processing", IEEE SPM 1999, Box 2). Line t of `lines` starts at
// element (t % na) * sa + (t / na) * sb and has n elements `stride` apart. The causal start
// sums the mirrored series over `horizon` terms when that is shorter than the line (terms
// below the 1e-10 tolerance), else in closed form over the whole line (z_n1 = z^(n-1)).
__global__ void bspline_lines_kernel(double* __restrict__ c, int64_t n, int64_t stride, int64_t lines,
                                     int64_t na, int64_t sa, int64_t sb, double z, int64_t horizon, double z_n1)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= lines || n == 1) return;
  double* p = c + (t % na) * sa + (t / na) * sb;
  const double gain = (1.0 - z) * (1.0 - 1.0 / z);
  for (int64_t i = 0; i < n; ++i) p[i * stride] *= gain;
  if (horizon < n) {
    double sum = p[0], zk = z;
    for (int64_t i = 1; i < horizon; ++i) {
      sum += zk * p[i * stride];
      zk *= z;
    }
    p[0] = sum;
  } else {
    const double iz = 1.0 / z;
    double zk = z, z2k = z_n1;
    double sum = p[0] + z2k * p[(n - 1) * stride];
    z2k *= z2k * iz;
    for (int64_t i = 1; i <= n - 2; ++i) {
      sum += (zk + z2k) * p[i * stride];
      zk *= z;
      z2k *= iz;
    }
    p[0] = sum / (1.0 - zk * zk);
  }
  for (int64_t i = 1; i < n; ++i) p[i * stride] += z * p[(i - 1) * stride];
  p[(n - 1) * stride] = (z / (z * z - 1.0)) * (z * p[(n - 2) * stride] + p[(n - 1) * stride]);
  for (int64_t i = n - 2; i >= 0; --i) p[i * stride] = z * (p[(i + 1) * stride] - p[i * stride]);
}

// ITK's mirror boundary for the B-spline support (BSplineInterpolateImageFunction::
// ApplyMirrorBoundaryConditions): one reflection about index 0 and one about n - 1. ITK leaves
// the range for lines shorter than 4; the clamp keeps those in it.
__device__ inline int64_t mirror_index(int64_t i, int64_t n)
{
  if (n == 1) return 0;
  if (i < 0) i = -i;
  if (i > n - 1) i = 2 * (n - 1) - i;
  return i < 0 ? 0 : (i > n - 1 ? n - 1 : i);
}

// B-spline coefficients with a mirrored apron of A.
__global__ void mirror_grid_kernel(const double* __restrict__ c, int X, int Y, int Z, int A,
                                   double* __restrict__ out, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t GX = X + 2 * A, GY = Y + 2 * A;
  const int64_t x = mirror_index(i % GX - A, X), y = mirror_index((i / GX) % GY - A, Y),
                z = mirror_index(i / (GX * GY) - A, Z);
  out[i] = c[x + (int64_t)X * (y + (int64_t)Y * z)];
}

// ---------------------------------------------------------------------------------------
// samplers

struct GridView {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t py, pz;
  int X, Y, Z;
};

__device__ inline float grid_load(const GridView& g, uint32_t e)
{
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(g.rsrc, (int)(e * 4u), 0, 0));
}

// Two doubles, or four floats, from grid element e on, as one 16-byte load.
__device__ inline void grid_load2_d(const GridView& g, uint32_t e, double* v)
{
  const auto r = __builtin_amdgcn_raw_buffer_load_b128(g.rsrc, (int)(e * 8u), 0, 0);
  v[0] = __hiloint2double((int)r[1], (int)r[0]);
  v[1] = __hiloint2double((int)r[3], (int)r[2]);
}

__device__ inline void grid_load4(const GridView& g, uint32_t e, float* v)
{
  const auto r = __builtin_amdgcn_raw_buffer_load_b128(g.rsrc, (int)(e * 4u), 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(r[i]);
}

// itk::Math::RoundHalfIntegerUp of a float index as ITK 5.1 computes it on x86-64 with SSE2:
// round-to-nearest-even of 2x + 0.5 (two float additions), then an arithmetic shift right.
__device__ inline int round_half_up(float x) { return ((int)__builtin_rintf(x + x + 0.5f)) >> 1; }

// itk::Math::Floor of a float index, the same way: round-to-nearest-even of 2x - 0.5, shifted.
__device__ inline int itk_floor(float x) { return ((int)__builtin_rintf(x + x - 0.5f)) >> 1; }

// LinearInterpolateImageFunction::EvaluateAtContinuousIndex (zero apron A = 4): per axis the
// base floor(x) clamped to the volume, the float fraction x - base, and an upper neighbour that
// falls back to the base past the last voxel (a fraction <= 0 weighs it 0); corners and lerps
// in double, x then y then z, rounded to float once. Only the anti-aliased casts use it: plain
// linear casts run the trilinear kernels.
__device__ inline float sample_linear(const GridView& g, float x, float y, float z)
{
  const float p[3] = {x, y, z};
  const int n[3] = {g.X, g.Y, g.Z};
  int b[3], u[3];
  double w[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int bk = min(max((int)floorf(p[k]), 0), n[k] - 1);
    const float dk = p[k] - (float)bk;
    b[k] = bk + 4;
    u[k] = ((bk + 1 > n[k] - 1) ? bk : bk + 1) + 4;
    w[k] = (dk > 0.0f) ? (double)dk : 0.0;
  }
  auto V = [&](int i, int j, int k) -> double {
    return (double)grid_load(g, (uint32_t)i + g.py * (uint32_t)j + g.pz * (uint32_t)k);
  };
  const double v000 = V(b[0], b[1], b[2]), v100 = V(u[0], b[1], b[2]);
  const double v010 = V(b[0], u[1], b[2]), v110 = V(u[0], u[1], b[2]);
  const double v001 = V(b[0], b[1], u[2]), v101 = V(u[0], b[1], u[2]);
  const double v011 = V(b[0], u[1], u[2]), v111 = V(u[0], u[1], u[2]);
  const double x00 = v000 + (v100 - v000) * w[0];
  const double x10 = v010 + (v110 - v010) * w[0];
  const double x01 = v001 + (v101 - v001) * w[0];
  const double x11 = v011 + (v111 - v011) * w[0];
  const double xx0 = x00 + (x10 - x00) * w[1];
  const double xx1 = x01 + (x11 - x01) * w[1];
  return (float)(xx0 + (xx1 - xx0) * w[2]);
}

// NearestNeighborInterpolateImageFunction::EvaluateAtContinuousIndex: the voxel at the rounded
// index (zero apron A = 4).
__device__ inline float sample_nn(const GridView& g, float x, float y, float z)
{
  const uint32_t ix = (uint32_t)(round_half_up(x) + 4), iy = (uint32_t)(round_half_up(y) + 4),
                 iz = (uint32_t)(round_half_up(z) + 4);
  return grid_load(g, ix + g.py * iy + g.pz * iz);
}

// Lanczos-4 windowed-sinc weights of the 8 taps floor(x) - 3 .. floor(x) + 4 at fractional
// offset d = x - floor(x): w[i] = sinc(t) * sinc(t / 4) at t = d + 3 - i, with sinc(u) =
// sin(pi u) / (pi u), which is WindowedSincInterpolateImageFunction's Sinc(t) times
// LanczosWindowFunction<4>(t). sin(pi t) = (-1)^k sin(pi d) and sin(pi t / 4) follows from
// sin(pi d / 4), cos(pi d / 4) and the angle k pi / 4 (k = 3 - i), so three sinpi/cospi calls
// give all eight. At d = 0 the weights are the unit impulse on tap 3, as ITK special-cases.
// Double precision throughout (d + 3 - i is exact).
__device__ inline void lanczos4_weights(double d, double w[8])
{
  if (d == 0.0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = (i == 3) ? 1.0 : 0.0;
    return;
  }
  constexpr double h = 0.70710678118654752440;  // sqrt(1/2)
  constexpr double kCos[8] = {-h, 0.0, h, 1.0, h, 0.0, -h, -1.0};  // cos(k pi / 4), k = 3 - i
  constexpr double kSin[8] = {h, 1.0, h, 0.0, -h, -1.0, -h, 0.0};  // sin(k pi / 4)
  constexpr double kFourOverPi2 = 0.40528473456935108578;         // 4 / pi^2
  const double s = sinpi(d), sq = sinpi(0.25 * d), cq = cospi(0.25 * d);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const double t = d + (double)(3 - i);
    const double st = ((3 - i) & 1) ? -s : s;
    const double sq_t = fma(sq, kCos[i], cq * kSin[i]);
    w[i] = (kFourOverPi2 * st * sq_t) / (t * t);
  }
}

// Uniform cubic B-spline weights of the taps floor(x) - 1 .. floor(x) + 2 at t = x - floor(x).
__device__ inline void bspline3_weights(double t, double w[4])
{
  const double t2 = t * t, t3 = t2 * t, u = 1.0 - t;
  w[0] = (u * u * u) * (1.0 / 6.0);
  w[1] = fma(0.5, t3, 2.0 / 3.0 - t2);
  w[2] = fma(-0.5, t3, fma(0.5, t2, fma(0.5, t, 1.0 / 6.0)));
  w[3] = t3 * (1.0 / 6.0);
}

// The interpolators with many taps. Per axis a position's taps are the kN grid elements from
// floor(p) + 1 on (the voxel grid's apron of 4 puts tap floor(p) - 3 there, the coefficients' apron
// of 2 tap floor(p) - 1), with separable weights.
//
// WindowedSincInterpolateImageFunction<Image<float,3>, 4, LanczosWindowFunction<4>,
// ConstantBoundaryCondition>::EvaluateAtContinuousIndex
struct SincTaps {
  static constexpr int kN = 8;
  using Elem = float;
  __device__ static int cell(float p) { return itk_floor(p); }
  __device__ static void weights(float p, int cell, double (&w)[8]) { lanczos4_weights((double)p - (double)cell, w); }
  __device__ static void row(const GridView& g, uint32_t e, float (&v)[8])
  {
    grid_load4(g, e, v);
    grid_load4(g, e + 4u, v + 4);
  }
};

// BSplineInterpolateImageFunction (order 3)::EvaluateAtContinuousIndex
struct BSplineTaps {
  static constexpr int kN = 4;
  using Elem = double;
  __device__ static int cell(float p) { return (int)floorf(p); }
  __device__ static void weights(float p, int cell, double (&w)[4]) { bspline3_weights((double)(p - (float)cell), w); }
  __device__ static void row(const GridView& g, uint32_t e, double (&v)[4])
  {
    grid_load2_d(g, e, v);
    grid_load2_d(g, e + 2u, v + 2);
  }
};

// The sample at p: the taps' rows (row(c, j, k, v): row j of plane k for the cell c) are summed along
// x into their plane's sum and those into the sample's, in double and in that order.
template <class T, class Row>
__device__ __forceinline__ float sample_taps(const float (&p)[3], Row row)
{
  constexpr int kN = T::kN;
  double w[3][kN];
  int c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    c[k] = T::cell(p[k]);
    T::weights(p[k], c[k], w[k]);
  }
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < kN; ++k) {
    double plane = 0.0;
#pragma unroll
    for (int j = 0; j < kN; ++j) {
      typename T::Elem v[kN];
      row(c, j, k, v);
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < kN; ++i) sum = fma(w[0][i], (double)v[i], sum);
      plane = fma(w[1][j], sum, plane);
    }
    acc = fma(w[2][k], plane, acc);
  }
  return (float)acc;
}

// ---------------------------------------------------------------------------------------
// anti-aliasing jitter

// The SplitMix64 output function (Steele, Lea and Flood, "Fast splittable pseudorandom number
// generators", OOPSLA 2014).
__device__ inline uint64_t splitmix64(uint64_t state)
{
  uint64_t z = state;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Jitter of ray k of pixel `pixel` (the reference's range index: projection * rows * cols + row
// * cols + col), component 0 (column) or 1 (row): uniform on [-0.5, 0.5) in steps of 2^-24, as
// std::uniform_real_distribution<float>(-0.5, 0.5) draws it (xregRayCastLineIntCPU.cpp:162-174).
// The reference seeds a Mersenne Twister from std::random_device, so its jitter is never
// reproducible; here it is a pure function of (seed, pixel, ray, component): counter-based
// SplitMix64, the same on the device and in any process.
__device__ inline float aa_jitter(uint64_t seed, uint64_t pixel, int k, int comp)
{
  const uint64_t counter = (pixel << 17) | ((uint64_t)k << 1) | (uint64_t)comp;
  const uint64_t h = splitmix64(seed + 0x9E3779B97F4A7C15ull * (counter + 1));
  return (float)(uint32_t)(h >> 40) * 0x1.0p-24f - 0.5f;
}

// Minimum over the wave, in every lane.
__device__ inline int wave_min(int v)
{
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xf, 0xf, false));   // lanes ^ 1
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xf, 0xf, false));   // lanes ^ 2
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false));  // the other half of 8
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xf, 0xf, false));  // the other half of 16
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xf, 0xf, false));  // the rows before
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xf, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}

// The sum or maximum of one ray's samples for the interpolators with many taps. The 64 rays of a
// workgroup of one wave go through the volume together, kWin samples at a time; the box of grid
// elements that these samples' taps lie in is loaded into LDS once, 16 bytes per lane straight from
// the buffer load, and the samples take their rows from there: neighbouring rays and samples share
// nearly all of them, and gathered from memory they cost 16 clocks of a CU and more per 16 bytes of
// 64 lanes, whatever is shared.
// Boxes that do not fit (rays further apart) are tried at half the window, then gathered.
// Measured, us, 128 x 128 x 96 voxels of 2 mm, 1 mm steps, against rays gathered one by one in blocks
// of four waves: B-spline 4 images of 192 x 192 864 -> 465 (LDS reads 75% of the kernel's clocks, VALU
// 42%, mostly FP64), 16 images 3400 -> 1550, 16 of 96 x 96 1120 -> 650, 32 of 48 x 48 1290 -> 740; sinc
// 4530 -> 3220, 5190 -> 3870 (96 x 96), 6260 -> 3440. Window: 8 samples 490, 16 465, 32 590; evaluating
// consecutive samples with the same taps together 445, sinc 3830 (lanes wait for each other); reading
// four rows ahead 455. LDS 8 / 10 / 16 KB: 96 x 96 685 / 660 / 628, 16 images 1556 / 1530 / 1650.
constexpr int kTapsLds = 12288;

template <class T, int kOp>
__device__ __forceinline__ float cast_taps(const GridView& g, const Ray& ray, bool inside)
{
  using E = typename T::Elem;
  constexpr int kPer = 16 / (int)sizeof(E);  // elements per 16-byte lane
  constexpr int kWin = 16, kBudget = kTapsLds / (int)sizeof(E);
  extern __shared__ __attribute__((aligned(16))) char taps_lds[];
  E* lds = (E*)taps_lds;
  const int lane = threadIdx.x;
  const int GX = (int)g.py, GY = (int)(g.pz / g.py), GZ = g.Z + (GY - g.Y);
  const int n = inside ? ray.n : -1;
  float acc = (kOp == XRH_LINE_INT_SUM) ? 0.0f : -3.402823466e+38f;
  float p[3] = {ray.sx, ray.sy, ray.sz};
  const float d[3] = {ray.dx, ray.dy, ray.dz};
  int win = kWin;
  for (int i = 0; __any(i <= n);) {
    // the box of the next `win` samples, in grid elements; the margin covers the rounding of the
    // positions, at most one per addition
    int lo[3], w[3], rows = 0, lpr = 0;
    bool fits = false;
    for (win = kWin;; win >>= 1) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float e = fmaf((float)min(win - 1, n - i), d[k], p[k]);
        const float m = fmaf(fmaxf(fabsf(p[k]), fabsf(e)), 2.0e-6f, 0.01f);
        const int l = wave_min(i <= n ? (int)floorf(fminf(p[k], e) - m) : 0x3fffffff);
        const int h = -wave_min(i <= n ? -(int)floorf(fmaxf(p[k], e) + m) : 0x3fffffff);
        const int G = k == 0 ? GX : (k == 1 ? GY : GZ);
        lo[k] = min(max(l + 1, 0), G - 1);
        w[k] = min(max(h + T::kN, lo[k]), G - 1) - lo[k] + 1;
      }
      lpr = (w[0] + kPer - 1) / kPer;
      rows = lpr > 0 && lpr <= 64 ? 64 / lpr : 0;
      fits = rows > 0 && w[1] <= kBudget && w[2] <= kBudget && lpr * kPer * w[1] <= kBudget &&
             lpr * kPer * w[1] * w[2] <= kBudget;
      if (fits || win <= kWin / 2) break;
    }
    if (!fits) win = kWin;
    const int sy = lpr * kPer, sz = sy * w[1];
    const int stop = min(i + win - 1, n);
    if (fits) {
      __syncthreads();  // the previous box has been read
      const int sub = lane / lpr;
      const uint32_t lane_off = ((uint32_t)sub * g.py + (uint32_t)(lane - sub * lpr) * kPer) * (uint32_t)sizeof(E);
      for (int z = 0; z < w[2]; ++z)
        for (int y = 0; y < w[1]; y += rows) {
          const uint32_t at = (uint32_t)(lo[2] + z) * g.pz + (uint32_t)(lo[1] + y) * g.py + (uint32_t)lo[0];
          if (sub < min(rows, w[1] - y)) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(g.rsrc, (__attribute__((address_space(3))) void*)(lds + z * sz + y * sy),
                                                     16, (int)(lane_off + at * (uint32_t)sizeof(E)), 0, 0, 0);
          }
        }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the clobber: no read of the box above the wait)
      __syncthreads();
    }
    const int org = lo[0] + sy * lo[1] + sz * lo[2] - (1 + sy + sz);
    for (; i <= stop; ++i) {
      float v;
      if (fits) {
        v = sample_taps<T>(p, [&](const int (&c)[3], int j, int k, E (&v)[T::kN]) {
          const E* r = lds + (c[0] + sy * (c[1] + j) + sz * (c[2] + k) - org);
#pragma unroll
          for (int t = 0; t < T::kN; ++t) v[t] = r[t];
        });
      } else {
        v = sample_taps<T>(p, [&](const int (&c)[3], int j, int k, E (&v)[T::kN]) {
          T::row(g, (uint32_t)(c[0] + 1) + g.py * (uint32_t)(c[1] + 1 + j) + g.pz * (uint32_t)(c[2] + 1 + k), v);
        });
      }
      acc = line_op<kOp>(acc, v);
#pragma unroll
      for (int k = 0; k < 3; ++k) p[k] = p[k] + d[k];
    }
  }
  return acc;
}

// The sum or maximum of one ray's samples for the interpolators with few taps.
template <int kOp, int kInterp>
__device__ __forceinline__ float cast_few(const GridView& g, const Ray& ray)
{
  float acc = (kOp == XRH_LINE_INT_SUM) ? 0.0f : -3.402823466e+38f;
  float px = ray.sx, py = ray.sy, pz = ray.sz;
  for (int i = 0; i <= ray.n; ++i) {
    acc = line_op<kOp>(acc, kInterp == XRH_INTERP_LINEAR ? sample_linear(g, px, py, pz) : sample_nn(g, px, py, pz));
    px = px + ray.dx;
    py = py + ray.dy;
    pz = pz + ray.dz;
  }
  return acc;
}

// One lane = one pixel: `rays` rays (1 without anti-aliasing), each the reference's float set-up
// through the (jittered) detector index, n + 1 samples at positions advanced by repeated float
// addition (:270-277), times the step; the rays' values are averaged as the reference does
// (aa_sum += sum * (1 / rays), :281-282) and stored as store_pixel does (RayCasterCPU::
// pre_compute semantics: ACCUM onto the buffer / background, REPLACE onto fill, :285). A workgroup
// is one wave, an 8 x 8 quadrant of a tile.
constexpr int kInterpThreads = 64, kInterpSplit = kThreads / kInterpThreads;

template <int kOp, int kInterp>
__global__ __launch_bounds__(kInterpThreads) void drr_interp_kernel(
    const DrrItem* __restrict__ items, const uint32_t* __restrict__ band_start, int64_t num_items,
    int bands, float* __restrict__ out, int accumulate, float fill, InterpGrid grid, int aa_rays,
    uint64_t aa_seed)
{
  const TileRef tr = decode_tile(band_start, num_items, bands, items, 1, kInterpSplit);
  if (!tr.valid) return;
  const DrrItem& it = items[tr.item];
  const int part = (int)(blockIdx.x / (uint32_t)bands) & (kInterpSplit - 1), lane = threadIdx.x;
  const int col = tr.tx * kTile + (part & 1) * 8 + (lane & 7), row = tr.ty * kTile + (part >> 1) * 8 + (lane >> 3);
  const bool inside = col < it.cam.cols && row < it.cam.rows;
  if (!__any(inside)) return;
  GridView g;
  g.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(grid.data), (short)0, (int)grid.bytes, 0x00020000);
  g.py = grid.py;
  g.pz = grid.pz;
  g.X = grid.X;
  g.Y = grid.Y;
  g.Z = grid.Z;
  const int64_t o = it.out_off + (int64_t)row * it.cam.cols + col;
  const int rays = aa_rays > 0 ? aa_rays : 1;
  const float inv = 1.0f / (float)rays;
  float aa_sum = 0.0f;
  for (int k = 0; k < rays; ++k) {
    float c = (float)col, r = (float)row;
    if (aa_rays > 0) {
      c = c + aa_jitter(aa_seed, (uint64_t)o, k, 0);
      r = r + aa_jitter(aa_seed, (uint64_t)o, k, 1);
    }
    const Ray ray = setup_ray_f32(it, c, r);
    float acc;
    if constexpr (kInterp == XRH_INTERP_SINC) acc = cast_taps<SincTaps, kOp>(g, ray, inside);
    else if constexpr (kInterp == XRH_INTERP_BSPLINE) acc = cast_taps<BSplineTaps, kOp>(g, ray, inside);
    else acc = cast_few<kOp, kInterp>(g, ray);
    if (ray.n >= 0) acc = acc * it.step;
    aa_sum = aa_sum + acc * inv;
  }
  if (!inside) return;
  const float prev = accumulate ? out[o] : fill;
  if constexpr (kOp == XRH_LINE_INT_SUM) out[o] = prev + aa_sum; else out[o] = (prev < aa_sum) ? aa_sum : prev;
}

template <int kOp, int kInterp>
void launch_interp_kernel(const DrrLaunch& L, const InterpGrid& g, dim3 grid, hipStream_t s, int accumulate,
                          int aa_rays, uint64_t aa_seed)
{
  const int lds = (kInterp == XRH_INTERP_SINC || kInterp == XRH_INTERP_BSPLINE) ? kTapsLds : 0;
  hipLaunchKernelGGL((drr_interp_kernel<kOp, kInterp>), grid, dim3(kInterpThreads), lds, s, L.items_dev, L.band_start_dev,
                     L.num_items, L.bands, L.out, accumulate, L.fill, g, aa_rays, aa_seed);
}

template <int kOp>
void launch_interp_op(const DrrLaunch& L, const InterpGrid& g, int32_t interp, dim3 grid, hipStream_t s,
                      int accumulate, int aa_rays, uint64_t aa_seed)
{
  switch (interp) {
    case XRH_INTERP_LINEAR:
      launch_interp_kernel<kOp, XRH_INTERP_LINEAR>(L, g, grid, s, accumulate, aa_rays, aa_seed);
      break;
    case XRH_INTERP_NN:
      launch_interp_kernel<kOp, XRH_INTERP_NN>(L, g, grid, s, accumulate, aa_rays, aa_seed);
      break;
    case XRH_INTERP_SINC:
      launch_interp_kernel<kOp, XRH_INTERP_SINC>(L, g, grid, s, accumulate, aa_rays, aa_seed);
      break;
    default:
      launch_interp_kernel<kOp, XRH_INTERP_BSPLINE>(L, g, grid, s, accumulate, aa_rays, aa_seed);
      break;
  }
}

std::mutex& grid_mutex()
{
  static std::mutex mu;
  return mu;
}

}  // namespace

const InterpGrid& interp_prepare(xrh_volume* v, int32_t interp)
{
  XRH_REQUIRE(v, "null volume");
  XRH_REQUIRE(interp >= XRH_INTERP_LINEAR && interp <= XRH_INTERP_BSPLINE, "bad interpolation method");
  const int k = (interp == XRH_INTERP_BSPLINE) ? kGridBSpline : kGridVoxels;
  std::lock_guard<std::mutex> lk(grid_mutex());
  if (v->grid_mem[k]) return v->grid[k];
  xrh_ctx* ctx = v->ctx;
  const VolDesc& d = v->desc;
  const int A = (k == kGridBSpline) ? 2 : 4;
  const int64_t X = d.X, Y = d.Y, Z = d.Z;
  const int64_t GX = X + 2 * A, GY = Y + 2 * A, GZ = Z + 2 * A;
  const int64_t n = GX * GY * GZ;
  const uint64_t esize = (k == kGridBSpline) ? 8 : 4;
  const uint64_t bytes = (uint64_t)n * esize;
  // grid offsets are 32-bit (buffer loads) and the tap arithmetic is unsigned 32-bit
  XRH_REQUIRE(bytes < 0xFFFFF000ull, "interpolation grid exceeds 4 GiB");
  const int threads = 256;
  void* mem = ctx_alloc(ctx, bytes);
  double* coef = nullptr;
  try {
    if (k == kGridVoxels) {
      hipLaunchKernelGGL(voxel_grid_kernel, dim3((unsigned)((n + threads - 1) / threads)), dim3(threads), 0,
                         ctx->stream, d, A, (float*)mem, n);
      XRH_HIP_CHECK(hipGetLastError());
    } else {
      const int64_t nv = X * Y * Z;
      coef = (double*)ctx_alloc(ctx, (uint64_t)nv * 8);
      hipLaunchKernelGGL(voxels_to_double_kernel, dim3((unsigned)((nv + threads - 1) / threads)), dim3(threads), 0,
                         ctx->stream, d, coef, nv);
      XRH_HIP_CHECK(hipGetLastError());
      const double z = std::sqrt(3.0) - 2.0;
      const int64_t horizon = (int64_t)std::ceil(std::log(1.0e-10) / std::log(std::fabs(z)));
      const int64_t len[3] = {X, Y, Z}, stride[3] = {1, X, X * Y};
      const int64_t na[3] = {Y * Z, X, X * Y}, sa[3] = {X, 1, 1}, sb[3] = {0, X * Y, 0};
      for (int ax = 0; ax < 3; ++ax) {  // x, then y, then z, as ITK filters the dimensions
        const int64_t lines = nv / len[ax];
        const int lt = 64;
        hipLaunchKernelGGL(bspline_lines_kernel, dim3((unsigned)((lines + lt - 1) / lt)), dim3(lt), 0, ctx->stream,
                           coef, len[ax], stride[ax], lines, na[ax], sa[ax], sb[ax], z, horizon,
                           std::pow(z, (double)(len[ax] - 1)));
        XRH_HIP_CHECK(hipGetLastError());
      }
      hipLaunchKernelGGL(mirror_grid_kernel, dim3((unsigned)((n + threads - 1) / threads)), dim3(threads), 0,
                         ctx->stream, (const double*)coef, (int)X, (int)Y, (int)Z, A, (double*)mem, n);
      XRH_HIP_CHECK(hipGetLastError());
    }
    XRH_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    if (coef) ctx_free(ctx, coef);
    coef = nullptr;
  } catch (...) {
    (void)hipStreamSynchronize(ctx->stream);
    if (coef) ctx_free(ctx, coef);
    ctx_free(ctx, mem);
    throw;
  }
  v->grid_mem[k] = mem;
  v->grid_bytes[k] = bytes;
  InterpGrid& g = v->grid[k];
  g.data = mem;
  g.bytes = (uint32_t)bytes;
  g.py = (uint32_t)GX;
  g.pz = (uint32_t)(GX * GY);
  g.apron = A;
  g.X = (int32_t)X;
  g.Y = (int32_t)Y;
  g.Z = (int32_t)Z;
  return g;
}

void launch_drr_interp(const DrrLaunch& L, const InterpGrid& g, int32_t interp, int32_t aa_rays, uint64_t aa_seed,
                       hipStream_t s)
{
  if (L.num_items <= 0 || L.max_band_tiles <= 0) return;
  XRH_REQUIRE(interp >= XRH_INTERP_LINEAR && interp <= XRH_INTERP_BSPLINE, "bad interpolation method");
  XRH_REQUIRE(aa_rays >= 0 && aa_rays <= XRH_MAX_AA_RAYS, "anti-aliasing rays out of range");
  XRH_REQUIRE(g.data && g.apron == ((interp == XRH_INTERP_BSPLINE) ? 2 : 4), "interpolation grid not prepared");
  const int64_t nblocks = L.max_band_tiles * L.bands * kInterpSplit;
  XRH_REQUIRE(nblocks < (int64_t)INT32_MAX, "too many DRR tiles in one launch");
  const dim3 grid((unsigned)nblocks);
  const int accumulate = (L.store == XRH_STORE_ACCUM) ? 1 : 0;
  if (L.kernel == XRH_LINE_INT_SUM) launch_interp_op<XRH_LINE_INT_SUM>(L, g, interp, grid, s, accumulate, aa_rays, aa_seed);
  else launch_interp_op<XRH_LINE_INT_MAX>(L, g, interp, grid, s, accumulate, aa_rays, aa_seed);
  XRH_HIP_CHECK(hipGetLastError());
}

}  // namespace xrh
