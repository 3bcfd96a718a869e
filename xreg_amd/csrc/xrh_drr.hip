// xrh_drr.hip -- line-integral DRR kernels for gfx950.
//
// Semantics follow RayCasterLineIntCPU::compute / ComputeLineInts
// (lib/ray_cast/xregRayCastLineIntCPU.cpp:105-349):
//   per ray: detector point (CameraModel::ind_pt_to_phys_det_pt), pinhole and direction in
//   volume index space, slab intersection against [0, N-1] limited to the source->detector
//   segment, 1e-3 parametric nudge, n = floor(chord / step_len), n+1 trilinear samples
//   accumulated with SUM or MAX, times the physical step; stored with the same operator.
//
// Mapping onto CDNA4:
//   - one lane = one ray; a 256-lane workgroup owns a 16x16 detector tile and each of its
//     four wave64s an 8x8 sub-tile, so neighbouring lanes march neighbouring pixels and
//     their gathers hit the same cache lines;
//   - workgroups are ordered band-major and swizzled so that the workgroups that the
//     dispatcher sends to one XCD (blockIdx mod 8) all work on the same band of detector
//     rows across every projection: each XCD's L2 then holds one slab of the volume;
//   - the volume sits in HBM in an edge-padded layout read through buffer loads
//     (hardware range check: a stray offset returns 0, it can never fault); the quad (f32)
//     and oct (f16/bf16) layouts pre-pack interpolation corners so a sample costs 2 or 1
//     16-byte loads instead of 8 scalar gathers, the face layout (f32, the default) two loads
//     per cell;
//   - large launches march by slabs of the volume staged in LDS where that is the faster way
//     (drr_slab_lds); in small ones two or four waves share a ray (drr_parts);
//   - trilinear weights and lerps are FP32 in software: HIP's image/texture API is not
//     available for gfx950 (hipcc rejects tex3D for this target), so there is no hardware
//     filtering to fall back on.
#include "xrh_internal.h"
#include "xrh_ray.h"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstring>

namespace xrh {
namespace {

// ---------------------------------------------------------------------------------------
// trilinear sampling per layout. Formats: 0 f32 linear, 1 f32 quad, 2 f16 linear, 3 f16 oct,
// 4 bf16 linear, 5 bf16 oct, sampled one by one; 7 f32 coefficients, 11 f32 x-faces, 13 f32
// x-faces in bricks, fetched cell by cell (two 16-byte loads) and marched with march_cells. (16-bit oct
// cells, one load each, are faster sample by sample: 0.315 ns per ray against 0.353 by cells.)
constexpr bool is_cell_fmt(int fmt) { return fmt == 7 || fmt == 11 || fmt == 13; }

struct VolView {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t py;     // row pitch (elements)
  uint32_t pz;     // slice pitch (elements)
  uint32_t apron;  // 1 + py + pz: element index of voxel (0, 0, 0)
};

// a (1 - w) + b w as two fused multiply-adds: as cheap as a + (b - a) w but without its
// cancellation when the result is small next to a (tissue -> air edges), so the FP32 sample
// stays within about an ulp of ITK's double-precision lerp.
__device__ inline float lerp(float a, float b, float w) { return fmaf(w, b, fmaf(-w, a, a)); }

__device__ inline float tri(float v000, float v100, float v010, float v110, float v001,
                            float v101, float v011, float v111, float wx, float wy, float wz)
{
  // x, then y, then z -- the order of ITK's LinearInterpolateImageFunction
  const float x00 = lerp(v000, v100, wx);
  const float x10 = lerp(v010, v110, wx);
  const float x01 = lerp(v001, v101, wx);
  const float x11 = lerp(v011, v111, wx);
  const float xx0 = lerp(x00, x10, wy);
  const float xx1 = lerp(x01, x11, wy);
  return lerp(xx0, xx1, wz);
}

// The same for corners of 16-bit storage: their differences along x are exact in FP32 (11 or 8 bits of
// significand, unless one is over 2^13 times the other), so a + w (b - a) is rounded once. Two samples
// of one cell share them.
__device__ inline float tri16_x(float v000, float d00, float v010, float d10, float v001, float d01, float v011,
                                float d11, float wx, float wy, float wz)
{
  const float xx0 = lerp(fmaf(wx, d00, v000), fmaf(wx, d10, v010), wy);
  const float xx1 = lerp(fmaf(wx, d01, v001), fmaf(wx, d11, v011), wy);
  return lerp(xx0, xx1, wz);
}

__device__ inline float tri16(float v000, float v100, float v010, float v110, float v001,
                              float v101, float v011, float v111, float wx, float wy, float wz)
{
  return tri16_x(v000, v100 - v000, v010, v110 - v010, v001, v101 - v001, v011, v111 - v011, wx, wy, wz);
}

// The high minus the low half of a word, both f16, in FP32 (V_FMA_MIX_F32 converts its operands; from
// two conversions and a subtraction the compiler does not form it, and the gathering march over 256 x
// 256 x 200 f16 voxels takes 0.402 instead of 0.315 ns per ray).
__device__ inline float half_diff(uint32_t w)
{
  float d;
  asm("v_fma_mix_f32 %0, %1, 1.0, -%1 op_sel:[1,0,0] op_sel_hi:[1,0,1]" : "=v"(d) : "v"(w));
  return d;
}

// floor(x) converted to int in one instruction (V_CVT_FLR_I32_F32). Inline asm counts as
// convergent, so the sample loops below are unrolled by hand.
__device__ inline int cvt_floor(float x)
{
  int r;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

// a * b + c for 24-bit unsigned a and uniform b as one V_MAD_U32_U24 (the compiler otherwise
// forms two multiplies and a three-way add)
__device__ inline uint32_t mad_u24(uint32_t a, uint32_t b, uint32_t c)
{
  uint32_t r;
  asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
}

// the same for signed 24-bit a and c (V_MAD_I32_I24)
__device__ inline int32_t mad_i24(int32_t a, int32_t b, int32_t c)
{
  int32_t r;
  asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
}

// Element index of the base corner of cell (ix, iy, iz). kPadded: the position was already in the
// padded grid's index frame (FP64 ray set-up), so no apron offset is needed.
template <int kFmt, bool kPadded>
__device__ inline uint32_t element(const VolView& v, int ix, int iy, int iz)
{
  if constexpr (kFmt == 13) {
    // bricked x-faces: padded cell (ix+1, iy+1, iz+1), brick (./4) in brick order with the
    // brick pitches in py / pz, 5x4x4 faces per brick (x fastest, the last x-face repeated)
    const uint32_t ax = (uint32_t)(kPadded ? ix : ix + 1), ay = (uint32_t)(kPadded ? iy : iy + 1),
                   az = (uint32_t)(kPadded ? iz : iz + 1);
    const uint32_t brick = __umul24(az >> 2, v.pz) + __umul24(ay >> 2, v.py) + (ax >> 2);
    const uint32_t local = __umul24(az & 3u, 20u) + __umul24(ay & 3u, 5u) + (ax & 3u);
    return __umul24(brick, (uint32_t)kBrickFaces) + local;
  } else if constexpr (kPadded) {
    // padded indices are >= 0 for every position within a voxel of the index box
    return mad_u24((uint32_t)iz, v.pz, mad_u24((uint32_t)iy, v.py, (uint32_t)ix));
  } else {
    // ix, iy, iz >= -1 and the pitches < 2^23, so the signed 24-bit multiply-adds are exact;
    // v.apron = 1 + py + pz shifts past the apron
    return (uint32_t)mad_i24(iz, (int32_t)v.pz, mad_i24(iy, (int32_t)v.py, ix)) + v.apron;
  }
}

template <int kFmt, bool kPadded>
__device__ inline float sample(const VolView& v, float x, float y, float z)
{
  // x - floor(x) (V_FRACT_F32) and floor(x) as int: two instructions per axis
  const float wx = __builtin_amdgcn_fractf(x), wy = __builtin_amdgcn_fractf(y), wz = __builtin_amdgcn_fractf(z);
  const uint32_t e = element<kFmt, kPadded>(v, cvt_floor(x), cvt_floor(y), cvt_floor(z));
  if constexpr (kFmt == 0) {
    const int o = (int)(e * 4u);
    const int oy = (int)(v.py * 4u);
    const int sz = (int)(v.pz * 4u);
    const float v000 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v.rsrc, o, 0, 0));
    const float v100 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v.rsrc, o + 4, 0, 0));
    const float v010 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v.rsrc, o + oy, 0, 0));
    const float v110 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v.rsrc, o + oy + 4, 0, 0));
    const float v001 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v.rsrc, o, sz, 0));
    const float v101 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v.rsrc, o + 4, sz, 0));
    const float v011 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v.rsrc, o + oy, sz, 0));
    const float v111 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v.rsrc, o + oy + 4, sz, 0));
    return tri(v000, v100, v010, v110, v001, v101, v011, v111, wx, wy, wz);
  } else if constexpr (kFmt == 1) {
    const int o = (int)(e * 16u);
    const int sz = (int)(v.pz * 16u);
    const auto q0 = __builtin_amdgcn_raw_buffer_load_b128(v.rsrc, o, 0, 0);
    const auto q1 = __builtin_amdgcn_raw_buffer_load_b128(v.rsrc, o, sz, 0);
    return tri(__uint_as_float(q0[0]), __uint_as_float(q0[1]), __uint_as_float(q0[2]),
               __uint_as_float(q0[3]), __uint_as_float(q1[0]), __uint_as_float(q1[1]),
               __uint_as_float(q1[2]), __uint_as_float(q1[3]), wx, wy, wz);
  } else if constexpr (kFmt == 2 || kFmt == 4) {
    const int o = (int)(e * 2u);
    const int oy = (int)(v.py * 2u);
    const int sz = (int)(v.pz * 2u);
    uint32_t r[8];
    r[0] = __builtin_amdgcn_raw_buffer_load_b16(v.rsrc, o, 0, 0);
    r[1] = __builtin_amdgcn_raw_buffer_load_b16(v.rsrc, o + 2, 0, 0);
    r[2] = __builtin_amdgcn_raw_buffer_load_b16(v.rsrc, o + oy, 0, 0);
    r[3] = __builtin_amdgcn_raw_buffer_load_b16(v.rsrc, o + oy + 2, 0, 0);
    r[4] = __builtin_amdgcn_raw_buffer_load_b16(v.rsrc, o, sz, 0);
    r[5] = __builtin_amdgcn_raw_buffer_load_b16(v.rsrc, o + 2, sz, 0);
    r[6] = __builtin_amdgcn_raw_buffer_load_b16(v.rsrc, o + oy, sz, 0);
    r[7] = __builtin_amdgcn_raw_buffer_load_b16(v.rsrc, o + oy + 2, sz, 0);
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = (kFmt == 2) ? h2f(r[i]) : bf2f(r[i]);
    return tri16(f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7], wx, wy, wz);
  } else {
    const int o = (int)(e * 16u);
    const auto q = __builtin_amdgcn_raw_buffer_load_b128(v.rsrc, o, 0, 0);
    float f[4], d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (kFmt == 3) {
        f[i] = h2f(q[i] & 0xffffu);
        d[i] = half_diff(q[i]);
      } else {
        f[i] = bf2f(q[i] & 0xffffu);
        d[i] = bf2f(q[i] >> 16) - f[i];
      }
    }
    return tri16_x(f[0], d[0], f[1], d[1], f[2], d[2], f[3], d[3], wx, wy, wz);
  }
}

// Empty-space skipping. Walks from sample i towards sample `end` (dir = +1 or -1) over samples
// that lie in bricks whose one-voxel-dilated trilinear support holds only zero voxels, so
// their interpolated value is exactly 0 and leaving them out of a SUM changes nothing. At a
// brick at Chebyshev distance d >= 1 from the nearest occupied brick, the cube of bricks
// within d-1 is empty: every sample up to the cube's exit face is skipped and the walk
// continues with the first sample past it (at least one sample per iteration, so at most
// |end - i| + 1 iterations). The walk runs in brick units (positions scaled by 2^-shift,
// exact) with branch-free exit faces: b + d moving up an axis, b + 1 - d moving down, none
// along an axis the ray does not move on. Its positions, start + i*step in float, differ from
// the sample loop's by far less than the one-voxel dilation. Returns the first sample (in walk
// order) that may be non-zero.
__device__ __forceinline__ int skip_empty(const DrrItem& it, const Ray& r, int i, int end, int dir, float org)
{
  const float B = (float)(1 << it.skip_shift), invB = __builtin_ldexpf(1.0f, -it.skip_shift);
  // ray in brick units
  const float bx0 = (r.sx - org) * invB, by0 = (r.sy - org) * invB, bz0 = (r.sz - org) * invB;
  const float dbx = r.dx * invB, dby = r.dy * invB, dbz = r.dz * invB;
  // per axis: exit face b + o + s (d - 1), samples to reach it (face - p) * k (+ h: infinite
  // when the walk does not move along the axis)
  const float vx = dir > 0 ? r.dx : -r.dx, vy = dir > 0 ? r.dy : -r.dy, vz = dir > 0 ? r.dz : -r.dz;
  const float sx = vx > 0.0f ? 1.0f : -1.0f, sy = vy > 0.0f ? 1.0f : -1.0f, sz = vz > 0.0f ? 1.0f : -1.0f;
  const float ox = vx > 0.0f ? 1.0f : 0.0f, oy = vy > 0.0f ? 1.0f : 0.0f, oz = vz > 0.0f ? 1.0f : 0.0f;
  const float kx = vx != 0.0f ? B * __builtin_amdgcn_rcpf(vx) : 0.0f;
  const float ky = vy != 0.0f ? B * __builtin_amdgcn_rcpf(vy) : 0.0f;
  const float kz = vz != 0.0f ? B * __builtin_amdgcn_rcpf(vz) : 0.0f;
  const float hx = vx != 0.0f ? 0.0f : 3.0e38f, hy = vy != 0.0f ? 0.0f : 3.0e38f, hz = vz != 0.0f ? 0.0f : 3.0e38f;
  const float gx1 = (float)(it.skip_gx - 1), gy1 = (float)(it.skip_gy - 1), gz1 = (float)(it.skip_gz - 1);
  // the map is below 2^24 bytes and gy * gz below 2^24 (checked when it is built), so the
  // 24-bit multiply-adds below are exact and a stray index reads 0 from the buffer range check
  const auto map = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(it.skip), (short)0,
                                                     it.skip_gx * it.skip_gy * it.skip_gz, 0x00020000);
  while (dir > 0 ? (i <= end) : (i >= end)) {
    const float fi = (float)i;
    const float px = fmaf(fi, dbx, bx0), py = fmaf(fi, dby, by0), pz = fmaf(fi, dbz, bz0);
    const float fx = __builtin_amdgcn_fmed3f(floorf(px), 0.0f, gx1);
    const float fy = __builtin_amdgcn_fmed3f(floorf(py), 0.0f, gy1);
    const float fz = __builtin_amdgcn_fmed3f(floorf(pz), 0.0f, gz1);
    const uint32_t e = mad_u24(mad_u24((uint32_t)fz, (uint32_t)it.skip_gy, (uint32_t)fy), (uint32_t)it.skip_gx,
                               (uint32_t)fx);
    const int d = __builtin_amdgcn_raw_buffer_load_b8(map, (int)e, 0, 0);
    if (d == 0) break;
    const float dm1 = (float)(d - 1);
    const float tx = fmaf((fmaf(sx, dm1, ox) + fx) - px, kx, hx);
    const float ty = fmaf((fmaf(sy, dm1, oy) + fy) - py, ky, hy);
    const float tz = fmaf((fmaf(sz, dm1, oz) + fz) - pz, kz, hz);
    const float s = fminf(fminf(tx, ty), tz);
    const int jump = (s >= 1.0f) ? (int)fminf(s, 1.0e9f) + 1 : 1;
    i += dir * jump;
  }
  return i;
}

// Sample range [first, last] that can hold non-zero values (SUM with an empty-space map), or
// the whole ray [0, n]. FP64 set-up rays start in the padded frame (org 1).
template <int kOp, int kGeom>
__device__ __forceinline__ void sample_range(const DrrItem& it, const Ray& r, int& first, int& last)
{
  first = 0;
  last = r.n;
  if (kOp == XRH_LINE_INT_SUM && it.skip) {
    const float org = (kGeom == XRH_GEOM_FP64) ? 1.0f : 0.0f;
    first = skip_empty(it, r, 0, r.n, 1, org);
    last = (first <= r.n) ? skip_empty(it, r, r.n, first, -1, org) : first - 1;
  }
}

__device__ inline double wave_sum_d(double v)
{
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// ---------------------------------------------------------------------------------------
// kernels

constexpr int kSetupItems = 8, kSetupThreads = 64, kSetupCopy = 256;  // items, lanes, words copied per workgroup

__global__ __launch_bounds__(kSetupThreads) void drr_setup_kernel(const PoseIn* __restrict__ poses,
                                                                  const VolDesc* __restrict__ vols,
                                                                  const CamDev* __restrict__ cams,
                                                                  DrrItem* __restrict__ items, int64_t n,
                                                                  int item_blocks, SetupCopy copy)
{
#pragma clang fp contract(off)
  constexpr int kWords = (int)sizeof(PoseIn) / 8, kLoads = (kSetupItems * kWords + kSetupThreads - 1) / kSetupThreads;
  static_assert(sizeof(PoseIn) % 8 == 0, "poses are read in 8-byte words");
  const int tid = threadIdx.x;
  if ((int)blockIdx.x >= item_blocks) {
    const uint64_t w0 = (uint64_t)(blockIdx.x - item_blocks) * kSetupCopy;
#pragma unroll
    for (int k = 0; k < kSetupCopy / kSetupThreads; ++k) {
      const uint64_t w = w0 + (uint64_t)(k * kSetupThreads + tid);
      if (w < copy.words[0]) copy.dst[0][w] = copy.src[0][w];
      else if (w - copy.words[0] < copy.words[1]) copy.dst[1][w - copy.words[0]] = copy.src[1][w - copy.words[0]];
    }
    return;
  }
  // the workgroup's poses, read together: they may be in host memory
  __shared__ uint64_t words[kSetupItems * kWords];
  const int64_t i0 = (int64_t)blockIdx.x * kSetupItems;
  const int m = (int)min((int64_t)kSetupItems, n - i0);
  uint64_t buf[kLoads];
#pragma unroll
  for (int k = 0; k < kLoads; ++k) {
    const int w = k * kSetupThreads + tid;
    buf[k] = (w < m * kWords) ? ((const uint64_t*)(poses + i0))[w] : 0;
  }
#pragma unroll
  for (int k = 0; k < kLoads; ++k) {
    const int w = k * kSetupThreads + tid;
    if (w < m * kWords) words[w] = buf[k];
  }
  __syncthreads();
  if (tid >= m) return;
  const int64_t i = i0 + tid;
  PoseIn p;
  __builtin_memcpy(&p, &words[tid * kWords], sizeof(PoseIn));
  const VolDesc& v = vols[p.vol];
  DrrItem it;
  // phys->idx * cam->phys: Affine*Affine product (xregRayCastLineIntCPU.cpp:207-208), float
  float T[12];
  for (int k = 0; k < 12; ++k) T[k] = (float)p.pose[k];
  for (int r = 0; r < 3; ++r) {
    const float* a = &v.p2i[4 * r];
    for (int c = 0; c < 3; ++c) it.M[4 * r + c] = (a[0] * T[c] + a[1] * T[4 + c]) + a[2] * T[8 + c];
    it.M[4 * r + 3] = ((a[0] * T[3] + a[1] * T[7]) + a[2] * T[11]) + a[3];
  }
  // the same in double from the FP64 pose
  for (int r = 0; r < 3; ++r) {
    const double* a = &v.p2i_d[4 * r];
    for (int c = 0; c < 3; ++c) {
      it.Md[4 * r + c] = a[0] * p.pose[c] + a[1] * p.pose[4 + c] + a[2] * p.pose[8 + c];
    }
    it.Md[4 * r + 3] = a[0] * p.pose[3] + a[1] * p.pose[7] + a[2] * p.pose[11] + a[3];
  }
  it.cam = cams[p.cam];
  it.vol = v.data;
  it.vol_bytes = v.bytes;
  it.raw = v.raw;
  it.raw_bytes = v.raw_bytes;
  it.raw_py = v.X + 2;
  it.raw_pz = (v.X + 2) * (v.Y + 2);
  it.X = v.X;
  it.Y = v.Y;
  it.Z = v.Z;
  it.pitch_y = v.pitch_y;
  it.pitch_z = v.pitch_z;
  it.step = p.step;
  it.out_off = p.out_off;
  it.ncc_zf = p.ncc_zf;
  it.bg = p.bg;
  it.tiles_x = (it.cam.cols + kTile - 1) / kTile;
  it.tiles_y = (it.cam.rows + kTile - 1) / kTile;
  it.skip = v.skip;
  it.skip_gx = v.skip_gx;
  it.skip_gy = v.skip_gy;
  it.skip_gz = v.skip_gz;
  it.skip_shift = v.skip_shift;
  items[i] = it;
}

// ---------------------------------------------------------------------------------------
// marching. A ray's samples 0..n are summed in kSegs segments of seg_len(n) consecutive samples,
// each segment from zero and the segments' sums in order. The order is a property of the ray, so
// one lane can march a whole ray (large launches) or several waves can share it (small ones) and
// every pixel comes out the same bit for bit.
constexpr int kWindow = 16;
constexpr int kSegs = 8;
__device__ inline int seg_len(int n) { return (n + kSegs * kWindow) / (kSegs * kWindow) * kWindow; }

template <int kOp>
__device__ inline float line_init()
{
  return (kOp == XRH_LINE_INT_SUM) ? 0.0f : -3.402823466e+38f;
}

// Index of the segment that holds sample i (i < 2^23, exact after the correction).
__device__ inline int seg_of(int i, int seg)
{
  int k = (int)((float)i * __builtin_amdgcn_rcpf((float)seg));
  k -= (k * seg > i) ? 1 : 0;
  k += ((k + 1) * seg <= i) ? 1 : 0;
  return k;
}

// Position of the next sample under FP32 ray set-up: the reference advances by repeated float
// addition (:276), over samples that are skipped too. (FP64 set-up: start + i * step.)
struct Pos {
  float x, y, z;
  __device__ void advance(const Ray& r, int count)
  {
    for (int k = 0; k < count; ++k) {
      x = x + r.dx;
      y = y + r.dy;
      z = z + r.dz;
    }
  }
};

// Two adjacent 16-byte elements: the cell's value at local coordinates (wx, wy, wz).
template <int kFmt>
__device__ inline float cell_value(const float (&a)[4], const float (&b)[4], float wx, float wy, float wz)
{
  if constexpr (kFmt == 7) {
    // trilinear polynomial: planes w^0 and w^1
    const float p0 = fmaf(wy, fmaf(wx, a[3], a[2]), fmaf(wx, a[1], a[0]));
    const float p1 = fmaf(wy, fmaf(wx, b[3], b[2]), fmaf(wx, b[1], b[0]));
    return fmaf(wz, p1, p0);
  } else {
    // the faces at x and x + 1: their edges along y, between those along z, then along x
    const float a0 = fmaf(wy, a[1], a[0]), a1 = fmaf(wy, a[3], a[2]);
    const float b0 = fmaf(wy, b[1], b[0]), b1 = fmaf(wy, b[3], b[2]);
    return lerp(fmaf(wz, a1 - a0, a0), fmaf(wz, b1 - b0, b0), wx);
  }
}

// Samples [i, last] of a ray, cell by cell: each iteration fetches the cell of the lane's next
// sample and evaluates that sample and, if it is in the same cell, the one after it.
//
// What bounds the march is the gather: a 16-byte buffer load takes 16.5 clocks of a CU's
// address/data path however many of the wave's lanes are active (measured, L1 resident), so a
// loop that steps by samples and loads for the lanes that changed cell pays two loads per sample
// (at half-voxel steps some lane of 64 always changes). Stepping by cells keeps every lane in
// every load: about 0.6 pairs of loads per sample. The second sample's local coordinates are the
// first's plus the step (FP64 set-up), which also saves its index arithmetic; under FP32 set-up
// they are taken from the reference's own position, whose cell is exact. As unsigned integers
// the three coordinates' largest is below that of 1.0f exactly when all lie in [0, 1).
// The lanes of a wave wait for each other at the ends of windows of `window` samples, of which the first is
// that of sample `from` (at most i): at nearly the same depth they fetch the same cells. Which samples form a pair
// follows from the ray's own first sample alone.
template <int kGeom, int kOp, int kFmt>
__device__ __forceinline__ float march_cells(const Ray& ray, const VolView& vv, Pos& pos, int i, int last, int seg,
                                             int from, int window)
{
  float tot = line_init<kOp>(), acc = line_init<kOp>();
  int seg_last = (seg_of(i, seg) + 1) * seg - 1, win_last = from | (window - 1);
  float f = (float)i;  // sample indices as floats (exact: n < 2^23)
  for (;;) {
    const float fstop = (float)min(win_last, last), fpair = (float)min(seg_last, last);
    while (f <= fstop) {
      float x, y, z;
      if constexpr (kGeom == XRH_GEOM_FP32) {
        x = pos.x;
        y = pos.y;
        z = pos.z;
      } else {
        x = fmaf(f, ray.dx, ray.sx);
        y = fmaf(f, ray.dy, ray.sy);
        z = fmaf(f, ray.dz, ray.sz);
      }
      float wx = __builtin_amdgcn_fractf(x), wy = __builtin_amdgcn_fractf(y), wz = __builtin_amdgcn_fractf(z);
      const uint32_t e = element<kFmt, kGeom == XRH_GEOM_FP64>(vv, cvt_floor(x), cvt_floor(y), cvt_floor(z));
      const uint32_t o = e * (kFmt == 7 ? 32u : 16u);
      const auto la = __builtin_amdgcn_raw_buffer_load_b128(vv.rsrc, (int)o, 0, 0);
      const auto lb = __builtin_amdgcn_raw_buffer_load_b128(vv.rsrc, (int)(o + 16u), 0, 0);
      float a[4], b[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        a[k] = __uint_as_float(la[k]);
        b[k] = __uint_as_float(lb[k]);
      }
      acc = line_op<kOp>(acc, cell_value<kFmt>(a, b, wx, wy, wz));
      f = f + 1.0f;
      if constexpr (kGeom == XRH_GEOM_FP32) {
        const float bx = x - wx, by = y - wy, bz = z - wz;  // floor
        pos.advance(ray, 1);
        wx = pos.x - bx;
        wy = pos.y - by;
        wz = pos.z - bz;
      } else {
        wx = wx + ray.dx;
        wy = wy + ray.dy;
        wz = wz + ray.dz;
      }
      const uint32_t top = max(max(__float_as_uint(wx), __float_as_uint(wy)), __float_as_uint(wz));
      if (top < 0x3f800000u && f <= fpair) {
        acc = line_op<kOp>(acc, cell_value<kFmt>(a, b, wx, wy, wz));
        f = f + 1.0f;
        if constexpr (kGeom == XRH_GEOM_FP32) pos.advance(ray, 1);
      }
    }
    const bool done = win_last >= last;
    if (done || win_last >= seg_last) {
      tot = line_op<kOp>(tot, acc);
      acc = line_init<kOp>();
      seg_last += seg;
    }
    if (done) break;
    win_last += window;
  }
  return tot;
}

// Samples [i, last] of one segment, two per iteration, each with its own loads.
template <int kGeom, int kOp, int kFmt>
__device__ __forceinline__ float march_samples(const Ray& ray, const VolView& vv, Pos& pos, int i, int last)
{
  float acc = line_init<kOp>();
  if constexpr (kGeom == XRH_GEOM_FP32) {
    for (; i < last; i += 2) {
      const float qx = pos.x + ray.dx, qy = pos.y + ray.dy, qz = pos.z + ray.dz;
      const float s0 = sample<kFmt, false>(vv, pos.x, pos.y, pos.z);
      const float s1 = sample<kFmt, false>(vv, qx, qy, qz);
      acc = line_op<kOp>(line_op<kOp>(acc, s0), s1);
      pos.x = qx + ray.dx;
      pos.y = qy + ray.dy;
      pos.z = qz + ray.dz;
    }
    if (i == last) {
      acc = line_op<kOp>(acc, sample<kFmt, false>(vv, pos.x, pos.y, pos.z));
      pos.advance(ray, 1);
    }
  } else {
    // sample indices as floats (exact: n < 2^23), advanced by float additions
    float f0 = (float)i;
    for (; i < last; i += 2) {
      const float f1 = f0 + 1.0f;
      const float s0 = sample<kFmt, true>(vv, fmaf(f0, ray.dx, ray.sx), fmaf(f0, ray.dy, ray.sy),
                                          fmaf(f0, ray.dz, ray.sz));
      const float s1 = sample<kFmt, true>(vv, fmaf(f1, ray.dx, ray.sx), fmaf(f1, ray.dy, ray.sy),
                                          fmaf(f1, ray.dz, ray.sz));
      acc = line_op<kOp>(line_op<kOp>(acc, s0), s1);
      f0 = f0 + 2.0f;
    }
    if (i == last) {
      acc = line_op<kOp>(acc, sample<kFmt, true>(vv, fmaf(f0, ray.dx, ray.sx), fmaf(f0, ray.dy, ray.sy),
                                                 fmaf(f0, ray.dz, ray.sz)));
    }
  }
  return acc;
}

// Samples [i, last] (i <= last) of one ray, summed segment by segment; the wave's lanes have their first
// samples from `from` on. `pos`: sample i's position under FP32 set-up; it ends past sample `last`.
template <int kGeom, int kOp, int kFmt>
__device__ __forceinline__ float march(const Ray& ray, const VolView& vv, Pos& pos, int i, int last, int seg, int from,
                                       int window)
{
  if constexpr (is_cell_fmt(kFmt)) {
    return march_cells<kGeom, kOp, kFmt>(ray, vv, pos, i, last, seg, from, window);
  } else {
    float tot = line_init<kOp>();
    for (int end = (seg_of(i, seg) + 1) * seg - 1; i <= last; end += seg) {
      const int stop = min(end, last);
      tot = line_op<kOp>(tot, march_samples<kGeom, kOp, kFmt>(ray, vv, pos, i, stop));
      i = stop + 1;
    }
    return tot;
  }
}

// The fused NCC epilogue: FP64 sums of m, m^2 and m * zero-mean fixed over the tile, one
// record per tile. Every thread of the block calls it (it synchronises).
__device__ inline void ncc_epilogue(const DrrItem& it, const TileRef& tr, bool inside, int col, int row, float pix,
                                    double* __restrict__ ncc_partials, int ncc_tiles)
{
  if (ncc_partials && it.ncc_zf) {
    // NCC epilogue: sums of m, m^2 and m * zero-mean fixed, FP64, one record per tile
    double s1 = 0.0, s2 = 0.0, sf = 0.0;
    if (inside) {
      const double m = (double)pix;
      const double f = (double)it.ncc_zf[(int64_t)row * it.cam.cols + col];
      s1 = m;
      s2 = m * m;
      sf = m * f;
    }
    s1 = wave_sum_d(s1);
    s2 = wave_sum_d(s2);
    sf = wave_sum_d(sf);
    __shared__ double red[4][3];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0 && w < 4) {
      red[w][0] = s1;
      red[w][1] = s2;
      red[w][2] = sf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double* dst = ncc_partials + ((int64_t)tr.item * ncc_tiles + (int64_t)tr.ty * it.tiles_x + tr.tx) * 4;
      dst[0] = (red[0][0] + red[1][0]) + (red[2][0] + red[3][0]);
      dst[1] = (red[0][1] + red[1][1]) + (red[2][1] + red[3][1]);
      dst[2] = (red[0][2] + red[1][2]) + (red[2][2] + red[3][2]);
      dst[3] = 0.0;
    }
  }
}

// Pixel store (REPLACE / ACCUM with the line kernel, RayCasterCPU::pre_compute semantics) and
// the fused NCC epilogue. Every thread of the block calls it (it synchronises).
template <int kOp>
__device__ inline void store_pixel(const DrrItem& it, const TileRef& tr, bool inside, int col, int row, float acc,
                                   float* __restrict__ out, int accumulate, float fill,
                                   double* __restrict__ ncc_partials, int ncc_tiles)
{
  float pix = 0.0f;
  if (inside) {
    const int64_t o = it.out_off + (int64_t)row * it.cam.cols + col;
    const float prev = accumulate ? out[o] : fill;
    const float aa = 0.0f + acc * 1.0f;
    if constexpr (kOp == XRH_LINE_INT_SUM) pix = prev + aa; else pix = (prev < aa) ? aa : prev;
    out[o] = pix;
  }
  ncc_epilogue(it, tr, inside, col, row, pix, ncc_partials, ncc_tiles);
}

__device__ inline VolView vol_view(const DrrItem& it)
{
  VolView vv;
  vv.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(it.vol), (short)0, (int)it.vol_bytes, 0x00020000);
  vv.py = it.pitch_y;
  vv.pz = it.pitch_z;
  vv.apron = 1u + it.pitch_y + it.pitch_z;
  return vv;
}

// One ray of one item: the line integral (SUM) or maximum (MAX) of its samples times the step,
// or the kernel's initial value when the ray misses the volume. Called by every lane of the
// wave (`inside` false for lanes past the detector edge), so that the lanes can agree on a
// start, the wave's earliest first sample: neighbouring rays, which enter the volume at
// nearly the same depth, then fetch the same cells in the same iteration (C2: L1 tag accesses
// -7.5%, L1 tag-conflict stalls -40%, DRR -2%). By cells a lane waits for its own first sample;
// sample by sample it marches from the common one, over samples that lie in empty bricks and are
// exactly 0. Either way its sum is the same as from its own first sample, bit for bit.
template <int kGeom, int kOp, int kFmt>
__device__ __forceinline__ float cast_range(const DrrItem& it, const Ray& ray, int i, int last, int window)
{
  float acc = line_init<kOp>();
  // wave minimum of the first samples of the lanes with samples (all lanes take part)
  int start = (i <= last) ? i : 0x7fffffff;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) start = min(start, __shfl_xor(start, off, 64));
  if (ray.n >= 0) {
    if (i <= last) {
      // sample by sample the lanes start together, on samples that are zero
      if constexpr (!is_cell_fmt(kFmt)) i = start;
      Pos pos{ray.sx, ray.sy, ray.sz};
      if constexpr (kGeom == XRH_GEOM_FP32) pos.advance(ray, i);
      acc = march<kGeom, kOp, kFmt>(ray, vol_view(it), pos, i, last, seg_len(ray.n), start, window);
    }
    acc = acc * it.step;
  }
  return acc;
}

// Ray set-up and sample range of a pixel ([0, -1] and n = -1 for none).
template <int kGeom, int kOp>
__device__ __forceinline__ Ray begin_ray(const DrrItem& it, int col, int row, bool inside, int& first, int& last)
{
  Ray ray;
  ray.n = -1;
  first = 0;
  last = -1;
  if (inside) {
    ray = (kGeom == XRH_GEOM_FP32) ? setup_ray_f32(it, (float)col, (float)row) : setup_ray_f64(it, col, row);
    if (ray.n >= 0) sample_range<kOp, kGeom>(it, ray, first, last);
  }
  return ray;
}

template <int kGeom, int kOp, int kFmt>
__device__ __forceinline__ float cast_ray(const DrrItem& it, int col, int row, bool inside, int window)
{
  int first, last;
  const Ray ray = begin_ray<kGeom, kOp>(it, col, row, inside, first, last);
  return cast_range<kGeom, kOp, kFmt>(it, ray, first, last, window);
}

// ---------------------------------------------------------------------------------------
// slab marching. The gathering march is bound by the per-lane fetch path: 16.5 clocks of a CU per
// 16-byte load, more when its lanes touch more cache lines, and an L1 (32 KB for 32 waves) that
// holds none of them until the next layer when neighbouring rays are a voxel or more apart (96 x
// 96 rays over 256 x 256 x 200 voxels: L1 hits 49%, 5 TB/s of fabric traffic, VALU 12%). Here a
// workgroup moves through the volume slab by slab along the tile's main axis: the box of voxels
// that its 256 rays can reach in the next few layers is loaded into LDS once, as plain 4-byte
// voxels (a quarter of the face layout's bytes), 16 bytes per lane straight from the buffer load,
// and the rays take their cells from there. LDS serves a 64-lane read of two neighbouring voxels
// in about 5 clocks whatever lines they share, so lanes also need not stay in step.
//
// The box comes from the tile's corner rays: the pixel -> position map on a plane across the main
// axis is projective, so the corners' positions on the slab's two planes bound every ray between
// them. Slabs end on cell faces, so no cell straddles two. A cell's faces are formed
// from its voxels by the float operations that built the face layout (16-bit storage: the gathering
// march's lerps, from voxels kept as floats), and samples segment as there: the values are the
// gathering march's bit for bit, and tiles whose box
// does not fit (rays several voxels apart, oblique tiles) take that march.
//
// Measured, FP64 set-up, launches of 1 to 1.8 million rays, ns per ray, gathering sample by sample (before) / by
// cells / slabs: 256 x 256 x 200 voxels at 0.39 voxels between rays 0.430 / 0.372 / 0.349, 0.78: 0.60 / 0.553 /
// 0.438, 1.55: 1.39 / 1.07 / 1.02; 512 x 512 x 400 voxels at 0.39: 1.01 / 0.817 / 0.585, 0.78: 1.34 / 1.36 / 0.841,
// 1.55: 3.5 / 2.8 / 1.84. Layers per slab:
// 8 / 12 / 16 at 0.39: 0.386 / 0.351 / 0.353; along x one 64-byte row of 16 voxels.
constexpr int kSlabDepth = 12, kSlabDepthX = 15;

// One axis of a 3-vector by a uniform index.
template <class T>
__device__ inline T pick(int axis, T x, T y, T z)
{
  return axis == 0 ? x : (axis == 1 ? y : z);
}

__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// v from another lane of the row by a DPP control word
template <int kCtrl>
__device__ inline float dpp(float v)
{
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, true));
}

// A box of voxels in LDS: voxel (x, y, z) of the padded grid at x - x0 + sy (y - y0) + sz (z - z0).
struct Box {
  int x0, y0, z0, wx, wy, wz;
  int lpr, rows;  // lanes per row (16 bytes each) and rows per load
  int sy, sz;
  __device__ int floats() const { return sz * wz; }
  __device__ void pitch()
  {
    lpr = (wx + 3) >> 2;
    rows = 64 / lpr;
    sy = 4 * lpr;
    sz = sy * wy;
  }
};

// Loads the box from the padded voxels (pitches py, pz), 16 bytes per lane straight into LDS, as
// many rows of one z as fit per instruction (a row's last lane may overhang into its padding).
__device__ inline void stage_box(__amdgpu_buffer_rsrc_t src, const Box& b, uint32_t py, uint32_t pz, float* lds)
{
  const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6);
  const int sub = lane / b.lpr;
  const uint32_t lane_off = ((uint32_t)sub * py + (uint32_t)(lane - sub * b.lpr) * 4u) * 4u;
  const int groups = (b.wy + b.rows - 1) / b.rows;
  int z = 0, g = wave;
  while (g >= groups) {
    g -= groups;
    ++z;
  }
  while (z < b.wz) {
    const uint32_t row = (uint32_t)(b.z0 + z) * pz + (uint32_t)(b.y0 + g * b.rows) * py + (uint32_t)b.x0;
    float* dst = lds + z * b.sz + g * b.rows * b.sy;
    if (sub < min(b.rows, b.wy - g * b.rows)) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16,
                                               (int)(lane_off + row * 4u), 0, 0, 0);
    }
    g += kThreads / 64;
    while (g >= groups) {
      g -= groups;
      ++z;
    }
  }
}

struct LdsPair {
  float a, b;
};
// Two consecutive floats at an LDS byte address (one DS_READ2_B32).
__device__ inline LdsPair lds_pair(int addr)
{
  const auto* p = (const __attribute__((address_space(3))) float*)(uintptr_t)(uint32_t)addr;
  return {p[0], p[1]};
}

// Margin of the boxes around the corner rays (voxels). A sample lies off its exact line by the rounding
// of its start, step and position: in all at most some 5e-7 of the volume's largest edge across the main
// axis, with what its offset along that axis moves the line there (slopes up to 2) and the lines' own
// rounding to float, kept at 1e-6. FP32 set-up carries the detector point through 13 rounded operations
// and the start of the samples through three more, 6e-8 of the largest intermediate (tile_corner's size) each:
// 1e-6 of it per axis, 3e-6 with the offset along the main axis.
constexpr float kSlabMargin = 0.05f, kSlabMarginEdge = 1.0e-6f, kSlabMarginSetup = 3.0e-6f;

// Source and detector point of the pixel (col, row) in the index frame, in double and from the parameters
// that the rays' set-up uses. `size` (FP32 set-up): with the absolute value of every product and term, so
// the points' sum bounds what the set-up's operations meet.
template <int kGeom>
__device__ __forceinline__ void tile_corner(const DrrItem& it, double col, double row, bool size, double ph[3],
                                            double dp[3])
{
  if constexpr (kGeom == XRH_GEOM_FP64) {
    double det[3];
    ind_to_det_d(it.cam, col, row, det);
    affine_pt_d(it.Md, it.cam.pinhole_d, ph);
    affine_pt_d(it.Md, det, dp);
  } else {
    auto term = [&](float a, double b) {
      const double t = (double)a * b;
      return size ? fabs(t) : t;
    };
    auto rowd = [&](const float* m, const double (&p)[3]) { return (term(m[0], p[0]) + term(m[1], p[1])) + term(m[2], p[2]); };
    const double q[3] = {(double)it.cam.det_z * col, (double)it.cam.det_z * row, (double)it.cam.det_z};
    const double r[3] = {rowd(&it.cam.kinv[0], q), rowd(&it.cam.kinv[3], q), rowd(&it.cam.kinv[6], q) + term(it.cam.z_adj, 1.0)};
    double det[3], pin[3];
    for (int k = 0; k < 3; ++k) {
      det[k] = rowd(&it.cam.einv[4 * k], r) + term(it.cam.einv[4 * k + 3], 1.0);
      pin[k] = term(it.cam.pinhole[k], 1.0);
    }
    for (int k = 0; k < 3; ++k) {
      const double t = term(it.M[4 * k + 3], 1.0);
      ph[k] = rowd(&it.M[4 * k], pin) + t;
      dp[k] = rowd(&it.M[4 * k], det) + t;
    }
  }
}

// cast_ray by slabs. Every thread of the block calls it (it synchronises); `lds` holds `budget`
// floats.
template <int kGeom, int kOp, int kFmt>
__device__ __forceinline__ float cast_ray_slab(const DrrItem& it, const TileRef& tr, int col, int row, bool inside,
                                      float* lds, int budget, int window)
{
  __shared__ double corner[4][3];
  __shared__ double origin[3];
  __shared__ float reach[3][4];
  __shared__ float setup_size;

  int first, last;
  const Ray ray = begin_ray<kGeom, kOp>(it, col, row, inside, first, last);
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid < (kGeom == XRH_GEOM_FP32 ? 8 : 4)) {
    // the lines through the tile's corner pixels, padded index frame
    const bool size = tid >= 4;
    double ph[3], dp[3];
    tile_corner<kGeom>(it, (double)(tr.tx * kTile + (tid & 1) * (kTile - 1)),
                       (double)(tr.ty * kTile + ((tid >> 1) & 1) * (kTile - 1)), size, ph, dp);
    if (!size) {
      for (int k = 0; k < 3; ++k) {
        corner[tid][k] = dp[k] - ph[k];
        if (tid == 0) origin[k] = ph[k] + 1.0;
      }
    } else if (tid == 7) {  // (the largest column and row)
      setup_size = (float)fmax(fmax(ph[0] + dp[0], ph[1] + dp[1]), ph[2] + dp[2]);
    }
  }
  __syncthreads();
  // main axis of the tile: the largest component of its middle direction
  const float mx = (float)(corner[0][0] + corner[3][0]), my = (float)(corner[0][1] + corner[3][1]),
              mz = (float)(corner[0][2] + corner[3][2]);
  const int A = uni((fabsf(mx) >= fabsf(my) && fabsf(mx) >= fabsf(mz)) ? 0 : (fabsf(my) >= fabsf(mz) ? 1 : 2));
  const int B = A == 0 ? 1 : 0, C = A == 2 ? 1 : 2;
  const bool up = uni(pick(A, mx, my, mz) > 0.0f ? 1 : 0) != 0;
  bool ok = it.raw != nullptr;
  for (int k = 0; k < 4; ++k) {
    const double d = up ? corner[k][A] : -corner[k][A];
    ok = ok && d > 0.0 && 2.0 * d >= fabs(corner[k][B]) && 2.0 * d >= fabs(corner[k][C]);
  }
  // this lane's line of the hull: corner lane & 3, axis B or C, as position = u + v * (position on A).
  // (u in double: a source far from the volume is a large number, of which little remains)
  const int hk = lane & 3, hax = (lane & 8) ? C : B;
  const double hc = corner[hk][hax], ha = corner[hk][A];
  const float hr = __builtin_amdgcn_rcpf((float)ha), h0 = (float)hc * hr;
  const double hvd = (double)h0 + fma(-(double)h0, ha, hc) * (double)hr;  // hc / ha to about 1e-13
  const float hv = (float)hvd, hu = (float)(origin[hax] - origin[A] * hvd);
  // the cells along A that the block's samples reach. The margin covers the rounding of the lines
  // and the samples, which grows with their coordinates; under FP32 set-up also that of the set-up
  // itself and the samples' drift, at most one rounding per addition.
  constexpr float kOff = (kGeom == XRH_GEOM_FP64) ? 0.0f : 1.0f;
  const float sA = pick(A, ray.sx, ray.sy, ray.sz), dA = pick(A, ray.dx, ray.dy, ray.dz);
  const float edge = (float)max(max(it.X, it.Y), it.Z);
  float lo = 3.0e38f, hi = -3.0e38f, margin = kSlabMargin + kSlabMarginEdge * edge;
  if (kGeom == XRH_GEOM_FP32) margin = fmaf(kSlabMarginSetup, setup_size, margin);
  if (first <= last) {
    if (kGeom == XRH_GEOM_FP32) margin = fmaf((float)last * edge, 6.0e-8f, margin);
    const float p0 = fmaf((float)first, dA, sA) + kOff, p1 = fmaf((float)last, dA, sA) + kOff;
    lo = fminf(p0, p1);
    hi = fmaxf(p0, p1);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, off, 64));
    hi = fmaxf(hi, __shfl_xor(hi, off, 64));
    if (kGeom == XRH_GEOM_FP32) margin = fmaxf(margin, __shfl_xor(margin, off, 64));
  }
  if (lane == 0) {
    reach[0][tid >> 6] = lo;
    reach[1][tid >> 6] = hi;
    reach[2][tid >> 6] = margin;
  }
  __syncthreads();
  lo = fminf(fminf(reach[0][0], reach[0][1]), fminf(reach[0][2], reach[0][3]));
  hi = fmaxf(fmaxf(reach[1][0], reach[1][1]), fmaxf(reach[1][2], reach[1][3]));
  if (kGeom == XRH_GEOM_FP32) margin = fmaxf(fmaxf(reach[2][0], reach[2][1]), fmaxf(reach[2][2], reach[2][3]));
  const int nA = pick(A, it.X, it.Y, it.Z), nB = pick(B, it.X, it.Y, it.Z), nC = pick(C, it.X, it.Y, it.Z);
  const bool any = uni(lo <= hi ? 1 : 0) != 0;
  const int alo = uni(any ? min(max((int)floorf(lo - margin), 0), nA) : 0);
  const int ahi = uni(any ? min(max((int)floorf(hi + margin), 0), nA) : -1);
  const int total = ahi - alo + 1;
  // the box of cells [a, a + n) along A. `whole`: not cut at the volume's faces (for its size), and
  // one voxel wider per axis.
  auto box_of = [&](int a, int n, bool whole) {
    const float v = fmaf((float)((lane & 4) ? a + n : a), hv, hu);
    float l = fminf(v, dpp<0xB1>(v)), h = fmaxf(v, dpp<0xB1>(v));  // lanes ^ 1
    l = fminf(l, dpp<0x4E>(l));                                    // lanes ^ 2
    h = fmaxf(h, dpp<0x4E>(h));
    l = fminf(l, dpp<0x141>(l));                                   // the other half of 8 lanes
    h = fmaxf(h, dpp<0x141>(h));
    const int il = (int)floorf(__builtin_amdgcn_fmed3f(l - margin, -1.0e6f, 1.0e6f));
    const int ih = (int)floorf(__builtin_amdgcn_fmed3f(h + margin, -1.0e6f, 1.0e6f)) + 1;
    const int lb = __builtin_amdgcn_readlane(il, 0), hb = __builtin_amdgcn_readlane(ih, 0);
    const int lc = __builtin_amdgcn_readlane(il, 8), hc = __builtin_amdgcn_readlane(ih, 8);
    const int b0 = min(max(lb, 0), nB), b1 = min(max(hb, 1), nB + 1);
    const int c0 = min(max(lc, 0), nC), c1 = min(max(hc, 1), nC + 1);
    const int wb = whole ? min(hb - lb + 2, nB + 2) : b1 - b0 + 1, wc = whole ? min(hc - lc + 2, nC + 2) : c1 - c0 + 1;
    Box b;
    b.x0 = A == 0 ? a : b0;
    b.wx = A == 0 ? n + 1 : wb;
    b.y0 = A == 1 ? a : (A == 0 ? b0 : c0);
    b.wy = A == 1 ? n + 1 : (A == 0 ? wb : wc);
    b.z0 = A == 2 ? a : c0;
    b.wz = A == 2 ? n + 1 : wc;
    b.wx = max(b.wx, 2);
    b.wy = max(b.wy, 2);
    b.wz = max(b.wz, 2);
    b.pitch();
    return b;
  };
  // the most cells per slab whose box fits at both ends (the uncut widths are convex along A)
  int depth = 0;
  if (any && __builtin_amdgcn_readfirstlane(__all(ok && margin < 1.0f) ? 1 : 0)) {
    for (depth = (A == 0) ? kSlabDepthX : kSlabDepth; depth >= 1; depth = (depth >= 8) ? depth - 1 : depth >> 1) {
      const int n = min(depth, total);
      const Box b0 = box_of(alo, n, true), b1 = box_of(ahi + 1 - n, n, true);
      if (b0.wx <= 256 && b1.wx <= 256 && b0.floats() <= budget && b1.floats() <= budget) break;
    }
  }
  if (depth < 2) return cast_range<kGeom, kOp, kFmt>(it, ray, first, last, window);

  const auto src = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(it.raw), (short)0, (int)it.raw_bytes, 0x00020000);
  const float flast = (float)last, fseg_len = (float)seg_len(ray.n);
  float f = (first <= last) ? (float)first : flast + 1.0f;
  float fseg = 0.0f;
  float tot = line_init<kOp>(), acc = line_init<kOp>();
  Pos pos{ray.sx, ray.sy, ray.sz};
  const float qs = up ? sA : -sA, qd = up ? dA : -dA, qr = __builtin_amdgcn_rcpf(qd);
  const int lds_addr = (int)(uintptr_t)(__attribute__((address_space(3))) float*)lds;
  float q = fmaf(f, qd, qs);
  if (first <= last) {
    const int seg = seg_len(ray.n);
    fseg = fminf((float)((seg_of(first, seg) + 1) * seg - 1), flast);
    if constexpr (kGeom == XRH_GEOM_FP32) {
      pos.advance(ray, first);
      q = up ? pick(A, pos.x, pos.y, pos.z) : -pick(A, pos.x, pos.y, pos.z);
    }
  }
  for (int t = 0; t < total;) {
    const int n = min(depth, total - t), a = up ? alo + t : ahi + 1 - t - n;
    const Box b = box_of(a, n, false);
    __syncthreads();  // the previous slab has been read
    stage_box(src, b, it.raw_py, it.raw_pz, lds);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the clobber: no read of the box above the wait)
    __syncthreads();
    // samples of the slab: q below its far face, as one comparison
    const float face = up ? (float)(a + n) - kOff : -((float)a - kOff);
    const float lim = up ? (face > 0.0f ? __uint_as_float(__float_as_uint(face) - 1u) : -1.0e-30f) : face;
    float fslab = flast;
    if constexpr (kGeom == XRH_GEOM_FP64) {
      // the last of them: an estimate within one sample, corrected with the samples' own positions
      fslab = floorf((lim - qs) * qr);
      if (fmaf(fslab + 1.0f, qd, qs) <= lim) fslab = fslab + 1.0f;
      if (fmaf(fslab, qd, qs) > lim) fslab = fslab - 1.0f;
      fslab = fminf(fslab, flast);
    }
    // LDS byte address of cell (0, 0, 0), row and slice pitch
    const int py = b.sy * 4, pz = b.sz * 4;
    int base = lds_addr + (int)kOff * (4 + py + pz) - (b.x0 * 4 + py * b.y0 + pz * b.z0);
    asm("" : "+s"(base));  // one value: the compiler would subtract x0 per sample
    for (;;) {
      const float fstop = fminf(fslab, fseg);
      while (f <= fstop && (kGeom == XRH_GEOM_FP64 || q <= lim)) {
        float x, y, z;
        if constexpr (kGeom == XRH_GEOM_FP32) {
          x = pos.x;
          y = pos.y;
          z = pos.z;
        } else {
          x = fmaf(f, ray.dx, ray.sx);
          y = fmaf(f, ray.dy, ray.sy);
          z = fmaf(f, ray.dz, ray.sz);
        }
        float wx = __builtin_amdgcn_fractf(x), wy = __builtin_amdgcn_fractf(y), wz = __builtin_amdgcn_fractf(z);
        const int c00 = mad_i24(cvt_floor(z), pz, mad_i24(cvt_floor(y), py, (cvt_floor(x) << 2) + base));
        const int c10 = c00 + py, c01 = c00 + pz, c11 = c10 + pz;
        float va[4], vb[4];
        const LdsPair r00 = lds_pair(c00), r10 = lds_pair(c10), r01 = lds_pair(c01), r11 = lds_pair(c11);
        if constexpr (kFmt == 11) {
          va[0] = r00.a;
          vb[0] = r00.b;
          va[1] = r10.a - r00.a;
          vb[1] = r10.b - r00.b;
          va[2] = r01.a;
          vb[2] = r01.b;
          va[3] = r11.a - r01.a;
          vb[3] = r11.b - r01.b;
        } else {
          va[0] = r00.b - r00.a;
          va[1] = r10.b - r10.a;
          va[2] = r01.b - r01.a;
          va[3] = r11.b - r11.a;
        }
        auto value = [&] {
          if constexpr (kFmt == 11) return cell_value<11>(va, vb, wx, wy, wz);
          else return tri16_x(r00.a, va[0], r10.a, va[1], r01.a, va[2], r11.a, va[3], wx, wy, wz);
        };
        acc = line_op<kOp>(acc, value());
        f = f + 1.0f;
        if constexpr (kGeom == XRH_GEOM_FP32) {
          const float bx = x - wx, by = y - wy, bz = z - wz;  // floor
          pos.advance(ray, 1);
          q = q + qd;
          wx = pos.x - bx;
          wy = pos.y - by;
          wz = pos.z - bz;
        } else if constexpr (kFmt != 11) {
          // as the gathering march of these formats, from the sample's own position
          wx = fmaf(f, ray.dx, ray.sx) - (x - wx);
          wy = fmaf(f, ray.dy, ray.sy) - (y - wy);
          wz = fmaf(f, ray.dz, ray.sz) - (z - wz);
        } else {
          wx = wx + ray.dx;
          wy = wy + ray.dy;
          wz = wz + ray.dz;
        }
        const uint32_t top = max(max(__float_as_uint(wx), __float_as_uint(wy)), __float_as_uint(wz));
        if (top < 0x3f800000u && f <= fseg) {
          acc = line_op<kOp>(acc, value());
          f = f + 1.0f;
          if constexpr (kGeom == XRH_GEOM_FP32) {
            pos.advance(ray, 1);
            q = q + qd;
          }
        }
      }
      // a lane that reached the end of its segment goes on to the next one in this slab
      const bool roll = f > fseg && f <= flast;
      if (f > fseg) {
        tot = line_op<kOp>(tot, acc);
        acc = line_init<kOp>();
        fseg = (f > flast) ? 3.0e38f : fminf(fseg + fseg_len, flast);
      }
      if (!__any(roll)) break;
    }
    t += n;
  }
  return (ray.n >= 0) ? tot * it.step : line_init<kOp>();
}

// The same ray shared by kParts waves of a workgroup of kParts * 256 threads (thread t: pixel
// t % 256, part t / 256): part p sums segments p, p + kParts, ... and every part adds all
// segments in order, so the value is cast_ray's bit for bit. The first two parts walk over the
// empty space from one end each. Every thread of the block calls it (it synchronises).
template <int kGeom, int kOp, int kFmt, int kParts>
__device__ __forceinline__ float cast_ray_split(const DrrItem& it, int col, int row, bool inside, int window)
{
  static_assert(kParts >= 2 && kSegs % kParts == 0, "segments are dealt evenly");
  __shared__ float sums[kSegs][kThreads];
  __shared__ int ends[2][kThreads];
  const int px = threadIdx.x & (kThreads - 1), part = threadIdx.x / kThreads;
  Ray ray;
  ray.n = -1;
  if (inside) {
    ray = (kGeom == XRH_GEOM_FP32) ? setup_ray_f32(it, (float)col, (float)row) : setup_ray_f64(it, col, row);
  }
  const bool skip = kOp == XRH_LINE_INT_SUM && it.skip;
  int first = 0, last = ray.n;
  if (skip) {
    const float org = (kGeom == XRH_GEOM_FP64) ? 1.0f : 0.0f;
    if (part == 0) ends[0][px] = (ray.n >= 0) ? skip_empty(it, ray, 0, ray.n, 1, org) : 0;
    if (part == 1) ends[1][px] = (ray.n >= 0) ? skip_empty(it, ray, ray.n, 0, -1, org) : -1;
    __syncthreads();
    first = ends[0][px];
    last = ends[1][px];
  }
  const int seg = seg_len(ray.n);
  Pos pos{ray.sx, ray.sy, ray.sz};
  int at = 0;
#pragma clang loop unroll(disable)
  for (int k = part; k < kSegs; k += kParts) {
    const int i = max(first, k * seg), stop = min(last, k * seg + seg - 1);
    float acc = line_init<kOp>();
    if (i <= stop) {
      if constexpr (kGeom == XRH_GEOM_FP32) pos.advance(ray, i - at);
      acc = march<kGeom, kOp, kFmt>(ray, vol_view(it), pos, i, stop, seg, i, window);
      at = stop + 1;
    }
    sums[k][px] = acc;
  }
  __syncthreads();
  float acc = line_init<kOp>();
  if (ray.n >= 0) {
#pragma unroll
    for (int k = 0; k < kSegs; ++k) acc = line_op<kOp>(acc, sums[k][px]);
    acc = acc * it.step;
  }
  __syncthreads();  // the next object's cast reuses the shared arrays
  return acc;
}

// kParts: the waves that share a ray, 0 for slab marching with `budget` floats of dynamic LDS. Rays
// that gather by cells wait for each other every `window` samples.
template <int kGeom, int kOp, int kFmt, int kParts>
__device__ __forceinline__ float cast_pixel(const DrrItem& it, const TileRef& tr, int col, int row, bool inside,
                                            int budget, int window)
{
  if constexpr (kParts == 0) {
    extern __shared__ __attribute__((aligned(16))) float box_lds[];
    return cast_ray_slab<kGeom, kOp, kFmt>(it, tr, col, row, inside, box_lds, budget, window);
  } else if constexpr (kParts == 1) return cast_ray<kGeom, kOp, kFmt>(it, col, row, inside, window);
  else return cast_ray_split<kGeom, kOp, kFmt, kParts>(it, col, row, inside, window);
}

template <int kGeom, int kOp, int kFmt, int kParts>
__global__ __launch_bounds__(kThreads * (kParts > 1 ? kParts : 1), kParts == 0 ? 4 : 8) void drr_kernel(
    const DrrItem* __restrict__ items, const uint32_t* __restrict__ band_start, int64_t num_items,
    int bands, float* __restrict__ out, int accumulate, float fill,
    double* __restrict__ ncc_partials, int ncc_tiles, int shape, int budget, int window)
{
  const TileRef tr = decode_tile(band_start, num_items, bands, items);
  if (!tr.valid) return;
  const DrrItem& it = items[tr.item];
  int col, row;
  lane_pixel(tr.tx, tr.ty, shape, col, row);
  const bool inside = (col < it.cam.cols) && (row < it.cam.rows);
  const float acc = cast_pixel<kGeom, kOp, kFmt, kParts>(it, tr, col, row, inside, budget, window);
  // the first part stores the pixels
  const bool mine = inside && (kParts <= 1 || threadIdx.x < kThreads);
  store_pixel<kOp>(it, tr, mine, col, row, acc, out, accumulate, fill, ncc_partials, ncc_tiles);
}

// Several objects per item (Intensity2D3DRegi::obj_fn with more than one volume,
// xregIntensity2D3DRegi.cpp:598-629): entries item * objs + k, k = 0..objs-1, are cast in
// object order into the item's pixels, the first onto its background image (or `fill`), the
// others added with the line kernel -- per pixel the same float operations as one REPLACE
// launch followed by ACCUM launches. The item's first entry carries the output offset, the
// detector and the fused NCC reference.
template <int kGeom, int kOp, int kFmt, int kParts>
__global__ __launch_bounds__(kThreads * (kParts > 1 ? kParts : 1), kParts == 0 ? 7 : 8) void drr_objects_kernel(
    const DrrItem* __restrict__ items, const uint32_t* __restrict__ band_start, int64_t num_items,
    int bands, float* __restrict__ out, float fill, double* __restrict__ ncc_partials, int ncc_tiles,
    int shape, int budget, int window, int objs)
{
  const TileRef tr = decode_tile(band_start, num_items, bands, items, objs);
  if (!tr.valid) return;
  const DrrItem& it0 = items[tr.item * objs];
  int col, row;
  lane_pixel(tr.tx, tr.ty, shape, col, row);
  const bool inside = (col < it0.cam.cols) && (row < it0.cam.rows);
  const int64_t px = (int64_t)row * it0.cam.cols + col;
  float pix = 0.0f;
  if (inside) pix = it0.bg ? it0.bg[px] : fill;
  for (int k = 0; k < objs; ++k) {
    const float aa =
        0.0f + cast_pixel<kGeom, kOp, kFmt, kParts>(items[tr.item * objs + k], tr, col, row, inside, budget, window) * 1.0f;
    if (inside) {
      if constexpr (kOp == XRH_LINE_INT_SUM) pix = pix + aa; else pix = (pix < aa) ? aa : pix;
    }
    if constexpr (kParts == 0) __syncthreads();  // the next cast reuses the shared arrays
  }
  const bool mine = inside && (kParts <= 1 || threadIdx.x < kThreads);
  if (mine) out[it0.out_off + px] = pix;
  ncc_epilogue(it0, tr, mine, col, row, pix, ncc_partials, ncc_tiles);
}

template <int kGeom>
__global__ __launch_bounds__(kThreads) void drr_count_kernel(
    const DrrItem* __restrict__ items, const uint32_t* __restrict__ band_start, int64_t num_items,
    int bands, unsigned long long* __restrict__ counter, int32_t* __restrict__ steps)
{
  const TileRef tr = decode_tile(band_start, num_items, bands, items);
  if (!tr.valid) return;
  const DrrItem& it = items[tr.item];
  int col, row;
  lane_pixel(tr.tx, tr.ty, 0, col, row);
  double cnt = 0.0, evaluated = 0.0;
  if ((col < it.cam.cols) && (row < it.cam.rows)) {
    const Ray ray = (kGeom == XRH_GEOM_FP32) ? setup_ray_f32(it, (float)col, (float)row) : setup_ray_f64(it, col, row);
    if (steps) steps[it.out_off + (int64_t)row * it.cam.cols + col] = ray.n;
    cnt = (double)(ray.n + 1);
    if (ray.n >= 0) {
      int first, last;
      sample_range<XRH_LINE_INT_SUM, kGeom>(it, ray, first, last);
      evaluated = (double)(last - first + 1);
    }
  }
  cnt = wave_sum_d(cnt);
  evaluated = wave_sum_d(evaluated);
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&counter[0], (unsigned long long)cnt);
    atomicAdd(&counter[1], (unsigned long long)evaluated);
  }
}

// Compute units of the current device (cached per device).
int device_cus()
{
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cache[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev] = n;
  }
  return cache[dev];
}

// Waves that share a ray in a launch of `tiles` workgroups: the most for which all of them are
// resident at once (32 waves per CU). A launch of few rays is bound by the longest rays' chain of
// dependent gathers and by idle CUs, which sharing shortens and fills; one that fills the GPU
// only pays for the shared set-up (30 items of 256 x 256, two objects: 1.07 ms whole, 1.22 ms by
// two). One pose, FP64 set-up, DRR kernel: 192 x 192 over 128 x 128 x 96 voxels 30.5
// whole, 27.2 by two, 21.4 by four; 384 x 384 over 256 x 256 x 200 voxels 102, 80, 90 us.
//
// Rays `spacing` voxels apart (0: not known) share no cache lines, and waves at several depths of the
// same rays then evict each other's: over 512 tiles a wave takes whole rays from 0.95 voxels on (us,
// shared by two / whole: 546 tiles at 1.94 voxels 478 / 386, 686 at 2.26 1037 / 790, 624 at 1.0 510 /
// 387); up to 512 FP32 rays are shared by four while there are few or they are close, else by two (four /
// two: 252 tiles at 1.03 80 / 95, 64 at 1.88 217 / 240, 128 at 1.88 214 / 227, 100 at 3.0 248 / 259, 200 at 3.0 243 /
// 239, 507 at 1.01 177 / 161; whole / two: 72 at 2.77 427 / 260, 200 at 2.66 339 / 275), and 16-bit rays, with half the loads, by four up to
// 1.75 voxels (210 tiles at 1.67 four / two 111 / 117), from there by two only up to 128 tiles (whole / two:
// 50 at 3.76 286 / 263, 280 at 3.22 267 / 281, 440 at 1.82 181 / 199).
// Where rays are close and gather, sharing by two pays up to twice as many tiles (16-bit, whole / shared:
// 1392 at 0.39 345 / 321, 1440 at 0.31 207 / 178, 1736 at 0.36 162 / 146, 1596 at 0.45 217 / 203).
int drr_parts(int64_t tiles, float spacing, int slab, int32_t storage)
{
  const int64_t waves = tiles * (kThreads / 64), room = 32ll * device_cus();
  if (waves * 4 <= room) {
    if (storage != XRH_F32) return spacing < 1.75f ? 4 : (waves * 16 <= room ? 2 : 1);
    return (spacing < 0.95f || waves * (spacing < 1.65f ? 8 : 16) <= room) ? 4 : 2;
  }
  if (slab == 0 && spacing > 0.0f && spacing < 0.75f && waves <= room) return 2;
  return (waves * 2 <= room && spacing < 0.95f) ? 2 : 1;
}

// LDS bytes of a workgroup's boxes for rays `spacing` voxels apart: eight, four or three workgroups per CU,
// with the 272 bytes that the kernel holds beside them.
int slab_lds(float spacing)
{
  return !(spacing > 0.0f) ? 0 : (spacing < 0.95f ? 20160 : (spacing < 2.7f ? 40640 : 54208));
}

// Samples between the points where the lanes of whole rays gathering by cells wait for each other. In
// step, lanes touch the fewest cache lines; apart, every iteration keeps all lanes loading, at two samples
// a load where the cells allow it. Close rays share lines over many samples, sparse rays none over more than
// one. us with windows of 16, 8, 4 and 1 samples, by voxels between rays, over 215 MB / 1.7 GB of faces: 0.39
// 554, 559, 609, 748 / 1441, 1504, 1661, 2041; 0.47 574, 570, 618, 743 / 1178, 1167, 1274, 1568; 0.58 671, 633,
// 658, 770 / 1067, 984, 995, 1176; 0.67 794, 705, 692, 785 / 1221, 1075, 1042, 1188; 0.78 969, 873, 817, 814 /
// 1466, 1316, 1210, 1249; 0.93 1203, 1117, 1054, 912 / 1983, 1816, 1670, 1461; with the LDS of gather_lds 1.16
// 1268, 1221, 1250, 1422 and 1.55 1849, 1783, 1757, 1618. (26 MB: 0.39 313, 323, 355, 423; 0.78 448, 411, 411, 449;
// 1.55 886, 834, 789, 708.) Bricks and coefficients spread a cell's neighbours over more lines and want the
// lanes in step earlier (1.7 GB of faces: bricks 0.58 1287, 1217, 1202, 1316, 0.67 1467, 1417, 1362, 1369, 0.78 1978,
// 1820, 1733, 1623; coefficients 0.58 1398, 1318, 1252, 1299, 0.67 1659, 1515, 1402, 1335).
int gather_window(float spacing, int32_t layout)
{
  const bool face = layout == kLayoutFace;
  if (!(spacing >= 0.45f)) return kWindow;
  if (spacing < (face ? 0.63f : 0.55f)) return 8;
  if (spacing < (face ? 0.85f : 0.63f)) return 4;
  return (spacing >= 1.1f && spacing < 1.45f) ? 4 : 1;
}

// LDS bytes that a workgroup of whole gathered rays reserves, unused, over a volume that the caches do not
// hold: from about a voxel between rays on, four workgroups on a CU leave each other's lines in its L1 and
// take less time than eight, and from 2.7 voxels on three (us without / with 40 / 54 KB, 215 MB of faces, the
// best window of each: 1.03 voxels 1100 / 1091 / - , 1.16 1330 / 1221 / 1737, 1.55 1941 / 1618 / 1926, 3.1 3888 /
// 3340 / 3176; f16 cells 0.78 718 / 731 / 1260, 1.16 1355 / 1123 / 1381, 1.55 1963 / 1665 / 1648, 3.1 4387 / 3788 /
// 3388).
int gather_lds(float spacing) { return (spacing >= 1.1f) ? slab_lds(spacing) : 0; }

// The same where four waves share a ray: they are at four depths of it, and sparse rays meet no lines of each
// other's (us, 16 / 4 / 1 samples: 128 tiles at 1.16 voxels 92 / 97 / 114, 72 at 1.43 116 / 111 / 110, at 1.55 102 / 102 /
// 116, 64 at 1.88 232 / 217 / 218, at 2.33 122 / 114 / 120, 100 at 3.0 282 / 257 / 248).
int shared_window(float spacing) { return spacing >= 2.7f ? 1 : (spacing >= 1.3f ? 4 : kWindow); }

// How a launch marches. Slabs need the plain voxels of every volume beside a face or oct layout.
struct March {
  int parts;   // waves that share a ray
  bool slabs;  // whole rays by slabs
  int lds;     // dynamic LDS bytes: the boxes of the slabs, or held unused by whole rays that gather
  int window;  // samples between the points where a wave's lanes wait
};

March drr_march(const DrrLaunch& L, int64_t tiles)
{
  // XRH_CELL_REUSE=0 / =1 force shared rays / whole rays, by slabs whatever the sizes (read per launch, so
  // a process can switch between calls); otherwise a tuned variant decides, else the launch
  const char* env = std::getenv("XRH_CELL_REUSE");
  const int reuse = env ? (std::strcmp(env, "0") != 0 ? 1 : 0) : L.reuse;
  const bool able = L.plain && (L.storage == XRH_F32 ? L.layout == kLayoutFace : L.layout == kLayoutOct);
  const int slab = !able ? 0
                   : (env && reuse > 0) ? slab_lds(L.ray_spacing)
                                        : drr_slab_lds(L.ray_spacing, L.geom, L.vol_bytes, L.storage, tiles);
  March m;
  m.parts = (reuse > 0) ? 1 : (reuse == 0) ? std::max(drr_parts(tiles, 0.0f, 0, L.storage), 2)
                                           : drr_parts(tiles, L.ray_spacing, slab, L.storage);
  m.slabs = m.parts == 1 && slab > 0;
  m.lds = m.slabs ? slab : 0;
  m.window = m.parts == 1 ? gather_window(L.ray_spacing, L.layout) : (m.parts == 4 ? shared_window(L.ray_spacing) : kWindow);
  // (launches that could go by slabs and do not are better off without)
  if (!able && m.parts == 1 && L.vol_bytes >= kSlabBytes &&
      (L.storage == XRH_F32 ? L.layout != kLayoutQuad && L.layout != kLayoutLinear : L.layout == kLayoutOct)) {
    m.lds = gather_lds(L.ray_spacing);
  }
  return m;
}

}  // namespace

int64_t drr_launch_plan(const DrrLaunch& L)
{
  const March m = drr_march(L, L.max_band_tiles * L.bands);
  return ((int64_t)m.lds * 64 + m.window) * 16 + m.parts * 2 + (m.slabs ? 1 : 0);
}

namespace {

template <int kGeom, int kOp>
void launch_fmt(const DrrLaunch& L, dim3 grid, hipStream_t s, int accumulate, float fill)
{
#define XRH_LAUNCH_PARTS(F, P)                                                                        \
  do {                                                                                                \
    const dim3 threads(kThreads * (P > 1 ? P : 1));                                                   \
    if (L.objs > 1) {                                                                                 \
      hipLaunchKernelGGL((drr_objects_kernel<kGeom, kOp, F, P>), grid, threads, m.lds, s, L.items_dev,  \
                         L.band_start_dev, L.num_items, L.bands, L.out, fill, L.ncc_partials,         \
                         L.ncc_tiles_per_item, shape, m.lds / 4, m.window, L.objs);                   \
    } else {                                                                                          \
      hipLaunchKernelGGL((drr_kernel<kGeom, kOp, F, P>), grid, threads, m.lds, s, L.items_dev,          \
                         L.band_start_dev, L.num_items, L.bands, L.out, accumulate, fill,             \
                         L.ncc_partials, L.ncc_tiles_per_item, shape, m.lds / 4, m.window);            \
    }                                                                                                 \
  } while (0)
#define XRH_LAUNCH_FMT(F)                         \
  do {                                            \
    if (m.parts == 4) XRH_LAUNCH_PARTS(F, 4);     \
    else if (m.parts == 2) XRH_LAUNCH_PARTS(F, 2); \
    else XRH_LAUNCH_PARTS(F, 1);                  \
  } while (0)
  const int shape = (L.wave_shape >= 0 && L.wave_shape <= 2) ? L.wave_shape : 0;
  const int fmt = (L.storage == XRH_F32)
                      ? (L.layout == kLayoutCoef ? 7
                                                 : (L.layout == kLayoutFace ? 11
                                                    : (L.layout == kLayoutBrick ? 13
                                                                                : (L.layout == kLayoutQuad ? 1 : 0))))
                : (L.storage == XRH_F16) ? (L.layout == kLayoutOct ? 3 : 2)
                                         : (L.layout == kLayoutOct ? 5 : 4);
  const March m = drr_march(L, (int64_t)grid.x * grid.y);
  if (m.slabs) {
    if (fmt == 11) XRH_LAUNCH_PARTS(11, 0);
    else if (fmt == 3) XRH_LAUNCH_PARTS(3, 0);
    else XRH_LAUNCH_PARTS(5, 0);
    return;
  }
  switch (fmt) {
    case 0: XRH_LAUNCH_FMT(0); break;
    case 1: XRH_LAUNCH_FMT(1); break;
    case 2: XRH_LAUNCH_FMT(2); break;
    case 3: XRH_LAUNCH_FMT(3); break;
    case 4: XRH_LAUNCH_FMT(4); break;
    case 5: XRH_LAUNCH_FMT(5); break;
    case 7: XRH_LAUNCH_FMT(7); break;
    case 13: XRH_LAUNCH_FMT(13); break;
    default: XRH_LAUNCH_FMT(11); break;
  }
#undef XRH_LAUNCH_FMT
#undef XRH_LAUNCH_PARTS
}

}  // namespace

// LDS bytes of a slab-marching launch whose rays are `spacing` voxels apart on average (0: not
// known) and whose largest volume's face layout has `bytes`; 0 to gather. Gathering stays the
// better march for close rays over a volume that the caches hold (0.39 voxels apart, ns per ray
// by gathering / slabs: 26 MB of faces 0.190 / 0.197 with FP64 set-up, 0.191 / 0.219 with FP32;
// 215 MB 0.355 / 0.330 and 0.357 / 0.371; 1.7 GB 0.748 / 0.554 and 0.753 / 0.632). Otherwise eight
// workgroups per CU (the most) while the boxes are small; four where the rays are about a voxel
// apart and more, for boxes of several layers; three past the point where most boxes no longer fit
// and the tiles gather, for which fewer waves per L1 are the better choice. ns per ray with 20 /
// 40 / 54 KB: 256 x 256 x 200 voxels at 0.58 voxels 0.397 / 0.485 / 0.758, at 0.78 0.440 / 0.516 /
// 0.828, at 1.16 0.787 / 0.625 / 0.940, at 1.55 1.30 / 1.05 / 1.29, at 2.3 2.22 / 1.91 / 2.28; 512 x
// 512 x 400 voxels at 3.1 6.06 / 5.66 / 5.32.
//
// Volumes of under 64 MB (kSlabBytes) gather at any distance (40 MB, 2016 tiles at 0.70 voxels: 179 / 211 us).
// With 16-bit storage a gathered sample is one load instead of an FP32 cell's two, so slabs pay later
// (ns per ray by gathering / slabs, f16): 215 MB, FP64 set-up, at 0.19 voxels 0.315 / 0.316, 0.39 0.348 /
// 0.360, 0.58 0.364 / 0.401, 0.78 0.495 / 0.440, 1.55 1.31 / 1.02; FP32 set-up 0.39 0.32 / 0.38, 0.78
// 0.49 / 0.45, 1.55 1.29 / 1.05. 1.7 GB, FP64: 0.39 0.65 / 0.60, 0.78 1.13 / 0.80, 1.55 3.1 / 1.8. 26
// MB: 0.39 0.209 / 0.219, 0.78 0.233 / 0.279, 1.55 0.47 / 0.62. They also need more tiles, for the four
// workgroups per CU that their boxes leave room for: 112 MB, 2360 tiles at 1.71 428 / 592 us; 289 MB,
// 2430 at 0.84 339 / 382; 556 MB, 2112 at 1.60 1019 / 937.
int drr_slab_lds(float spacing, int32_t geom, uint64_t bytes, int32_t storage, int64_t tiles)
{
  if (!(spacing > 0.0f) || bytes < kSlabBytes) return 0;
  const bool fp32 = geom == XRH_GEOM_FP32;
  if (storage == XRH_F32) {
    if (fp32 && spacing < 0.5f && bytes < (256ull << 20)) return 0;
  } else {
    const bool large = bytes >= (512ull << 20);
    const int64_t cus = device_cus();
    if (spacing < 0.7f && (fp32 || !large)) return 0;
    if (tiles < (large ? 8 : 16) * cus || bytes < (128ull << 20)) return 0;
  }
  return slab_lds(spacing);
}

bool drr_whole_rays(const DrrLaunch& L) { return drr_march(L, L.max_band_tiles * L.bands).parts == 1; }

std::string drr_tune_key(const DrrLaunch& L, int32_t max_rows, int32_t max_cols, int64_t workgroups)
{
  auto octave = [](double x) { return x > 0.0 ? std::ilogb(x) : INT_MIN; };
  const int per_cu = octave((double)(workgroups / std::max(device_cus(), 1)));
  const int spacing = L.ray_spacing > 0.0f ? octave((double)L.ray_spacing * L.ray_spacing) : INT_MIN;  // half octaves
  std::string key;
  for (int64_t v : {(int64_t)L.storage, (int64_t)L.layout, (int64_t)L.geom, (int64_t)L.kernel,
                    (int64_t)std::max(L.objs, 1), (int64_t)L.plain, (int64_t)max_rows, (int64_t)max_cols,
                    (int64_t)per_cu, (int64_t)octave((double)L.vol_bytes), (int64_t)spacing}) {
    key += std::to_string(v) + " ";
  }
  return key;
}

TilePlan build_tiles(const std::vector<int32_t>& rows, const std::vector<int32_t>& cols, int32_t bands)
{
  TilePlan p;
  p.bands = bands < 1 ? 1 : bands;
  const int64_t n = (int64_t)rows.size();
  p.band_start.assign((size_t)p.bands * (n + 1), 0);
  p.max_band_tiles = 0;
  for (int b = 0; b < p.bands; ++b) {
    uint32_t acc = 0;
    for (int64_t i = 0; i < n; ++i) {
      const int tiles = ((cols[i] + kTile - 1) / kTile) * ((rows[i] + kTile - 1) / kTile);
      p.band_start[(size_t)b * (n + 1) + i] = acc;
      acc += band_first_tile(i, tiles, b + 1, p.bands) - band_first_tile(i, tiles, b, p.bands);
    }
    p.band_start[(size_t)b * (n + 1) + n] = acc;
    if ((int64_t)acc > p.max_band_tiles) p.max_band_tiles = acc;
  }
  return p;
}

void launch_drr_setup(const DrrLaunch& L, hipStream_t s, const SetupCopy& copy)
{
  if (L.num_items <= 0) return;
  const int64_t entries = L.num_items * (L.objs > 1 ? L.objs : 1);
  const int64_t item_blocks = (entries + kSetupItems - 1) / kSetupItems;
  const int64_t copy_blocks = (int64_t)((copy.words[0] + copy.words[1] + kSetupCopy - 1) / kSetupCopy);
  hipLaunchKernelGGL(drr_setup_kernel, dim3((unsigned)(item_blocks + copy_blocks)), dim3(kSetupThreads), 0, s,
                     L.poses_dev, L.vols_dev, L.cams_dev, L.items_dev, entries, (int)item_blocks, copy);
  XRH_HIP_CHECK(hipGetLastError());
}

void launch_drr(const DrrLaunch& L, hipStream_t s)
{
  if (L.num_items <= 0 || L.max_band_tiles <= 0) return;
  const int64_t nblocks = L.max_band_tiles * L.bands;
  XRH_REQUIRE(nblocks < (int64_t)INT32_MAX, "too many DRR tiles in one launch");
  const dim3 grid((unsigned)nblocks);
  if (L.sample_counter) {
    XRH_REQUIRE(L.objs <= 1, "sample counts are taken per single-object item");
    if (L.geom == XRH_GEOM_FP32) {
      hipLaunchKernelGGL((drr_count_kernel<XRH_GEOM_FP32>), grid, dim3(kThreads), 0, s, L.items_dev,
                         L.band_start_dev, L.num_items, L.bands,
                         (unsigned long long*)L.sample_counter, L.ray_steps);
    } else {
      hipLaunchKernelGGL((drr_count_kernel<XRH_GEOM_FP64>), grid, dim3(kThreads), 0, s, L.items_dev,
                         L.band_start_dev, L.num_items, L.bands,
                         (unsigned long long*)L.sample_counter, L.ray_steps);
    }
    XRH_HIP_CHECK(hipGetLastError());
    return;
  }
  const int accumulate = (L.store == XRH_STORE_ACCUM) ? 1 : 0;
  const float fill = L.fill;
  if (L.geom == XRH_GEOM_FP32) {
    if (L.kernel == XRH_LINE_INT_SUM) launch_fmt<XRH_GEOM_FP32, XRH_LINE_INT_SUM>(L, grid, s, accumulate, fill);
    else launch_fmt<XRH_GEOM_FP32, XRH_LINE_INT_MAX>(L, grid, s, accumulate, fill);
  } else {
    if (L.kernel == XRH_LINE_INT_SUM) launch_fmt<XRH_GEOM_FP64, XRH_LINE_INT_SUM>(L, grid, s, accumulate, fill);
    else launch_fmt<XRH_GEOM_FP64, XRH_LINE_INT_MAX>(L, grid, s, accumulate, fill);
  }
  XRH_HIP_CHECK(hipGetLastError());
}

}  // namespace xrh
