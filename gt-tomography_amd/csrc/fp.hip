// Ray-driven cone-beam forward projector for gfx950.
//
// Math: xray/conebeam_projection.cu:412-528 (one ray per detector pixel, the
// source->pixel segment clipped to the volume box by the slab method,
// n = int(samples_per_pixel*nx) left-Riemann trilinear samples, result scaled
// by the step length in mm).
//
// Common design
//  * The per-ray setup (rotation, slab clipping, step length, start point and
//    increment in texel space) runs in FP64, once per ray.  Only the sample
//    loop is FP32.  Each sample position is p0 + m*q with one FMA per axis, so
//    coordinate error does not grow along the ray.
//  * Interpolation is done by hand (no texture unit) from a zero-bordered copy
//    of the volume (1 voxel before, 2 after on every axis): coordinates are
//    clamped to [-1, n] and the border supplies the zeros of the reference's
//    border addressing mode, so the inner loops carry no bounds tests.
//  * Storage may be FP32 or BF16 (arithmetic is FP32 either way).
//
// Engine 1 (default): detector-column sharing.
//  All rays of one detector column (one view, one u) lie in the vertical plane
//  through the source.  Their x/y slab limits are identical, and the z slab
//  never raises a1 (its lower limit is <= 0), so unless a ray leaves through
//  the top or bottom face its (a1, a2) -- and therefore its x/y sample
//  positions -- equal the column's at every step m.  One wave owns a column:
//  per step it bilinearly interpolates the z-line at the shared (x, y) from a
//  z-fastest copy of the volume (coalesced loads, 64 consecutive z per
//  instruction) into LDS, and every ray then does one z-lerp from LDS.  The
//  arithmetic order (x-lerps, y-lerp, z-lerp) and sample coordinates are those
//  of engine 0, so both engines produce bitwise-identical projections.  Rays
//  clipped by the z slab are taken 8 samples of 8 rays at a time (fp_gather),
//  where they are many by a kernel of their own (k_fp_clip).  Blocks are remapped
//  so each XCD walks a contiguous run of columns (neighbouring columns share
//  z-lines in that XCD's L2).
//
// Engine 0: one thread per ray, 16x16 detector tiles, x-fastest padded
// volume, 8 gathers per sample.  Also the basis of the exact transpose.
#include <algorithm>
#include <climits>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "cbct_internal.h"
#include "fp_cells.h"

// Working copy of cbct_fp_noalloc: device memory the library owns for the
// life of the process (one copy per GPU, each at its own address), so that
// call allocates nothing.  Host code uses the per-device address from
// hipGetSymbolAddress, never this name.
constexpr size_t FP_SCRATCH_BYTES = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[FP_SCRATCH_BYTES];

namespace {

struct FPParams {
  int nu, nv, n;
  int nx, ny, nz;
  unsigned px, pxy;           // x-fastest padded strides (elements)
  unsigned pz, pzx;           // z-fastest padded strides: z + pz*(x + px*y)
  double lx, ly, lz;
  double fu, fv, sad, sdd;
  float cx, cy, cz;           // clamp limits in padded texel space (= n_axis + 1)
  unsigned vg;                // column engine: views per launch group (see col_block)
  unsigned lds_stp;           // column engine: floats of LDS before the parked step lengths
  int split;                  // column engine: rays not shared are k_fp_clip's
};

template <typename T>
__device__ __forceinline__ float ld(const T *p, unsigned i);
template <>
__device__ __forceinline__ float ld<float>(const float *p, unsigned i) {
  return p[i];
}
template <>
__device__ __forceinline__ float ld<unsigned short>(const unsigned short *p, unsigned i) {
  return bf16_to_f32(p[i]);
}

// Ray setup in FP64.  Every engine takes its parameters from these functions,
// and only the explicit fma calls fuse, so that the same ray has the same bits
// whatever surrounds the call.

// Column part (shared by every ray with detector column i).
struct ColSetup {
  double S0, S1, d0, d1, dd, lo, hi;  // dd: d0^2 + d1^2; lo/hi: slab limits from the x and y faces
};

__device__ __forceinline__ ColSetup col_setup(const FPParams &P, const ViewD &vw, int i) {
#pragma clang fp contract(off)
  ColSetup C;
  const double c = vw.c, s = vw.s;
  C.S0 = s * P.sad;  // R(theta) (0,-SAD,0)
  C.S1 = -c * P.sad;
  const double pu = fma((i + 0.5) / P.nu - 0.5, P.fu, vw.off_u);
  const double add = P.sdd - P.sad;
  C.d0 = fma(c, pu, -(s * add)) - C.S0;
  C.d1 = fma(s, pu, c * add) - C.S1;
  C.dd = fma(C.d1, C.d1, C.d0 * C.d0);
  const double hx = P.lx * 0.5, hy = P.ly * 0.5;
  double tA = (hx - C.S0) / C.d0, tB = (-hx - C.S0) / C.d0;
  C.lo = fmin(tB, tA);
  C.hi = fmax(tB, tA);
  tA = (hy - C.S1) / C.d1;
  tB = (-hy - C.S1) / C.d1;
  C.lo = fmax(C.lo, fmin(tB, tA));
  C.hi = fmin(C.hi, fmax(tB, tA));
  return C;
}

// Detector height of row j.
__device__ __forceinline__ double row_height(const FPParams &P, const ViewD &vw, int j) {
#pragma clang fp contract(off)
  return fma((j + 0.5) / P.nv - 0.5, P.fv, vw.off_v);
}

// Start, increment (in texel space: normalised * N - 0.5, plus 1 for the leading
// zero border) and step length of the n samples on [a1, a2]; span = a2 - a1, h =
// span / n.  The x/y part does not depend on the row.
__device__ __forceinline__ void ray_xy(const FPParams &P, const ColSetup &C, double a1, double h,
                                       float &px, float &qx, float &py, float &qy) {
#pragma clang fp contract(off)
  px = (float)fma(fma(a1, C.d0, C.S0) / P.lx + 0.5, (double)P.nx, 0.5);
  py = (float)fma(fma(a1, C.d1, C.S1) / P.ly + 0.5, (double)P.ny, 0.5);
  qx = (float)(C.d0 / P.lx * h * P.nx);
  qy = (float)(C.d1 / P.ly * h * P.ny);
}
__device__ __forceinline__ void ray_z(const FPParams &P, const ColSetup &C, double d2, double a1,
                                      double span, double h, float &pz, float &qz, float &step) {
#pragma clang fp contract(off)
  pz = (float)fma((a1 * d2) / P.lz + 0.5, (double)P.nz, 0.5);
  qz = (float)(d2 / P.lz * h * P.nz);
  step = (float)(sqrt(fma(d2, d2, C.dd)) * fabs(span) / P.n);
}

struct RaySetup {
  float p[3], q[3], step;
};

// Row j's ray of the column: clipped to the z slab [-t, t], sampled.
__device__ __forceinline__ RaySetup ray_finish(const FPParams &P, const ViewD &vw,
                                               const ColSetup &C, int j) {
#pragma clang fp contract(off)
  RaySetup R;
  const double d2 = row_height(P, vw, j);
  const double t = fabs(P.lz * 0.5 / d2);
  const double a1 = fmax(fmax(C.lo, -t), 0.0);
  const double a2 = fmin(fmin(C.hi, t), 1.0);
  const double span = a2 - a1, h = span / P.n;
  ray_xy(P, C, a1, h, R.p[0], R.q[0], R.p[1], R.q[1]);
  ray_z(P, C, d2, a1, span, h, R.p[2], R.q[2], R.step);
  return R;
}

__device__ __forceinline__ float clampf(float v, float hi) { return fminf(fmaxf(v, 0.0f), hi); }

// ------------------------------------------------------------------ engine 0
template <typename T>
__global__ void __launch_bounds__(256) k_fp_ray(FPParams P, const ViewD *__restrict__ views,
                                                const T *__restrict__ vol, float *__restrict__ proj,
                                                int accumulate) {
  const int i = blockIdx.x * 16 + threadIdx.x;
  const int j = blockIdx.y * 16 + threadIdx.y;
  const int k = blockIdx.z;
  if (i >= P.nu || j >= P.nv) return;
  const ViewD vw = views[k];
  const RaySetup R = ray_finish(P, vw, col_setup(P, vw, i), j);
  float acc = 0.0f;
  const unsigned px = P.px, pxy = P.pxy;
  for (int m = 0; m < P.n; ++m) {
    const float fm = (float)m;
    const float sx = clampf(fmaf(fm, R.q[0], R.p[0]), P.cx);
    const float sy = clampf(fmaf(fm, R.q[1], R.p[1]), P.cy);
    const float sz = clampf(fmaf(fm, R.q[2], R.p[2]), P.cz);
    const float flx = floorf(sx), fly = floorf(sy), flz = floorf(sz);
    const float ax = sx - flx, ay = sy - fly, az = sz - flz;
    const unsigned base = (unsigned)flx + px * (unsigned)fly + pxy * (unsigned)flz;
    const float v000 = ld(vol, base), v100 = ld(vol, base + 1);
    const float v010 = ld(vol, base + px), v110 = ld(vol, base + px + 1);
    const float v001 = ld(vol, base + pxy), v101 = ld(vol, base + pxy + 1);
    const float v011 = ld(vol, base + pxy + px), v111 = ld(vol, base + pxy + px + 1);
    const float c00 = fmaf(ax, v100 - v000, v000);
    const float c10 = fmaf(ax, v110 - v010, v010);
    const float c01 = fmaf(ax, v101 - v001, v001);
    const float c11 = fmaf(ax, v111 - v011, v011);
    const float c0 = fmaf(ay, c10 - c00, c00);
    const float c1 = fmaf(ay, c11 - c01, c01);
    acc += fmaf(az, c1 - c0, c0);
  }
  const size_t idx = (size_t)i + (size_t)P.nu * ((size_t)j + (size_t)P.nv * k);
  const float r = acc * R.step;
  proj[idx] = accumulate ? proj[idx] + r : r;
}

// Exact transpose of k_fp_ray: scatter y*step*w into the padded accumulator.
__global__ void __launch_bounds__(256) k_fp_ray_transpose(FPParams P, const ViewD *__restrict__ views,
                                                          const float *__restrict__ proj,
                                                          float *__restrict__ acc_pad) {
  const int i = blockIdx.x * 16 + threadIdx.x;
  const int j = blockIdx.y * 16 + threadIdx.y;
  const int k = blockIdx.z;
  if (i >= P.nu || j >= P.nv) return;
  const ViewD vw = views[k];
  const RaySetup R = ray_finish(P, vw, col_setup(P, vw, i), j);
  const float y = proj[(size_t)i + (size_t)P.nu * ((size_t)j + (size_t)P.nv * k)] * R.step;
  if (y == 0.0f) return;
  const unsigned px = P.px, pxy = P.pxy;
  for (int m = 0; m < P.n; ++m) {
    const float fm = (float)m;
    const float sx = clampf(fmaf(fm, R.q[0], R.p[0]), P.cx);
    const float sy = clampf(fmaf(fm, R.q[1], R.p[1]), P.cy);
    const float sz = clampf(fmaf(fm, R.q[2], R.p[2]), P.cz);
    const float flx = floorf(sx), fly = floorf(sy), flz = floorf(sz);
    const float ax = sx - flx, ay = sy - fly, az = sz - flz;
    const unsigned base = (unsigned)flx + px * (unsigned)fly + pxy * (unsigned)flz;
    const float bx = 1.0f - ax, by = 1.0f - ay, bz = 1.0f - az;
    atomicAdd(acc_pad + base, bx * by * bz * y);
    atomicAdd(acc_pad + base + 1, ax * by * bz * y);
    atomicAdd(acc_pad + base + px, bx * ay * bz * y);
    atomicAdd(acc_pad + base + px + 1, ax * ay * bz * y);
    atomicAdd(acc_pad + base + pxy, bx * by * az * y);
    atomicAdd(acc_pad + base + pxy + 1, ax * by * az * y);
    atomicAdd(acc_pad + base + pxy + px, bx * ay * az * y);
    atomicAdd(acc_pad + base + pxy + px + 1, ax * ay * az * y);
  }
}

// ------------------------------------------------------------------ engine 1
__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// Raw buffer loads: 32-bit byte offsets, corner offsets in SGPRs, and zero
// for any offset past the end of the buffer.
template <typename T>
__device__ __forceinline__ float bload(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff);
template <>
__device__ __forceinline__ float bload<float>(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  // the builtin returns the raw 32-bit word
  return __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
}
template <>
__device__ __forceinline__ float bload<unsigned short>(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                       unsigned soff) {
  return bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(r, (int)voff, (int)soff, 0));
}

// Two consecutive elements (byte offset voff+soff, 4- or 8-byte aligned) as
// floats: one dwordx2 load for FP32, one dword load for BF16.
template <typename T>
__device__ __forceinline__ float2 bload2(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff);
template <>
__device__ __forceinline__ float2 bload2<float>(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                unsigned soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0);
  return make_float2(__uint_as_float((unsigned)v[0]), __uint_as_float((unsigned)v[1]));
}
template <>
__device__ __forceinline__ float2 bload2<unsigned short>(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                         unsigned soff) {
  const unsigned w = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0);
  return make_float2(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u));
}

// a = (a.lo, b.lo), b = (a.hi, b.hi), lo / hi: lanes 0-31 / 32-63
__device__ __forceinline__ void swap32(unsigned &a, unsigned &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// The four corner z-lines (00, 10, 01, 11: x + (line & 1), y + (line >> 1)) of
// one (x, y) cell over a window of 64 Z z, Z per lane, kept as loaded (BF16
// pairs stay packed) and unpacked in the combine.  The texture address unit
// takes four lanes per clock whatever their width, so a load instruction costs
// it 16 clocks (measured: 8 and 16 bytes per lane the same), and it binds small
// FP32 windows, whose steps have few vector instructions (80% busy at 128^3).
//   window piece   FP32                                 BF16
//   256 z          16 bytes per lane                    (pieces of 128)
//   192 z          12 bytes per lane                    (128 + 64)
//   128 z          two lines per load, 16 bytes per     4 bytes per lane
//                  lane, one in each half of the lanes;
//                  permlane swaps (fix) then give every
//                  lane the same z of both
//   64 z           4 bytes per lane                     2 bytes per lane
// Two lines per load took 128^3, 180 views, from 0.75 to 0.69 ms; 16 bytes per
// lane instead of two loads of 8, 512^3, 720 views, from 163 to 156.  BF16
// steps have the unpacking on top and are bound by the vector unit: wider or
// shared loads cost them more than they save (512^3, 720 views: 8 or 16 bytes
// per lane 3% slower; four lines per load at 128^3 0.65 -> 0.72 ms).
template <typename T, int Z>
struct Cell {
  static constexpr bool F = sizeof(T) == 4;
  static constexpr int Q = F ? Z / 4 : 0, R = Z - 4 * Q;   // 256-z pieces; the rest
  static constexpr bool TRIPLE = R == 3 && F;
  static constexpr int PAIRS = TRIPLE ? 0 : R / 2, ONE = R & 1 && !TRIPLE ? 1 : 0;
  static constexpr int WORDS = F ? Z : PAIRS + ONE;   // per line
  static constexpr unsigned E = sizeof(T), BP = 256 * E * Q, BO = BP + 128 * E * PAIRS;   // pieces' bytes
  unsigned w[4][WORDS];
  unsigned vh;   // lanes' byte offsets when the halves hold different lines

  __device__ __forceinline__ void setup(int lane, unsigned so_x) {
    vh = 16 * (lane & 31) + (lane & 32 ? so_x : 0);
  }
  // B: byte offset of line 00 at the window's first z
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int lane, unsigned B, unsigned so_x,
                                       unsigned so_y) {
    const unsigned S[4] = {B, B + so_x, B + so_y, B + so_x + so_y};
    if constexpr (PAIRS && F) {   // words 2 and 3 of a load are the other line's, after fix
#pragma unroll
      for (int c = 0; c < 4; c += 2) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(vh + BP), (int)S[c], 0);
        w[c][4 * Q] = v[0]; w[c][4 * Q + 1] = v[1]; w[c + 1][4 * Q] = v[2]; w[c + 1][4 * Q + 1] = v[3];
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(16 * lane + 1024 * q), (int)S[c], 0);
        w[c][4 * q] = v[0]; w[c][4 * q + 1] = v[1]; w[c][4 * q + 2] = v[2]; w[c][4 * q + 3] = v[3];
      }
      if constexpr (TRIPLE) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(r, (int)(12 * lane + BP), (int)S[c], 0);
        w[c][4 * Q] = v[0]; w[c][4 * Q + 1] = v[1]; w[c][4 * Q + 2] = v[2];
      }
      if constexpr (!F) {
#pragma unroll
        for (int p = 0; p < PAIRS; ++p)
          w[c][p] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)(4 * lane + 256 * p), (int)S[c], 0);
      }
      if constexpr (ONE) {
        if constexpr (F) w[c][WORDS - 1] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)(4 * lane + BO), (int)S[c], 0);
        else w[c][WORDS - 1] = (unsigned)__builtin_amdgcn_raw_buffer_load_b16(r, (int)(2 * lane + BO), (int)S[c], 0);
      }
    }
  }
  // once per load: the loaded words into their lines' registers
  __device__ __forceinline__ void fix() {
    if constexpr (PAIRS && F) {
#pragma unroll
      for (int i = 4 * Q; i < 4 * Q + 2; ++i) {
        swap32(w[0][i], w[1][i]);
        swap32(w[2][i], w[3][i]);
      }
    }
  }
  // line c's value number t of the lane (in the order of the pieces)
  __device__ __forceinline__ float at(int c, int t) const {
    if constexpr (F) return __uint_as_float(w[c][t]);
    else if (t == Z - 1 && ONE) return __uint_as_float(w[c][WORDS - 1] << 16);
    else return __uint_as_float(t & 1 ? w[c][t >> 1] & 0xffff0000u : w[c][t >> 1] << 16);
  }
  // the bilinear z-line at weights (ax, ay) into LDS
  __device__ __forceinline__ void combine(float *zl, int lane, float ax, float ay) const {
    float o[Z];
#pragma unroll
    for (int t = 0; t < Z; ++t) {
      const float v00 = at(0, t), v01 = at(2, t);
      const float c0 = fmaf(ax, at(1, t) - v00, v00);
      const float c1 = fmaf(ax, at(3, t) - v01, v01);
      o[t] = fmaf(ay, c1 - c0, c0);
    }
    store(zl, lane, o);
  }
  // a lane's Z values to their places of the z-line in LDS
  static __device__ __forceinline__ void store(float *zl, int lane, const float (&o)[Z]) {
    int k = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q, k += 4)
      *reinterpret_cast<float4 *>(&zl[256 * q + 4 * lane]) = make_float4(o[k], o[k + 1], o[k + 2], o[k + 3]);
    if constexpr (TRIPLE) {
#pragma unroll
      for (int t = 0; t < 3; ++t) zl[256 * Q + 3 * lane + t] = o[k + t];
    }
#pragma unroll
    for (int p = 0; p < PAIRS; ++p, k += 2)
      *reinterpret_cast<float2 *>(&zl[256 * Q + 128 * p + (F ? 4 * (lane & 31) + 2 * (lane >> 5) : 2 * lane)]) =
          make_float2(o[k], o[k + 1]);
    if constexpr (ONE) zl[256 * Q + 128 * PAIRS + lane] = o[k];
  }
};

// Order one wave's LDS writes before its later LDS reads of other lanes'
// data (and the reads before the next writes).  A wave's LDS operations
// complete in issue order, so only the compiler has to be held back.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Voxels z and z + 1 at element e of the z-fastest copy (byte offset of a
// neighbouring line in soff): one 8-byte load; BF16 takes the four voxels from
// the even z on and picks two.
template <typename T>
__device__ __forceinline__ float2 zpair(__amdgpu_buffer_rsrc_t r, unsigned e, unsigned soff);
template <>
__device__ __forceinline__ float2 zpair<float>(__amdgpu_buffer_rsrc_t r, unsigned e, unsigned soff) {
  return bload2<float>(r, e * 4u, soff);
}
template <>
__device__ __forceinline__ float2 zpair<unsigned short>(__amdgpu_buffer_rsrc_t r, unsigned e,
                                                        unsigned soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)((e & ~1u) * 2u), (int)soff, 0);
  const unsigned w = __builtin_amdgcn_alignbit((unsigned)v[1], (unsigned)v[0], (e & 1u) << 4);
  return make_float2(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u));
}

// Elements e and e + 1 (z and z + 1) of k_pack_cells' copy: the voxel and its
// neighbours at x + 1, y + 1 and both.
template <typename T>
__device__ __forceinline__ void cell_pair(__amdgpu_buffer_rsrc_t r, unsigned e, float4 &lo, float4 &hi);
template <>
__device__ __forceinline__ void cell_pair<float>(__amdgpu_buffer_rsrc_t r, unsigned e, float4 &lo, float4 &hi) {
  const auto a = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(e * 16u), 0, 0);
  const auto b = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(e * 16u + 16u), 0, 0);
  lo = make_float4(__uint_as_float(a[0]), __uint_as_float(a[1]), __uint_as_float(a[2]), __uint_as_float(a[3]));
  hi = make_float4(__uint_as_float(b[0]), __uint_as_float(b[1]), __uint_as_float(b[2]), __uint_as_float(b[3]));
}
template <>
__device__ __forceinline__ void cell_pair<unsigned short>(__amdgpu_buffer_rsrc_t r, unsigned e, float4 &lo,
                                                          float4 &hi) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(e * 8u), 0, 0);
  auto low = [](unsigned w) { return __uint_as_float(w << 16); };
  auto high = [](unsigned w) { return __uint_as_float(w & 0xffff0000u); };
  lo = make_float4(low(v[0]), high(v[0]), low(v[1]), high(v[1]));
  hi = make_float4(low(v[2]), high(v[2]), low(v[3]), high(v[3]));
}

// The sum over its n samples of each lane's ray R (lanes with mine unset: 0),
// for 64 adjacent rows of one detector column whose x/y positions are their
// own (rays that leave through the volume's top or bottom).  One ray per lane
// would scatter every load over up to 64 (x, y) lines, since neighbouring rows
// end at different depths and so step at different lengths; instead a wave
// takes 8 consecutive samples of 8 adjacent rays at a time and leaves the
// values in LDS; after the 64 rays' 8 samples each lane adds its own ray's, in
// order.  Sample positions and the order of the lerps and sums are the per-ray
// engine's (the same bits).  The texture address unit binds it: it takes four
// lanes per clock when they hit one line, else one lane per line, so lanes run
// along a ray (steps of a clipped ray stay within a voxel or two; 28 cache
// accesses per load) and not across rays (40).  CELLS: the copy of k_pack_cells,
// whose elements hold the four (x, y) corners: half the loads.  256 x 256 x 160
// voxels, 90 views of 512 x 384, 30% of the rays clipped: 8.4 ms for the whole
// projection from the plain copy, 5.6 from the packed one (k_fp_clip), 40.8 with
// one ray per lane.
//   lds: 64 x 6 floats of ray parameters, 64 x FPG_ROW floats of samples
constexpr int FPG_ROW = 12;   // 8 samples, 16-byte aligned rows off the same banks
constexpr int FPG_LDS = 64 * 6 + 64 * FPG_ROW;
template <typename T, bool CELLS>
__device__ __forceinline__ float fp_gather(const FPParams &P, const RaySetup &R, const bool mine,
                                           const T *__restrict__ vt, unsigned vt_bytes, int lane,
                                           float *lds) {
  const unsigned esz = sizeof(T);
  const unsigned so_x = P.pz * esz, so_y = P.pzx * esz, so_xy = (P.pzx + P.pz) * esz;
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void *)vt, (short)0, (int)vt_bytes, 0x00020000);
  float4 *par4 = reinterpret_cast<float4 *>(lds);
  float2 *par2 = reinterpret_cast<float2 *>(lds + 64 * 4);
  float *smp = lds + 64 * 6;
  par4[lane] = make_float4(R.p[0], R.q[0], R.p[1], R.q[1]);
  par2[lane] = make_float2(R.p[2], R.q[2]);
  const unsigned long long rays = __builtin_amdgcn_ballot_w64(mine);
  wave_lds_sync();
  const int lr = lane >> 3, ls = lane & 7;
  float acc = 0.0f;
  for (int mb = 0; mb < P.n; mb += 8) {
    const float fm = (float)(mb + ls);
#pragma unroll 4
    for (int o = 0; o < 8; ++o) {   // rays 8 o .. 8 o + 7
      if (!((rays >> (8 * o)) & 0xffull)) continue;
      const float4 a = par4[8 * o + lr];
      const float2 b = par2[8 * o + lr];
      // clamped coordinates are finite and in [0, n + 1]: med3 equals
      // fminf(fmaxf()), truncation equals floor
      const float sx = __builtin_amdgcn_fmed3f(fmaf(fm, a.y, a.x), 0.0f, P.cx);
      const float sy = __builtin_amdgcn_fmed3f(fmaf(fm, a.w, a.z), 0.0f, P.cy);
      const float sz = __builtin_amdgcn_fmed3f(fmaf(fm, b.y, b.x), 0.0f, P.cz);
      const float ax = __builtin_amdgcn_fractf(sx), ay = __builtin_amdgcn_fractf(sy);
      const float az = __builtin_amdgcn_fractf(sz);
      const unsigned e = ((unsigned)(int)sy * P.px + (unsigned)(int)sx) * P.pz + (unsigned)(int)sz;
      float c00, c10, c01, c11;   // x-lerped (y, z) corners
      if constexpr (CELLS) {
        float4 lo, hi;   // (x, y) corners at z and z + 1
        cell_pair<T>(rsrc, e, lo, hi);
        c00 = fmaf(ax, lo.y - lo.x, lo.x);
        c10 = fmaf(ax, lo.w - lo.z, lo.z);
        c01 = fmaf(ax, hi.y - hi.x, hi.x);
        c11 = fmaf(ax, hi.w - hi.z, hi.z);
      } else {
        const float2 v00 = zpair<T>(rsrc, e, 0), v10 = zpair<T>(rsrc, e, so_x);
        const float2 v01 = zpair<T>(rsrc, e, so_y), v11 = zpair<T>(rsrc, e, so_xy);
        c00 = fmaf(ax, v10.x - v00.x, v00.x);
        c10 = fmaf(ax, v11.x - v01.x, v01.x);
        c01 = fmaf(ax, v10.y - v00.y, v00.y);
        c11 = fmaf(ax, v11.y - v01.y, v01.y);
      }
      const float c0 = fmaf(ay, c10 - c00, c00);
      const float c1 = fmaf(ay, c11 - c01, c01);
      smp[(8 * o + lr) * FPG_ROW + ls] = fmaf(az, c1 - c0, c0);
    }
    wave_lds_sync();
    if (mine) {
      const int cnt = min(8, P.n - mb);
      const float4 u = *reinterpret_cast<const float4 *>(&smp[lane * FPG_ROW]);
      const float4 v = *reinterpret_cast<const float4 *>(&smp[lane * FPG_ROW + 4]);
      const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
      if (cnt == 8) {
#pragma unroll
        for (int t = 0; t < 8; ++t) acc += x[t];
      } else {
#pragma unroll
        for (int t = 0; t < 7; ++t)
          if (t < cnt) acc += x[t];
      }
    }
    wave_lds_sync();
  }
  return acc;
}

// Block order of the column engine.  xcd_remap gives every XCD a contiguous
// range of W.  Within it, the blocks of P.vg adjacent views of one (column,
// row group) come one after another, so they run at the same time on one XCD
// and their rays, close together in the volume, share that XCD's L2; views
// past the last whole group of P.vg follow view by view.  vg = 1: view by
// view (column fastest).
__device__ __forceinline__ void col_block(const FPParams &P, unsigned W, unsigned ngroups,
                                          unsigned nblocks, int &i, int &grp, int &k) {
  const unsigned per_view = (unsigned)P.nu * ngroups;
  const unsigned nviews = nblocks / per_view;
  const unsigned vg = P.vg;
  const unsigned whole = (nviews / vg) * vg * per_view;
  unsigned vin = 0, rest = W;
  if (W < whole) {
    vin = W % vg;
    rest = W / vg;
  }
  i = (int)(rest % (unsigned)P.nu);
  const unsigned r2 = rest / (unsigned)P.nu;
  grp = (int)(r2 % ngroups);
  k = W < whole ? (int)((r2 / ngroups) * vg + vin) : (int)(r2 / ngroups);
}

// One 64-lane workgroup per (detector column, row group, view).  RPL rays per
// lane: rows j = row0 + r*64 + lane.
//   SSTEP = false, ZP = 1: per-step setup on the vector unit, one z per lane
//     and load (FP32 storage: measured fastest there).
//   SSTEP = true, ZP = 2: integer step setup in scalar registers, no per-ray
//     z clamp (shared rays stay inside the volume's z), two consecutive z per
//     lane and load (BF16 storage: one dword per lane instead of two 16-bit
//     loads, 1.5x faster there).
//   ZC > 0 (with SSTEP, ZP = 2): the z window of the whole ray (all its steps,
//     all shared rows) is fixed once; when it spans at most 64 ZC z, the four
//     corner z-lines of the current (x, y) cell stay in registers while the
//     ray stays in the cell (Cell) and all four are reloaded for the next
//     step's cell right after this step's combine.  Every load fetches the
//     whole window; z past the part a step needs are never read.
// All produce the same bits as the per-ray engine.
template <typename T, int RPL, bool SSTEP, int ZP, int ZC, int D>
__device__ __forceinline__ void fp_col_body(const FPParams &P, const ViewD *__restrict__ views,
                                            const T *__restrict__ vt, float *__restrict__ proj,
                                            int accumulate, unsigned ngroups, unsigned nblocks,
                                            unsigned vt_bytes) {
  extern __shared__ __align__(16) float zl[];  // one interpolated z-line (whole 128-wide chunks)
  int i, grp, k;
  col_block(P, xcd_remap(blockIdx.x, nblocks), ngroups, nblocks, i, grp, k);
  const int lane = threadIdx.x;
  const int row0 = grp * 64 * RPL;
  float pz[RPL], qz[RPL], acc[RPL];
  unsigned shared_mask = 0, valid_mask = 0;
  int gjmin, gjmax;
  float px0, qx, py0, qy;      // the column's x/y trace
  float pzl, qzl, pzh, qzh;    // z of the first and last shared rays
  float *stp = zl + P.lds_stp + lane;   // step lengths, parked in LDS until the end
  {
    const ViewD vw = views[k];
    const ColSetup C = col_setup(P, vw, i);
    const double a1c = fmax(C.lo, 0.0);
    const double a2c = fmin(C.hi, 1.0);
    const bool col_ok = (a2c - a1c) >= 0.0;   // h >= 0 keeps tz monotone in the row
    // the shared (a1, a2): x/y once per column, z per row
    const double span = a2c - a1c, h = span / P.n;
    ray_xy(P, C, a1c, h, px0, qx, py0, qy);
    int jmin = 0x7fffffff, jmax = -1;
#pragma unroll
    for (int r = 0; r < RPL; ++r) {
      const int j = row0 + r * 64 + lane;
      acc[r] = 0.0f;
      const double d2 = row_height(P, vw, j);
      const double t = fabs(P.lz * 0.5 / d2);   // the z slab is [-t, t]
      ray_z(P, C, d2, a1c, span, h, pz[r], qz[r], stp[64 * r]);
      if (j < P.nv) {
        valid_mask |= 1u << r;
        if (col_ok && fmax(fmax(C.lo, -t), 0.0) == a1c && fmin(fmin(C.hi, t), 1.0) == a2c) {
          shared_mask |= 1u << r;
          jmin = min(jmin, j);
          jmax = max(jmax, j);
        }
      }
      __builtin_amdgcn_sched_barrier(0);   // one ray's FP64 temporaries at a time
    }
    gjmin = wave_min_i(jmin);
    gjmax = wave_max_i(jmax);
  }
  // from their lanes (0 where there is no shared ray; not used then)
  auto of_row = [&](const float(&v)[RPL], int j) __attribute__((always_inline)) {
    const int slot = __builtin_amdgcn_readfirstlane((j - row0) >> 6);
    float x = 0.0f;
#pragma unroll
    for (int r = 0; r < RPL; ++r)
      if (slot == r) x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[r]), (j - row0) & 63));
    return x;
  };
  pzl = of_row(pz, gjmin);
  qzl = of_row(qz, gjmin);
  pzh = of_row(pz, gjmax);
  qzh = of_row(qz, gjmax);
  // Shared rays leave through the x and y faces, so their z texel coordinates
  // stay in [0.5, nz + 0.5] up to rounding (under 1e-3: nz <= 4096): the
  // per-ray clamp to [0, nz + 1] is the identity and is dropped (SSTEP).

  if (SSTEP && gjmax >= 0) {
#pragma unroll
    for (int r = 0; r < RPL; ++r)
      if (!(shared_mask & (1u << r))) {
        pz[r] = pzl;
        qz[r] = qzl;
      }
    const unsigned PZ = P.pz;
    const unsigned esz = sizeof(T);
    const unsigned so_x = PZ * esz, so_y = P.pzx * esz, so_xy = (P.pzx + PZ) * esz;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void *)vt, (short)0, (int)vt_bytes, 0x00020000);
    const unsigned lane_off = (unsigned)lane * esz;
    bool done = false;
    if constexpr (ZC > 0) {
      // The window: per step the rays read z in [zlo(m), zhi(m)], both linear
      // in m through the same fmaf as below (so monotone), hence extreme at
      // the first or last step.
      const float ml = (float)(P.n - 1);
      const int zlo_min = __builtin_amdgcn_readfirstlane((int)fminf(pzl, fmaf(ml, qzl, pzl)));
      const int zhi_max = __builtin_amdgcn_readfirstlane((int)fmaxf(pzh, fmaf(ml, qzh, pzh))) + 1;
      const int zb0 = zlo_min & ~3;   // pieces aligned to their width
      // (cell coordinates are packed as two 16-bit halves below)
      if (zhi_max - zb0 < 64 * ZC && P.cx < 65535.0f && P.cy < 65535.0f) {
        done = true;
        const unsigned zoff = (unsigned)zb0 * esz;
        // byte offset of cell (c & 0xffff, c >> 16)'s line 00 at the window
        auto cell_base = [&](unsigned c) __attribute__((always_inline)) {
          return ((c >> 16) * P.px + (c & 0xffffu)) * PZ * esz + zoff;
        };
        // x/y position of step m, the same for the whole wave
        auto step_x = [&](float fm) { return __builtin_amdgcn_fmed3f(fmaf(fm, qx, px0), 0.0f, P.cx); };
        auto step_y = [&](float fm) { return __builtin_amdgcn_fmed3f(fmaf(fm, qy, py0), 0.0f, P.cy); };
        auto step_cell = [&](float fm) { return (unsigned)step_x(fm) | ((unsigned)step_y(fm) << 16); };
        if constexpr (D > 1) {
          // Few waves: the step's own latencies (lines from L2, the z-line
          // through LDS) are not hidden by other waves but by the steps
          // around it.  The lines of D steps are in flight, each step's reloaded
          // for D steps on once its combine has used them, and a step's reads
          // of its z-line (two buffers) return during the next step's combine.
          Cell<T, ZC> S[D];
          float pa[RPL], pb[RPL], paz[RPL];   // the last step's reads
#pragma unroll
          for (int r = 0; r < RPL; ++r) pa[r] = pb[r] = paz[r] = 0.0f;   // adds 0 before step 0
          const int last = P.n - 1;
          const unsigned c0 = step_cell((float)min(lane, last));
#pragma unroll
          for (int d = 0; d < D; ++d) {
            S[d].setup(lane, so_x);
            S[d].load(rsrc, lane, cell_base((unsigned)__builtin_amdgcn_readlane((int)c0, d)), so_x, so_y);
          }
          auto finish = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < RPL; ++r) acc[r] += fmaf(paz[r], pb[r] - pa[r], pa[r]);
          };
          for (int mb = 0; mb < P.n; mb += 64) {
            const float fml = (float)(mb + lane);
            const int axl = __float_as_int(__builtin_amdgcn_fractf(step_x(fml)));
            const int ayl = __float_as_int(__builtin_amdgcn_fractf(step_y(fml)));
            const int cn = (int)step_cell((float)min(mb + lane + D, last));   // D steps on
            const int cnt = __builtin_amdgcn_readfirstlane(min(64, P.n - mb));
            for (int l = 0; l < cnt; l += D) {
#pragma unroll
              for (int d = 0; d < D; ++d) {
                if (l + d >= cnt) break;
                float *z = zl + (d & 1) * 64 * ZC;
                S[d].fix();
                S[d].combine(z, lane, __int_as_float(__builtin_amdgcn_readlane(axl, l + d)),
                             __int_as_float(__builtin_amdgcn_readlane(ayl, l + d)));
                S[d].load(rsrc, lane, cell_base((unsigned)__builtin_amdgcn_readlane(cn, l + d)), so_x, so_y);
                finish();
                wave_lds_sync();
                const float fm = (float)(mb + l + d);
                const float *zr = z - zb0;
#pragma unroll
                for (int r = 0; r < RPL; ++r) {
                  const float tz = fmaf(fm, qz[r], pz[r]);
                  const int iz = (int)tz;
                  paz[r] = __builtin_amdgcn_fractf(tz);
                  pa[r] = zr[iz];
                  pb[r] = zr[iz + 1];
                }
                wave_lds_sync();
              }
            }
          }
          finish();
        } else {
          Cell<T, ZC> L;
          L.setup(lane, so_x);
          const float *zb = zl - zb0;
          // every ray's z-lerp from the combined z-line
          auto rays = [&](const float fm) __attribute__((always_inline)) {
#pragma unroll
              for (int r = 0; r < RPL; ++r) {
                const float tz = fmaf(fm, qz[r], pz[r]);  // in [0, nz+1]: as above
                const int iz = (int)tz;
                const float az = __builtin_amdgcn_fractf(tz);
                const float a = zb[iz], b = zb[iz + 1];
                acc[r] += fmaf(az, b - a, a);
              }
              wave_lds_sync();
          };
          // The x/y part of a step, the same for the whole wave, is evaluated for
          // 64 steps at once, step mb + lane in each lane (the same expressions
          // as per step, so the same values), and each step reads its cell and
          // weights back into scalar registers.  The lines of the next step's
          // cell, when it changes, are all four reloaded straight into their
          // registers once this step's combine has used them, so they arrive
          // while this step's rays run.  Keeping the lines that the two cells
          // share saves half the bytes, but the register moves wait on the loads:
          // 13.1 against 12.6 ms (FP32 copies, 512^3, 48 views).
          unsigned cur = (unsigned)__builtin_amdgcn_readfirstlane((int)step_cell(0.0f));
          L.load(rsrc, lane, cell_base(cur), so_x, so_y);
          bool fresh = true;   // loaded and not yet fixed
          for (int mb = 0; mb < P.n; mb += 64) {
            const float fml = (float)(mb + lane);
            const int axl = __float_as_int(__builtin_amdgcn_fractf(step_x(fml)));
            const int ayl = __float_as_int(__builtin_amdgcn_fractf(step_y(fml)));
            const int cn = (int)step_cell((float)(mb + lane + 1));   // the next step's
            const int cnt = __builtin_amdgcn_readfirstlane(min(64, P.n - mb));
            for (int l = 0; l < cnt; ++l) {
              const float ax = __int_as_float(__builtin_amdgcn_readlane(axl, l));
              const float ay = __int_as_float(__builtin_amdgcn_readlane(ayl, l));
              if (fresh) L.fix();
              L.combine(zl, lane, ax, ay);
              wave_lds_sync();
              const unsigned nxt = (unsigned)__builtin_amdgcn_readlane(cn, l);
              fresh = mb + l + 1 < P.n && nxt != cur;
              if (fresh) {
                L.load(rsrc, lane, cell_base(nxt), so_x, so_y);
                cur = nxt;
              }
              rays((float)(mb + l));
            }
          }
        }
      }
    }
    for (int m = 0; !done && m < P.n; ++m) {
      // Uniform per-step values: the float part on the VALU (same
      // expressions as the per-ray loop), the integer part moved to scalar
      // registers so the addressing below is scalar.
      const float fm = (float)m;
      const float sx = __builtin_amdgcn_fmed3f(fmaf(fm, qx, px0), 0.0f, P.cx);
      const float sy = __builtin_amdgcn_fmed3f(fmaf(fm, qy, py0), 0.0f, P.cy);
      const float ax = __builtin_amdgcn_fractf(sx), ay = __builtin_amdgcn_fractf(sy);
      const int ix = __builtin_amdgcn_readfirstlane((int)sx);
      const int iy = __builtin_amdgcn_readfirstlane((int)sy);
      const int zlo = __builtin_amdgcn_readfirstlane((int)fmaf(fm, qzl, pzl));
      const int zhi = __builtin_amdgcn_readfirstlane((int)fmaf(fm, qzh, pzh)) + 1;
      // z-line chunks: corner bases in SGPRs, lane offsets in one VGPR.
      // Offsets past the column read the next column or the allocation's
      // slack; those LDS slots lie beyond zhi and are never read.
      int zb0;
      if constexpr (ZP == 1) {
        zb0 = zlo;
        const int nch = (zhi - zlo + 64) >> 6;
        const unsigned B = (((unsigned)iy * P.px + (unsigned)ix) * PZ + (unsigned)zlo) * esz;
        for (int c = 0; c < nch; ++c) {
          const unsigned voff = lane_off + (unsigned)(64 * c) * esz;
          const float v00 = bload<T>(rsrc, voff, B), v10 = bload<T>(rsrc, voff, B + so_x);
          const float v01 = bload<T>(rsrc, voff, B + so_y), v11 = bload<T>(rsrc, voff, B + so_xy);
          const float c0 = fmaf(ax, v10 - v00, v00);
          const float c1 = fmaf(ax, v11 - v01, v01);
          zl[lane + 64 * c] = fmaf(ay, c1 - c0, c0);
        }
      } else {
        // two consecutive z per lane and load (128 z per instruction); the
        // line starts at an even z so the pair loads are aligned
        zb0 = zlo & ~1;
        const int nch = (zhi - zb0 + 128) >> 7;
        const unsigned B = (((unsigned)iy * P.px + (unsigned)ix) * PZ + (unsigned)zb0) * esz;
        for (int c = 0; c < nch; ++c) {
          const unsigned voff = 2 * lane_off + (unsigned)(128 * c) * esz;
          const float2 v00 = bload2<T>(rsrc, voff, B), v10 = bload2<T>(rsrc, voff, B + so_x);
          const float2 v01 = bload2<T>(rsrc, voff, B + so_y), v11 = bload2<T>(rsrc, voff, B + so_xy);
          float2 o;
          {
            const float c0 = fmaf(ax, v10.x - v00.x, v00.x);
            const float c1 = fmaf(ax, v11.x - v01.x, v01.x);
            o.x = fmaf(ay, c1 - c0, c0);
          }
          {
            const float c0 = fmaf(ax, v10.y - v00.y, v00.y);
            const float c1 = fmaf(ax, v11.y - v01.y, v01.y);
            o.y = fmaf(ay, c1 - c0, c0);
          }
          *reinterpret_cast<float2 *>(&zl[2 * lane + 128 * c]) = o;
        }
      }
      wave_lds_sync();
      const float *zb = zl - zb0;
#pragma unroll
      for (int r = 0; r < RPL; ++r) {
        const float tz = fmaf(fm, qz[r], pz[r]);  // in [0, nz+1]: as above
        const int iz = (int)tz;
        const float az = __builtin_amdgcn_fractf(tz);
        const float a = zb[iz], b = zb[iz + 1];
        acc[r] += fmaf(az, b - a, a);
      }
      wave_lds_sync();
    }
  } else if (!SSTEP && gjmax >= 0) {
    // rays outside the shared set read harmless in-range LDS entries
#pragma unroll
    for (int r = 0; r < RPL; ++r)
      if (!(shared_mask & (1u << r))) {
        pz[r] = pzl;
        qz[r] = qzl;
      }
    // Coordinates here are finite and the clamps keep them in [0, n+1], so
    // med3 equals fminf(fmaxf()), truncation equals floor and fract(t)
    // equals t - floor(t): same values as the per-ray loop.
    const unsigned PZ = P.pz;
    const unsigned esz = sizeof(T);
    const unsigned so_x = PZ * esz, so_y = P.pzx * esz, so_xy = (P.pzx + PZ) * esz;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void *)vt, (short)0, (int)vt_bytes, 0x00020000);
    for (int m = 0; m < P.n; ++m) {
      const float fm = (float)m;
      const float sx = __builtin_amdgcn_fmed3f(fmaf(fm, qx, px0), 0.0f, P.cx);
      const float sy = __builtin_amdgcn_fmed3f(fmaf(fm, qy, py0), 0.0f, P.cy);
      const float ax = __builtin_amdgcn_fractf(sx), ay = __builtin_amdgcn_fractf(sy);
      const int zlo = (int)__builtin_amdgcn_fmed3f(fmaf(fm, qzl, pzl), 0.0f, P.cz);
      const int zhi = (int)__builtin_amdgcn_fmed3f(fmaf(fm, qzh, pzh), 0.0f, P.cz) + 1;
      const int nch = (zhi - zlo + 64) >> 6;
      const unsigned base = ((unsigned)(int)sy * P.px + (unsigned)(int)sx) * PZ + (unsigned)zlo;
      for (int c = 0; c < nch; ++c) {
        const unsigned zi = min(base + (unsigned)(lane + 64 * c), base - (unsigned)zlo + PZ - 1);
        const unsigned voff = zi * esz;
        const float v00 = bload<T>(rsrc, voff, 0), v10 = bload<T>(rsrc, voff, so_x);
        const float v01 = bload<T>(rsrc, voff, so_y), v11 = bload<T>(rsrc, voff, so_xy);
        const float c0 = fmaf(ax, v10 - v00, v00);
        const float c1 = fmaf(ax, v11 - v01, v01);
        zl[lane + 64 * c] = fmaf(ay, c1 - c0, c0);
      }
      wave_lds_sync();
      const float *zb = zl - zlo;
#pragma unroll
      for (int r = 0; r < RPL; ++r) {
        const float tz = __builtin_amdgcn_fmed3f(fmaf(fm, qz[r], pz[r]), 0.0f, P.cz);
        const int iz = (int)tz;
        const float az = __builtin_amdgcn_fractf(tz);
        const float a = zb[iz], b = zb[iz + 1];
        acc[r] += fmaf(az, b - a, a);
      }
      wave_lds_sync();
    }
  }

  // the results take the step lengths' places in LDS
#pragma unroll
  for (int r = 0; r < RPL; ++r) stp[64 * r] *= acc[r];

  // Rays clipped by the z faces (or a column that misses the box) have x/y
  // positions of their own: the 64 rows of one register slot together.
  // The FP64 column setup is evaluated again (through an opaque copy of the
  // column index), which keeps its 20 registers out of the loops above.
  const unsigned todo = valid_mask & ~shared_mask;
  if (!P.split && __builtin_amdgcn_ballot_w64(todo != 0)) {
    int iw = __builtin_amdgcn_readfirstlane(i);
    asm volatile("" : "+s"(iw));
    const ViewD vw = views[k];
    const ColSetup C = col_setup(P, vw, iw);
#pragma nounroll
    for (int r = 0; r < RPL; ++r) {
      const bool mine = (todo >> r) & 1u;
      if (__builtin_amdgcn_ballot_w64(mine) == 0) continue;
      const RaySetup R = ray_finish(P, vw, C, row0 + r * 64 + lane);
      const float a = fp_gather<T, false>(P, R, mine, vt, vt_bytes, lane, zl);
      if (mine) stp[64 * r] = a * R.step;
    }
  }

#pragma unroll
  for (int r = 0; r < RPL; ++r) {
    if (!((P.split ? shared_mask : valid_mask) & (1u << r))) continue;
    const int j = row0 + r * 64 + lane;
    const size_t idx = (size_t)i + (size_t)P.nu * ((size_t)j + (size_t)P.nv * k);
    const float v = stp[64 * r];
    proj[idx] = accumulate ? proj[idx] + v : v;
  }
}

template <typename T, int RPL, bool SSTEP, int ZP>
__global__ void __launch_bounds__(64) k_fp_col(FPParams P, const ViewD *__restrict__ views,
                                               const T *__restrict__ vt, float *__restrict__ proj,
                                               int accumulate, unsigned ngroups, unsigned nblocks,
                                               unsigned vt_bytes) {
  fp_col_body<T, RPL, SSTEP, ZP, 0, 1>(P, views, vt, proj, accumulate, ngroups, nblocks, vt_bytes);
}

// The cached variant, held to five waves per SIMD, four from 8 rows per lane on
// (more rows spill at five).  512^3, 48 views, 6 rows per lane: four / five /
// six / seven waves 12.8 / 12.8 / 14.1 / 15.2 ms (FP32 copies), 11.0 / 11.1 /
// 11.2 / 12.3 (BF16); 291^3, 32 views, 8 rows: 1.61 / 1.70 / 2.03 / 2.19 and
// 1.49 / 1.57 / 1.63 / 1.82.
constexpr int colc_waves(int rpl, int d) { return d > 1 ? 2 : rpl >= 8 ? 4 : 5; }
template <typename T, int RPL, int ZC, int D>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(colc_waves(RPL, D))))
k_fp_colc(FPParams P, const ViewD *__restrict__ views, const T *__restrict__ vt,
          float *__restrict__ proj, int accumulate, unsigned ngroups, unsigned nblocks,
          unsigned vt_bytes) {
  fp_col_body<T, RPL, true, 2, ZC, D>(P, views, vt, proj, accumulate, ngroups, nblocks, vt_bytes);
}

// The rays that the column kernels with P.split leave out (those not shared),
// from the packed copy: one wave per 64 rows of a detector column.  Used where
// many rays are clipped (clip_cells).
template <typename T>
__global__ void __launch_bounds__(64) k_fp_clip(FPParams P, const ViewD *__restrict__ views,
                                                const T *__restrict__ cells, float *__restrict__ proj,
                                                int accumulate, unsigned nslots, unsigned nblocks,
                                                unsigned cell_bytes) {
  __shared__ __align__(16) float lds[FPG_LDS];
  int i, slot, k;
  col_block(P, xcd_remap(blockIdx.x, nblocks), nslots, nblocks, i, slot, k);
  const int lane = threadIdx.x, j = slot * 64 + lane;
  const ViewD vw = views[k];
  const ColSetup C = col_setup(P, vw, i);
  const double a1c = fmax(C.lo, 0.0), a2c = fmin(C.hi, 1.0);
  const double t = fabs(P.lz * 0.5 / row_height(P, vw, j));
  const bool shared = a2c - a1c >= 0.0 && fmax(fmax(C.lo, -t), 0.0) == a1c && fmin(fmin(C.hi, t), 1.0) == a2c;
  const bool mine = j < P.nv && !shared;
  if (__builtin_amdgcn_ballot_w64(mine) == 0) return;
  const RaySetup R = ray_finish(P, vw, C, j);
  const float a = fp_gather<T, true>(P, R, mine, cells, cell_bytes, lane, lds);
  if (mine) {
    const size_t idx = (size_t)i + (size_t)P.nu * ((size_t)j + (size_t)P.nv * k);
    const float v = a * R.step;
    proj[idx] = accumulate ? proj[idx] + v : v;
  }
}

// ------------------------------------------------------------ layouts
// Element conversion of the padded copies: identity, or FP32 -> BF16 when the
// context keeps its working copies in BF16.
template <typename TO, typename TI>
__device__ __forceinline__ TO to_storage(TI v) {
  return v;
}
template <>
__device__ __forceinline__ unsigned short to_storage<unsigned short, float>(float v) {
  return f32_to_bf16(v);
}

// Copy a volume into the x-fastest zero-bordered layout.
template <typename TI, typename T>
__global__ void __launch_bounds__(256) k_pad_volume(const TI *__restrict__ vol, T *__restrict__ out,
                                                    int nx, int ny, int nz, unsigned px,
                                                    unsigned py, unsigned pz) {
  const size_t total = (size_t)px * py * pz;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total;
       t += (size_t)gridDim.x * blockDim.x) {
    const unsigned a = (unsigned)(t % px);
    const unsigned b = (unsigned)((t / px) % py);
    const unsigned c = (unsigned)(t / ((size_t)px * py));
    const int x = (int)a - 1, y = (int)b - 1, z = (int)c - 1;
    T v = T(0);
    if (x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz)
      v = to_storage<T>(vol[(size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * z)]);
    out[t] = v;
  }
}

// Transposing copy into the z-fastest zero-bordered layout
// out[z' + pz*(x' + px*y')] = vol[x'-1, y'-1, z'-1] (0 outside).
// 32x32 (x', z') tiles through LDS so both the reads (along x) and the writes
// (along z) are coalesced.  grid = (ceil(pz/32), ceil(px/32), py), block 32x8.
template <typename TI, typename T>
__global__ void __launch_bounds__(256) k_pad_transpose(const TI *__restrict__ vol, T *__restrict__ out,
                                                       int nx, int ny, int nz, unsigned px,
                                                       unsigned pz) {
  __shared__ T tile[32][33];
  const int z0 = blockIdx.x * 32, x0 = blockIdx.y * 32, yp = blockIdx.z;
  const int y = yp - 1;
  const int tx = threadIdx.x, ty = threadIdx.y;
  // read: rows of x for 32 z
  for (int r = ty; r < 32; r += 8) {
    const int zp = z0 + r, xp = x0 + tx;
    const int x = xp - 1, z = zp - 1;
    T v = T(0);
    if (x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz)
      v = to_storage<T>(vol[(size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * z)]);
    tile[r][tx] = v;
  }
  __syncthreads();
  // write: columns of z for 32 x
  for (int r = ty; r < 32; r += 8) {
    const int xp = x0 + r, zp = z0 + tx;
    if (xp < (int)px && zp < (int)pz)
      out[(size_t)zp + (size_t)pz * ((size_t)xp + (size_t)px * yp)] = tile[tx][r];
  }
}

// Packed copy for k_fp_clip: element e of the z-fastest copy (px columns of pz
// per y) with its neighbours at x + 1, y + 1 and both, for x <= px - 2, y <= py
// - 2 (the rest is never read).  Four z per thread and 16-byte loads.
template <typename T>
__global__ void __launch_bounds__(256) k_pack_cells(const T *__restrict__ vt, T *__restrict__ out, unsigned pz,
                                                    unsigned px, unsigned py) {
  const unsigned n4 = pz / 4 * px * (py - 1);   // pz is a multiple of 16
  const size_t pzx = (size_t)pz * px;
  struct __align__(4 * sizeof(T)) V4 {
    T v[4];
  };
  for (unsigned t = blockIdx.x * 256 + threadIdx.x; t < n4; t += gridDim.x * 256) {
    const size_t e = (size_t)t * 4;
    if (t / (pz / 4) % px == px - 1) continue;
    const V4 a = *reinterpret_cast<const V4 *>(vt + e), b = *reinterpret_cast<const V4 *>(vt + e + pz);
    const V4 c = *reinterpret_cast<const V4 *>(vt + e + pzx), d = *reinterpret_cast<const V4 *>(vt + e + pzx + pz);
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<V4 *>(out + 4 * (e + i)) = V4{{a.v[i], b.v[i], c.v[i], d.v[i]}};
  }
}

// vol = (accumulate ? vol : 0) + interior(acc_pad)
__global__ void __launch_bounds__(256) k_unpad_add(const float *__restrict__ acc_pad,
                                                   float *__restrict__ vol, int nx, int ny, int nz,
                                                   unsigned px, unsigned pxy, int accumulate) {
  const size_t total = (size_t)nx * ny * nz;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total;
       t += (size_t)gridDim.x * blockDim.x) {
    const unsigned x = (unsigned)(t % nx);
    const unsigned y = (unsigned)((t / nx) % ny);
    const unsigned z = (unsigned)(t / ((size_t)nx * ny));
    const float v = acc_pad[(x + 1) + px * (y + 1) + (size_t)pxy * (z + 1)];
    vol[t] = accumulate ? vol[t] + v : v;
  }
}

__global__ void k_zero(size_t n, float *x) {
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n;
       t += (size_t)gridDim.x * blockDim.x)
    x[t] = 0.0f;
}

inline dim3 stride_grid(size_t n) {
  size_t b = (n + 255) / 256;
  if (b > 262144) b = 262144;
  if (b == 0) b = 1;
  return dim3((unsigned)b);
}

int make_params(cbct_ctx ctx, const cbct_geom *g, float spp, FPParams &P) {
  const float fn = spp * (float)g->nx;
  if (!(fn >= 1.0f) || fn > 1e6f)
    return cbct_fail(ctx, CBCT_ERR_ARG, "Error: conebeam_forwards_projection: samples per ray %g out of range", (double)fn);
  P.nu = g->nu;
  P.nv = g->nv;
  P.n = (int)fn;
  P.nx = g->nx;
  P.ny = g->ny;
  P.nz = g->nz;
  const size_t px = padded_dim(g->nx), py = padded_dim(g->ny), pz = padded_dim(g->nz);
  const size_t pzz = fp_zpadded(g->nz);
  if (px * py * pzz >= (1ull << 32) - 1)
    return cbct_fail(ctx, CBCT_ERR_UNSUPPORTED, "Error: conebeam_forwards_projection: volume too large for 32-bit indexing");
  (void)pz;
  P.px = (unsigned)px;
  P.pxy = (unsigned)(px * py);
  P.pz = (unsigned)pzz;
  P.pzx = (unsigned)(pzz * px);
  P.lx = g->lx;
  P.ly = g->ly;
  P.lz = g->lz;
  P.fu = g->fov_u;
  P.fv = g->fov_v;
  P.sad = g->sad;
  P.sdd = g->sdd;
  P.cx = (float)(g->nx + 1);
  P.cy = (float)(g->ny + 1);
  P.cz = (float)(g->nz + 1);
  P.vg = (unsigned)ctx->fp_view_group;
  P.lds_stp = 0;
  P.split = 0;
  return CBCT_OK;
}

template <typename T, int RPL, bool SSTEP, int ZP, int ZC, int D = 1>
void launch_col(const FPParams &P, hipStream_t s, const ViewD *views, const T *vt, float *proj,
                int acc, int nviews, unsigned vt_bytes) {
  const unsigned ngroups = (unsigned)((P.nv + 64 * RPL - 1) / (64 * RPL));
  // one z-line; the cached variants write their whole window
  const size_t zline = ((P.pz + 127) / 128) * 128;
  // and fp_gather's buffers take the same place afterwards
  const size_t line = std::max({zline, (size_t)64 * ZC, (size_t)FPG_LDS});
  FPParams Q = P;
  Q.lds_stp = (unsigned)line;
  const size_t lds = (line + 64 * RPL) * sizeof(float);
  // a launch covers at most 2^32 - 1 work-items: larger calls go out as
  // several launches over consecutive views (views are independent)
  const size_t per_view = (size_t)P.nu * ngroups;
  const int max_views = (int)std::max<size_t>(1, std::min<size_t>(nviews, ((1ull << 32) - 1) / 64 / per_view));
  for (int v0 = 0; v0 < nviews; v0 += max_views) {
    const int nvc = std::min(max_views, nviews - v0);
    const unsigned nblocks = (unsigned)(per_view * (size_t)nvc);
    const ViewD *vw = views + v0;
    float *pj = proj + (size_t)v0 * P.nu * P.nv;
    if constexpr (ZC > 0)
      hipLaunchKernelGGL((k_fp_colc<T, RPL, ZC, D>), dim3(nblocks), dim3(64), lds, s, Q, vw, vt, pj, acc,
                         ngroups, nblocks, vt_bytes);
    else
      hipLaunchKernelGGL((k_fp_col<T, RPL, SSTEP, ZP>), dim3(nblocks), dim3(64), lds, s, Q, vw, vt, pj,
                         acc, ngroups, nblocks, vt_bytes);
  }
}

// Column-engine variant and tile.  variant 0: per ray; 1: vector step setup,
// one z per load; 2: scalar step setup, two z per load; 3: variant 2 with the
// corner z-lines cached in registers over a whole-ray window of at most 64 zc z
// (k_fp_colc), zc z per lane.
struct FPChoice {
  int variant;
  int rpl;      // rows per lane
  int zc = 0;
  int vg = 0;   // views per launch group; 0 = the context's setting
};
// Deep variants (the lines of four steps in flight): windows of 64 and 128 z, up
// to 4 rows per lane, for launches of fewer waves than hide each other's
// latencies (8 per SIMD); a property of each launch, also of a tuned choice.  64^3, 9 views
// (864 waves) 40 -> 31 us with the padded copy, 96^3, 10 views (1500) 61 -> 51,
// 128^3, 24 views (6144) 136 -> 125; from 12288 waves on they cost 2-9%, and
// with wider windows they gain nothing.
constexpr int FP_DEEP_RPL = 4, FP_DEEP_ZC = 2;
constexpr size_t FP_DEEP_WAVES = 8192;

template <typename T, int RPL>
void launch_col_w(const FPParams &P, const FPChoice &c, hipStream_t s, const ViewD *views, const T *vt,
                  float *proj, int acc, int nviews, unsigned vt_bytes) {
  if (c.variant == 1) return launch_col<T, RPL, false, 1, 0>(P, s, views, vt, proj, acc, nviews, vt_bytes);
  if (c.variant == 2) return launch_col<T, RPL, true, 2, 0>(P, s, views, vt, proj, acc, nviews, vt_bytes);
  if constexpr (RPL <= FP_DEEP_RPL) {
    const size_t groups = (P.nv + 64 * RPL - 1) / (64 * RPL);
    const bool deep = c.zc <= FP_DEEP_ZC && groups * P.nu * nviews < FP_DEEP_WAVES;
    if (deep && c.zc == 1) return launch_col<T, RPL, true, 2, 1, 4>(P, s, views, vt, proj, acc, nviews, vt_bytes);
    if (deep && c.zc == 2) return launch_col<T, RPL, true, 2, 2, 4>(P, s, views, vt, proj, acc, nviews, vt_bytes);
  }
  switch (c.zc) {
    case 1: launch_col<T, RPL, true, 2, 1>(P, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 2: launch_col<T, RPL, true, 2, 2>(P, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 3: launch_col<T, RPL, true, 2, 3>(P, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 4: launch_col<T, RPL, true, 2, 4>(P, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 5: launch_col<T, RPL, true, 2, 5>(P, s, views, vt, proj, acc, nviews, vt_bytes); break;
    default: launch_col<T, RPL, true, 2, 6>(P, s, views, vt, proj, acc, nviews, vt_bytes); break;
  }
}

// Most rows per lane and most z per lane of a cached line.
constexpr int FP_RPL_MAX = 12, FP_ZC_MAX = 6;
// Configured tile; unset: 8 (engine 1 chooses by itself, see default_variant).
inline int col_tile(const cbct_ctx ctx) { return ctx->fp_max_rpl ? ctx->fp_max_rpl : 8; }

// Rows per lane that dispatch_col picks for max_rpl.
inline int rows_per_lane(int nv, int max_rpl) {
  const int need = (nv + 63) / 64;
  const int groups = (need + max_rpl - 1) / max_rpl;
  return (need + groups - 1) / groups;
}

// Launch with `rpl` rays per lane (1..12; rows_per_lane splits the rows
// into equal groups of whole 64-row blocks).  More rows per wave share one
// z-line load; fewer keep registers, and so occupancy, in check.
template <typename T>
void dispatch_col(const FPParams &P, const FPChoice &c, hipStream_t s, const ViewD *views, const T *vt,
                  float *proj, int acc, int nviews, unsigned vt_bytes) {
  switch (c.rpl) {
    case 1: launch_col_w<T, 1>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 2: launch_col_w<T, 2>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 3: launch_col_w<T, 3>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 4: launch_col_w<T, 4>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 5: launch_col_w<T, 5>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 6: launch_col_w<T, 6>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 7: launch_col_w<T, 7>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 8: launch_col_w<T, 8>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 9: launch_col_w<T, 9>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 10: launch_col_w<T, 10>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    case 11: launch_col_w<T, 11>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
    default: launch_col_w<T, 12>(P, c, s, views, vt, proj, acc, nviews, vt_bytes); break;
  }
}

// Bound on a row group's whole-ray z window in voxels, over all groups of rpl
// rows per lane.  A ray through detector height v (offset included) is at z =
// v t / SDD where t, its depth along the central ray, lies in [SAD - R, SAD + R]
// inside the box (R: half the box's xy diagonal); the window spans the extremes
// of v t over the group's rows and that depth range, no further than the box
// itself (rays that leave through its top or bottom are not shared), plus the
// texel, the window's alignment (3) and rounding slack.
double window_bound(const cbct_geom *g, int nv, int rpl, float omin, float omax) {
  const double R = 0.5 * std::sqrt((double)g->lx * g->lx + (double)g->ly * g->ly);
  const double t0 = (double)g->sad - R, t1 = (double)g->sad + R;
  const double pitch = (double)g->fov_v / nv, vz = (double)g->lz / g->nz, hz = 0.5 * g->lz;
  double worst = 0.0;
  for (int row0 = 0; row0 < nv; row0 += 64 * rpl) {
    const int row1 = std::min(nv, row0 + 64 * rpl) - 1;
    const double v0 = ((row0 + 0.5) / nv - 0.5) * g->fov_v + omin - 0.5 * pitch;
    const double v1 = ((row1 + 0.5) / nv - 0.5) * g->fov_v + omax + 0.5 * pitch;
    const double e[4] = {v0 * t0, v0 * t1, v1 * t0, v1 * t1};
    const double lo = std::min(std::min(e[0], e[1]), std::min(e[2], e[3])) / g->sdd;
    const double hi = std::max(std::max(e[0], e[1]), std::max(e[2], e[3])) / g->sdd;
    worst = std::max(worst, (std::min(hi, hz) - std::max(lo, -hz)) / vz);
  }
  return worst + 6.0;
}

// z per lane of the cached variant whose window holds every row group at rpl
// rows per lane (may exceed FP_ZC_MAX: no such variant).
int window_zc(cbct_ctx ctx, const cbct_geom *g, int nv, int rpl, int view0, int nviews) {
  float omin = 0.0f, omax = 0.0f;
  for (int k = 0; k < nviews; ++k) {
    const float ov = ctx->offsets[2 * (size_t)(view0 + k) + 1];
    omin = k ? fminf(omin, ov) : ov;
    omax = k ? fmaxf(omax, ov) : ov;
  }
  return (int)std::min(1e6, std::ceil(window_bound(g, nv, rpl, omin, omax) / 64.0));
}

// Engine 1's choice: the cached variant with the tile (rows per lane) and the
// window (64 zc z) that cost least per step over the whole column, among those
// whose window fits.  A step of one wave costs about 12 vector instructions, 7
// per row and lane and, per z and lane, 6 (FP32 copies) or 10 (BF16, unpacking
// included); a column has as many waves as row groups.  Measured beside it
// (FP32 copies): 128^3, 180 views, 192 rows: rpl 3 with zc 2 0.69 ms, zc 3 0.80,
// zc 4 0.97; rpl 2 in two groups 1.21; 291^3, 32 views, 500 rows: rpl 8 with zc 5
// 1.56 ms, 4 with 3 1.98, 3 with 2 2.15; 512^3, 48 views, 768 rows: 6 with 4
// 12.6, 4 with 3 13.9, 3 with 3 17.2.  Windows wider than 384 z take the
// per-step variant measured fastest for the storage type.
FPChoice default_variant(cbct_ctx ctx, const cbct_geom *g, const FPParams &P, int view0, int nviews,
                         size_t esz, int per_step) {
  FPChoice best{per_step, rows_per_lane(P.nv, col_tile(ctx))};
  int best_cost = INT_MAX;
  for (int r = ctx->fp_max_rpl ? ctx->fp_max_rpl : FP_RPL_MAX; r >= 1; --r) {
    const int rpl = rows_per_lane(P.nv, r);
    const int zc = window_zc(ctx, g, P.nv, rpl, view0, nviews);
    const int groups = (P.nv + 64 * rpl - 1) / (64 * rpl);
    const int cost = groups * (12 + 7 * rpl + (esz == 2 ? 10 : 6) * zc);
    if (zc <= FP_ZC_MAX && cost < best_cost) {
      best_cost = cost;
      best = {3, rpl, zc};
    }
  }
  return best;
}

// Autotuned choices, process-wide (cbct_fp_autotune): the geometry, the
// samples per ray and the working-copy element size pick (variant, tile).
struct TuneKey {
  int nx, ny, nz, nu, nv, esz;
  float lx, ly, lz, fu, fv, sad, sdd, spp;
  bool operator<(const TuneKey &o) const {
    return std::tie(nx, ny, nz, nu, nv, esz, lx, ly, lz, fu, fv, sad, sdd, spp) <
           std::tie(o.nx, o.ny, o.nz, o.nu, o.nv, o.esz, o.lx, o.ly, o.lz, o.fu, o.fv, o.sad, o.sdd,
                    o.spp);
  }
};
struct Tuned {
  FPChoice choice;
  double ms;
};
std::mutex g_tune_mu;
std::map<TuneKey, Tuned> g_tuned;

TuneKey tune_key(const cbct_geom *g, float spp, size_t esz) {
  return {g->nx, g->ny, g->nz, g->nu, g->nv, (int)esz, g->lx, g->ly, g->lz, g->fov_u, g->fov_v,
          g->sad, g->sdd, spp};
}

// The variant cbct_fp runs and its tile: variant 0 = per ray (engine 0, or a
// volume or z-line beyond the column engine's 32-bit byte offsets / 64 KB of
// LDS); engine 1: default_variant; engine 2: the other per-step variant;
// engines 3 and 4: the cached variants (configured tile).
FPChoice select_variant(cbct_ctx ctx, const cbct_geom *g, const FPParams &P, int view0, int nviews,
                        size_t esz, float spp) {
  const size_t vt_bytes = (size_t)P.pzx * padded_dim(g->ny) * esz;
  const size_t zline_bytes = ((P.pz + 127) / 128) * 128 * sizeof(float);
  const int rpl = rows_per_lane(P.nv, col_tile(ctx));
  if (ctx->fp_engine == 0 || vt_bytes + (size_t)P.pzx * esz * 2 >= (1ull << 31) || zline_bytes > 65536)
    return {0, rpl};
  if (ctx->fp_force_variant > 0)
    return {ctx->fp_force_variant, ctx->fp_force_rpl, ctx->fp_force_zc, ctx->fp_force_vg};
  const int per_step = esz == 2 ? 2 : 1;
  if (ctx->fp_engine == 2) return {3 - per_step, rpl};
  if (ctx->fp_engine >= 3) return {3, rpl, ctx->fp_engine == 3 ? 4 : 6};
  FPChoice tuned{0, 0};
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(tune_key(g, spp, esz));
    if (it != g_tuned.end()) tuned = it->second.choice;
  }
  // the key holds no detector offsets: a tuned tile's window is the call's own
  if (tuned.variant == 3) tuned.zc = window_zc(ctx, g, P.nv, tuned.rpl, view0, nviews);
  if (tuned.variant && tuned.zc <= FP_ZC_MAX) return tuned;
  return default_variant(ctx, g, P, view0, nviews, esz, per_step);
}

// Bytes of the padded working copy cbct_fp builds for this call (the
// variant's layout, element size esz).
size_t fp_working_bytes(cbct_ctx ctx, const cbct_geom *g, const FPParams &P, int view0, int nviews,
                        size_t esz, float spp) {
  const FPChoice choice = select_variant(ctx, g, P, view0, nviews, esz, spp);
  if (choice.variant == 0) return (size_t)P.pxy * padded_dim(g->nz) * esz;
  return ((size_t)P.pzx * padded_dim(g->ny) + 1024) * esz;
}

// Bytes of the packed copy from which k_fp_clip takes the rays that leave through
// the top or bottom; 0: they stay with the column kernels.
size_t clip_cells(cbct_ctx ctx, const cbct_geom *g, const FPParams &P, int view0, int nviews, size_t esz) {
  if (!ctx->fp_packed) return 0;
  double rows = 0.0;
  for (int k = 0; k < nviews; ++k) rows += fp_clipped_rows(g, ctx->offsets[2 * (size_t)(view0 + k) + 1]);
  return fp_cells_bytes(g, rows, P.n, esz);
}

// TI: the caller's volume type; T: the padded working copy's type.  The
// working copy goes to the context's workspace, or to `ext` when given (the
// caller has checked it holds fp_working_bytes).
template <typename TI, typename T>
int run_fp(cbct_ctx ctx, const cbct_geom *g, const FPParams &P, int view0, int nviews,
           const TI *vol, float *proj, int accumulate, hipStream_t s, float spp,
           void *ext = nullptr) {
  const size_t esz = sizeof(T);
  const ViewD *views = ctx->d_views_d + view0;
  const size_t vt_bytes = (size_t)P.pzx * padded_dim(g->ny) * esz;
  const FPChoice choice = select_variant(ctx, g, P, view0, nviews, esz, spp);
  if (choice.variant == 0) {
    const size_t npad = (size_t)P.pxy * padded_dim(g->nz);
    if (!ext) {
      int rc = cbct_reserve(ctx, ctx->ws->vol_pad, npad * esz);
      if (rc) return rc;
    }
    T *vp = static_cast<T *>(ext ? ext : ctx->ws->vol_pad.ptr);
    hipLaunchKernelGGL((k_pad_volume<TI, T>), stride_grid(npad), dim3(256), 0, s, vol, vp, g->nx, g->ny,
                       g->nz, P.px, (unsigned)padded_dim(g->ny), (unsigned)padded_dim(g->nz));
    CBCT_LAUNCH_CHECK(ctx, "k_pad_volume");
    dim3 block(16, 16);
    dim3 grid(ceil_div(g->nu, 16), ceil_div(g->nv, 16), nviews);
    cbct_prof_mark(ctx, PROF_FP, 0, s);
    hipLaunchKernelGGL(k_fp_ray<T>, grid, block, 0, s, P, views, vp, proj, accumulate);
    cbct_prof_mark(ctx, PROF_FP, 1, s);
    CBCT_LAUNCH_CHECK(ctx, "k_fp_ray");
    return CBCT_OK;
  }
  const size_t py = padded_dim(g->ny);
  const size_t npad = (size_t)P.pzx * py;
  // z-line chunk loads may run up to 127 elements past a column's end (those
  // values are never used); the slack keeps such reads inside this allocation
  if (!ext) {
    int rc = cbct_reserve(ctx, ctx->ws->vol_pad, (npad + 1024) * esz);
    if (rc) return rc;
  }
  T *vt = static_cast<T *>(ext ? ext : ctx->ws->vol_pad.ptr);
  dim3 tgrid(ceil_div(P.pz, 32), ceil_div(P.px, 32), (unsigned)py);
  hipLaunchKernelGGL((k_pad_transpose<TI, T>), tgrid, dim3(32, 8), 0, s, vol, vt, g->nx, g->ny, g->nz,
                     P.px, P.pz);
  CBCT_LAUNCH_CHECK(ctx, "k_pad_transpose");
  FPParams Q = P;
  if (choice.vg > 0) Q.vg = (unsigned)choice.vg;
  // without memory for the packed copy the column kernels take every ray
  const size_t cell_bytes = ext ? 0 : clip_cells(ctx, g, P, view0, nviews, esz);
  Q.split = cell_bytes && cbct_reserve_cells(ctx, cell_bytes, cbct_capturing(s));
  const unsigned nslots = ceil_div(P.nv, 64);
  T *cells = static_cast<T *>(ctx->ws->vol_cells.ptr);
  if (Q.split) {
    hipLaunchKernelGGL(k_pack_cells<T>, dim3(std::min(ceil_div(npad / 4, 256), 65536u)), dim3(256), 0, s, vt, cells,
                       P.pz, P.px, (unsigned)py);
    CBCT_LAUNCH_CHECK(ctx, "k_pack_cells");
  }
  cbct_prof_mark(ctx, PROF_FP, 0, s);
  dispatch_col<T>(Q, choice, s, views, vt, proj, accumulate, nviews, (unsigned)vt_bytes);
  if (Q.split) {
    // at most 2^32 - 1 work-items per launch, as launch_col
    const size_t per_view = (size_t)P.nu * nslots;
    const int max_views = (int)std::max<size_t>(1, std::min<size_t>(nviews, ((1ull << 32) - 1) / 64 / per_view));
    for (int v0 = 0; v0 < nviews; v0 += max_views) {
      const unsigned nblocks = (unsigned)(per_view * (size_t)std::min(max_views, nviews - v0));
      hipLaunchKernelGGL(k_fp_clip<T>, dim3(nblocks), dim3(64), 0, s, Q, views + v0, cells,
                         proj + (size_t)v0 * P.nu * P.nv, accumulate, nslots, nblocks, (unsigned)cell_bytes);
    }
  }
  cbct_prof_mark(ctx, PROF_FP, 1, s);
  CBCT_LAUNCH_CHECK(ctx, "k_fp_col");
  return CBCT_OK;
}

}  // namespace

extern "C" {

int cbct_fp_engine(cbct_ctx ctx, int engine) {
  if (!ctx) return CBCT_ERR_ARG;
  if (engine < 0 || engine > 4)
    return cbct_fail(ctx, CBCT_ERR_UNSUPPORTED, "cbct_fp_engine: engine %d not available", engine);
  ctx->fp_engine = engine;
  return CBCT_OK;
}

int cbct_fp_autotune(cbct_ctx ctx, const cbct_geom *g, int view0, int nviews, int dtype, float spp,
                     int retune, void *stream, double *best_ms) {
  if (!ctx) return CBCT_ERR_ARG;
  const char *who = "cbct_fp_autotune";
  int rc = cbct_check_geom(ctx, g, who);
  if (rc) return rc;
  rc = cbct_check_views(ctx, view0, nviews, who);
  if (rc) return rc;
  if (nviews <= 0) return cbct_fail(ctx, CBCT_ERR_ARG, "%s: no views", who);
  if (dtype != CBCT_F32 && dtype != CBCT_BF16)
    return cbct_fail(ctx, CBCT_ERR_UNSUPPORTED, "%s: unsupported volume dtype %d", who, dtype);
  FPParams P;
  rc = make_params(ctx, g, spp, P);
  if (rc) return rc;
  rc = cbct_set_device(ctx);
  if (rc) return rc;
  const size_t esz = (dtype == CBCT_BF16 || ctx->work_dtype == CBCT_BF16) ? 2 : 4;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(tune_key(g, spp, esz));
    if (it != g_tuned.end()) {
      if (!retune) {
        if (best_ms) *best_ms = it->second.ms;
        return CBCT_OK;
      }
      g_tuned.erase(it);   // time the built-in choice itself
    }
  }
  const int saved_engine = ctx->fp_engine;
  ctx->fp_engine = 1;
  const FPChoice heuristic = select_variant(ctx, g, P, view0, nviews, esz, spp);
  ctx->fp_engine = saved_engine;
  if (heuristic.variant == 0) return CBCT_OK;   // the column engines do not apply
  // candidates: the heuristic's; the cached variants at several tiles with the
  // windows they need; the per-step variant of the storage type
  std::vector<FPChoice> cand{heuristic};
  auto add = [&](int v, int r, int zc) {
    for (auto &c : cand)
      if (c.variant == v && c.rpl == r && c.zc == zc) return;
    cand.push_back({v, r, zc});
  };
  for (int m : {2, 4, 6, 8, 12}) {
    const int rpl = rows_per_lane(P.nv, m), zc = window_zc(ctx, g, P.nv, rpl, view0, nviews);
    if (zc <= FP_ZC_MAX) add(3, rpl, zc);
  }
  add(esz == 2 ? 2 : 1, rows_per_lane(P.nv, 8), 0);
  // scratch volume and projections (contents do not change the timing)
  const size_t nvox = (size_t)g->nx * g->ny * g->nz;
  const size_t nproj = (size_t)g->nu * g->nv * (size_t)nviews;
  void *vol = nullptr, *proj = nullptr;
  CBCT_HIP_CHECK(ctx, hipMalloc(&vol, nvox * (dtype == CBCT_BF16 ? 2 : 4)));
  if (hipMalloc(&proj, nproj * sizeof(float)) != hipSuccess) {
    (void)hipFree(vol);
    (void)hipGetLastError();
    return cbct_fail(ctx, CBCT_ERR_NOMEM, "%s: scratch allocation failed", who);
  }
  hipStream_t s = as_stream(stream);
  CallScope scope(ctx, s);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  const size_t vol_words = nvox * (dtype == CBCT_BF16 ? 2 : 4) / 4;   // whole 4-byte words
  hipLaunchKernelGGL(k_zero, stride_grid(vol_words), dim3(256), 0, s, vol_words, static_cast<float *>(vol));
  FPChoice best = heuristic;
  double best_t = 1e300;
  auto trial = [&](const FPChoice &c) {
    ctx->fp_force_variant = c.variant;
    ctx->fp_force_rpl = c.rpl;
    ctx->fp_force_zc = c.zc;
    ctx->fp_force_vg = c.vg;
    double t = 1e300;
    for (int rep = 0; rep < 3 && rc == CBCT_OK; ++rep) {   // first run warms up
      (void)hipEventRecord(e0, s);
      rc = cbct_fp(ctx, g, view0, nviews, vol, dtype, static_cast<float *>(proj), spp, 0, stream);
      (void)hipEventRecord(e1, s);
      if (rc == CBCT_OK && hipEventSynchronize(e1) == hipSuccess && rep > 0) {
        float ms = 0.0f;
        if (hipEventElapsedTime(&ms, e0, e1) == hipSuccess) t = std::min(t, (double)ms);
      }
    }
    if (t < best_t) {
      best_t = t;
      best = c;
    }
  };
  // the variants and tiles at the context's launch order, then the launch
  // order (views per group) for the fastest of them
  for (size_t c = 0; c < cand.size() && rc == CBCT_OK; ++c) trial(cand[c]);
  const FPChoice base = best;
  for (int vg : {1, 3, 6, 8})
    if (rc == CBCT_OK && vg != ctx->fp_view_group) trial({base.variant, base.rpl, base.zc, vg});
  ctx->fp_force_variant = 0;
  ctx->fp_force_rpl = 0;
  ctx->fp_force_zc = 0;
  ctx->fp_force_vg = 0;
  (void)hipStreamSynchronize(s);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipFree(vol);
  (void)hipFree(proj);
  if (rc) return rc;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned[tune_key(g, spp, esz)] = {best, best_t};
  }
  if (best_ms) *best_ms = best_t;
  return CBCT_OK;
}

int cbct_fp_autotune_clear(void) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tuned.clear();
  return CBCT_OK;
}

int cbct_fp_tile(cbct_ctx ctx, int max_rows_per_lane) {
  if (!ctx) return CBCT_ERR_ARG;
  if (max_rows_per_lane < 1 || max_rows_per_lane > 12)
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_fp_tile: rows per lane %d outside 1..12", max_rows_per_lane);
  ctx->fp_max_rpl = max_rows_per_lane;
  return CBCT_OK;
}

int cbct_fp_packed(cbct_ctx ctx, int on) {
  if (!ctx) return CBCT_ERR_ARG;
  ctx->fp_packed = on != 0;
  return CBCT_OK;
}

int cbct_fp_view_group(cbct_ctx ctx, int views) {
  if (!ctx) return CBCT_ERR_ARG;
  if (views < 1 || views > 64)
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_fp_view_group: %d views outside 1..64", views);
  ctx->fp_view_group = views;
  return CBCT_OK;
}

const char *cbct_fp_kernel(cbct_ctx ctx, const cbct_geom *g, int view0, int nviews, int dtype,
                           float spp) {
  if (!ctx || !g || cbct_check_geom(ctx, g, "cbct_fp_kernel") ||
      cbct_check_views(ctx, view0, nviews, "cbct_fp_kernel"))
    return "";
  FPParams P;
  if (make_params(ctx, g, spp, P)) return "";
  const size_t esz = (dtype == CBCT_BF16 || ctx->work_dtype == CBCT_BF16) ? 2 : 4;
  const int v = select_variant(ctx, g, P, view0, nviews, esz, spp).variant;
  return v == 0 ? "k_fp_ray" : v == 3 ? "k_fp_colc" : "k_fp_col";
}

}  // extern "C"

namespace {

// Argument checks and parameters shared by cbct_fp and cbct_fp_noalloc.
int fp_prepare(cbct_ctx ctx, const cbct_geom *g, int view0, int nviews, const void *vol, int dtype,
               float *proj, float spp, FPParams &P) {
  const char *who = "conebeam_forwards_projection";
  if (!vol || !proj)
    return cbct_fail(ctx, CBCT_ERR_ARG, "Error: %s: illegal array pointer provided", who);
  int rc = cbct_check_geom(ctx, g, who);
  if (rc) return rc;
  rc = cbct_check_views(ctx, view0, nviews, who);
  if (rc) return rc;
  if (dtype != CBCT_F32 && dtype != CBCT_BF16)
    return cbct_fail(ctx, CBCT_ERR_UNSUPPORTED, "Error: %s: unsupported volume dtype %d", who, dtype);
  if (nviews == 0) return CBCT_OK;   // nothing to do (the caller returns)
  if (nviews > 65535)
    return cbct_fail(ctx, CBCT_ERR_ARG, "Error: %s: at most 65535 views per call", who);
  if ((size_t)g->nu * (size_t)((g->nv + 63) / 64) * (size_t)nviews >= (1ull << 31))
    return cbct_fail(ctx, CBCT_ERR_ARG, "Error: %s: too many rays per call", who);
  rc = make_params(ctx, g, spp, P);
  if (rc) return rc;
  return cbct_set_device(ctx);
}

template <typename TI, typename T>
int run_fp_as(cbct_ctx ctx, const cbct_geom *g, const FPParams &P, int view0, int nviews,
              const void *vol, float *proj, int accumulate, hipStream_t s, float spp, void *ext) {
  return run_fp<TI, T>(ctx, g, P, view0, nviews, static_cast<const TI *>(vol), proj, accumulate, s,
                       spp, ext);
}

int run_fp_dtype(cbct_ctx ctx, const cbct_geom *g, const FPParams &P, int view0, int nviews,
                 const void *vol, int dtype, float *proj, int accumulate, hipStream_t s, float spp,
                 void *ext) {
  if (dtype == CBCT_BF16)
    return run_fp_as<unsigned short, unsigned short>(ctx, g, P, view0, nviews, vol, proj, accumulate,
                                                     s, spp, ext);
  if (ctx->work_dtype == CBCT_BF16)
    return run_fp_as<float, unsigned short>(ctx, g, P, view0, nviews, vol, proj, accumulate, s, spp,
                                            ext);
  return run_fp_as<float, float>(ctx, g, P, view0, nviews, vol, proj, accumulate, s, spp, ext);
}

// Per-device address of `scratch`, looked up on a device's first
// cbct_fp_noalloc call.
std::mutex g_scratch_mu;
void *g_scratch_ptr[64] = {};

int fp_scratch(cbct_ctx ctx, void **out) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (ctx->device < 0 || ctx->device >= 64)
    return cbct_fail(ctx, CBCT_ERR_UNSUPPORTED, "cbct_fp_noalloc: device %d out of range", ctx->device);
  if (!g_scratch_ptr[ctx->device]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return cbct_fail(ctx, CBCT_ERR_HIP, "cbct_fp_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
    g_scratch_ptr[ctx->device] = p;
  }
  *out = g_scratch_ptr[ctx->device];
  return CBCT_OK;
}

}  // namespace

extern "C" {

int cbct_fp(cbct_ctx ctx, const cbct_geom *g, int view0, int nviews, const void *vol, int dtype,
            float *proj, float spp, int accumulate, void *stream) {
  if (!ctx) return CBCT_ERR_ARG;
  FPParams P;
  int rc = fp_prepare(ctx, g, view0, nviews, vol, dtype, proj, spp, P);
  if (rc || nviews == 0) return rc;
  hipStream_t s = as_stream(stream);
  CallScope scope(ctx, s);
  return run_fp_dtype(ctx, g, P, view0, nviews, vol, dtype, proj, accumulate, s, spp, nullptr);
}

int cbct_fp_noalloc(cbct_ctx ctx, const cbct_geom *g, int view0, int nviews, const void *vol,
                    int dtype, float *proj, float spp, int accumulate, void *stream) {
  if (!ctx) return CBCT_ERR_ARG;
  FPParams P;
  int rc = fp_prepare(ctx, g, view0, nviews, vol, dtype, proj, spp, P);
  if (rc || nviews == 0) return rc;
  const size_t esz = (dtype == CBCT_BF16 || ctx->work_dtype == CBCT_BF16) ? 2 : 4;
  const size_t need = fp_working_bytes(ctx, g, P, view0, nviews, esz, spp);
  if (need > FP_SCRATCH_BYTES)
    return cbct_fail(ctx, CBCT_ERR_UNSUPPORTED,
                     "cbct_fp_noalloc: the volume's working copy needs %zu bytes, more than the %zu "
                     "bytes of scratch (use cbct_fp)", need, FP_SCRATCH_BYTES);
  void *ptr = nullptr;
  rc = fp_scratch(ctx, &ptr);
  if (rc) return rc;
  hipStream_t s = as_stream(stream);
  rc = run_fp_dtype(ctx, g, P, view0, nviews, vol, dtype, proj, accumulate, s, spp, ptr);
  // this call read the view table: a later cbct_views_set waits for it.  On an
  // event of its own, so that the end of the last call in the workspace stays
  // marked; calls that share the scratch are in order, so the last one's end is
  // the end of all
  if (rc == CBCT_OK && !cbct_capturing(s) && hipEventRecord(ctx->noalloc_done.e, s) == hipSuccess)
    ctx->noalloc_recorded = true;
  return rc;
}

int cbct_fp_transpose(cbct_ctx ctx, const cbct_geom *g, int view0, int nviews, const float *proj,
                      float *vol, float spp, int accumulate, void *stream) {
  if (!ctx) return CBCT_ERR_ARG;
  const char *who = "cbct_fp_transpose";
  if (!vol || !proj)
    return cbct_fail(ctx, CBCT_ERR_ARG, "Error: %s: illegal array pointer provided", who);
  int rc = cbct_check_geom(ctx, g, who);
  if (rc) return rc;
  rc = cbct_check_views(ctx, view0, nviews, who);
  if (rc) return rc;
  if (nviews > 65535)
    return cbct_fail(ctx, CBCT_ERR_ARG, "Error: %s: at most 65535 views per call", who);
  FPParams P;
  rc = make_params(ctx, g, spp, P);
  if (rc) return rc;
  rc = cbct_set_device(ctx);
  if (rc) return rc;
  hipStream_t s = as_stream(stream);
  CallScope scope(ctx, s);
  const size_t npad = (size_t)P.pxy * padded_dim(g->nz);
  rc = cbct_reserve(ctx, ctx->ws->vol_pad, npad * sizeof(float));
  if (rc) return rc;
  float *acc = static_cast<float *>(ctx->ws->vol_pad.ptr);
  hipLaunchKernelGGL(k_zero, stride_grid(npad), dim3(256), 0, s, npad, acc);
  CBCT_LAUNCH_CHECK(ctx, "k_zero");
  if (nviews > 0) {
    dim3 block(16, 16);
    dim3 grid(ceil_div(g->nu, 16), ceil_div(g->nv, 16), nviews);
    hipLaunchKernelGGL(k_fp_ray_transpose, grid, block, 0, s, P, ctx->d_views_d + view0, proj, acc);
    CBCT_LAUNCH_CHECK(ctx, "k_fp_ray_transpose");
  }
  const size_t nvox = (size_t)g->nx * g->ny * g->nz;
  hipLaunchKernelGGL(k_unpad_add, stride_grid(nvox), dim3(256), 0, s, acc, vol, g->nx, g->ny,
                     g->nz, P.px, P.pxy, accumulate);
  CBCT_LAUNCH_CHECK(ctx, "k_unpad_add");
  return CBCT_OK;
}

}  // extern "C"
