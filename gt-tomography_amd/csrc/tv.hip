// Isotropic TV primal-dual step, fused into one pass.
//
// The reference (operators/cuTVPrimalDualOperator.cu:10-106) runs a primal
// kernel that writes the projected gradient field p (3*Nvox floats) and a
// dual kernel that reads it back, with a device synchronisation in between.
// Here p never leaves the chip: a wave owns 64 x by TV_RY y and walks along z,
// evaluating the projected gradient once per voxel.  The dual's p(v-ey) and
// p(v-ez) are the thread's own from the row before and the slice before,
// p(v-ex) is the neighbouring lane's.  HBM traffic per voxel is 3 floats (read
// x, read + write out).  The arithmetic is the reference's, in the same order,
// but for the divisions by the norm (tv_grad), which may differ from plain ones in
// the last bit.
#include "cbct_internal.h"

namespace {

// Rows per wave.  A wave evaluates TV_RY + 2 gradients per slice (its rows, the
// row before them, and the column before lane 0, one lane per row); fewer rows
// evaluate more but keep more waves in flight (256^3: 2 rows 64 us, 4 rows 70).
constexpr int TV_RY = 2;

struct TVArgs {
  int nx, ny, nz, zchunk, nchunks;   // slices per wave, waves along z
  float scale, weight;               // (weight*sigma)/(1+sigma*alpha); weight
  int accumulate;                    // TV alone
  const float *s, *p;                // with updateG
  float tau, tl;
};

struct Grad {
  float x, y, z;
};

// Projected, scaled forward-difference gradient from a voxel's value and its
// three successors': cuTVPrimalKernel (operators/cuTVPrimalDualOperator.cu:10-38),
// g / max(1, |g|).  The norm's square root and the three divisions by it are
// one reciprocal square root and one reciprocal, each refined by its exact
// FMA residual (Markstein 1990), which gives the correctly rounded quotients
// but for rare last bits; the compiler's own sequences scale and fix up
// exponents that cannot occur here (52 against 29 instructions per gradient).
// Norms whose square overflows, infinities and NaN take the plain operations.
__device__ __forceinline__ Grad tv_grad(float c, float cx, float cy, float cz, float scale) {
  const float g0 = (cx - c) * scale, g1 = (cy - c) * scale, g2 = (cz - c) * scale;
  const float a = g0 * g0 + g1 * g1 + g2 * g2;
  if (!(a < INFINITY)) {
    const float den = fmaxf(1.0f, sqrtf(a));
    return {g0 / den, g1 / den, g2 / den};
  }
  const float am = fmaxf(a, 1.0f);   // max(1, |g|) = sqrt(max(1, |g|^2))
  const float y = __builtin_amdgcn_rsqf(am);
  float den = am * y;
  den = fmaf(fmaf(-den, den, am), 0.5f * y, den);
  float r = __builtin_amdgcn_rcpf(den);
  r = fmaf(fmaf(-den, r, 1.0f), r, r);
  auto div = [&](float g) __attribute__((always_inline)) {
    const float q = g * r;
    return fmaf(fmaf(-den, q, g), r, q);
  };
  return {div(g0), div(g1), div(g2)};
}

// UPDATE: xout = updateG(0 + TV(x), x, s, p) (solvers/osMOMSolverD.h:233-247);
// else out = (accumulate ? out : 0) + TV(x).  Periodic boundaries.
// One gradient per voxel (4 / 2 with the tile's borders) instead of four, with
// the cheaper divisions, takes the kernel from the vector unit's bound close to
// HBM's: 256^3, updateG, 128 -> 64 us (4.2 of the 4.8 TB/s that a device copy
// reaches; 77 us with the compiler's divisions); 448^3 677 -> 376 us.
template <bool UPDATE>
__global__ void __launch_bounds__(256) k_tv(TVArgs A, const float *__restrict__ in, float *__restrict__ out) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int x0 = blockIdx.x * 64, x = x0 + lane, y0 = (blockIdx.y * 4 + wave) * TV_RY;
  if (y0 >= A.ny) return;
  const int b = blockIdx.z / A.nchunks, z0 = (blockIdx.z % A.nchunks) * A.zchunk;
  const int z1 = min(z0 + A.zchunk, A.nz);
  const size_t plane = (size_t)A.nx * A.ny, vol = plane * A.nz * b;
  const float *v = in + vol;
  // lanes past the row read its last voxel and write nothing
  const int xc = min(x, A.nx - 1), xp = xc + 1 == A.nx ? 0 : xc + 1, xm = x0 == 0 ? A.nx - 1 : x0 - 1;
  // row r - 1 of the tile, periodic (rows past the volume's are not used)
  size_t row[TV_RY + 2];
#pragma unroll
  for (int r = 0; r < TV_RY + 2; ++r) {
    const int y = y0 + r - 1;
    row[r] = (size_t)(y < 0 ? A.ny - 1 : y < A.ny ? y : y % A.ny) * A.nx;
  }
  // the column before lane 0: lane t holds row t's
  const int yh = y0 + min(lane, TV_RY - 1), yh0 = yh % A.ny, yh1 = (yh + 1) % A.ny;
  const size_t h0 = (size_t)yh0 * A.nx, h1 = (size_t)yh1 * A.nx;

  float c[TV_RY + 2], pz[TV_RY], ch;
  int z = z0 == 0 ? A.nz - 1 : z0 - 1;   // the slice before the first, for its p(v-ez)
  const float *vz = v + plane * z;
#pragma unroll
  for (int r = 0; r < TV_RY + 2; ++r) c[r] = vz[row[r] + xc];
  ch = vz[h0 + xm];
  for (int k = z0 - 1; k < z1; ++k) {
    const int zn = z + 1 == A.nz ? 0 : z + 1;
    const float *vn = v + plane * zn;
    float n[TV_RY + 2], cx[TV_RY + 1];
#pragma unroll
    for (int r = 0; r < TV_RY + 2; ++r) n[r] = vn[row[r] + xc];
#pragma unroll
    for (int r = 0; r < TV_RY + 1; ++r) cx[r] = vz[row[r] + xp];
    const float nh = vn[h0 + xm], hx = vz[h0 + x0], hy = vz[h1 + xm];
    const float ph = tv_grad(ch, hx, hy, nh, A.scale).x;
    float py = tv_grad(c[0], cx[0], c[1], n[0], A.scale).y;
#pragma unroll
    for (int r = 0; r < TV_RY; ++r) {
      const Grad p0 = tv_grad(c[r + 1], cx[r + 1], c[r + 2], n[r + 1], A.scale);
      // lane - 1's p0.x; lane 0 keeps the column before
      const float px = __int_as_float(__builtin_amdgcn_update_dpp(
          __builtin_amdgcn_readlane(__float_as_int(ph), r), __float_as_int(p0.x), 0x138, 0xf, 0xf, false));
      // negative divergence times the weight: cuTVDualKernel (:41-66)
      float t = 0.0f;
      t += px - p0.x;
      t += py - p0.y;
      t += pz[r] - p0.z;
      py = p0.y;
      pz[r] = p0.z;
      if (k >= z0 && x < A.nx && y0 + r < A.ny) {
        const float tv = t * A.weight;
        const size_t i = vol + plane * z + row[r + 1] + x;
        if constexpr (UPDATE) {
          const float g = 0.0f + tv, pr = A.p[i];
          float xv = fmaf(-A.tau, g, c[r + 1]);
          xv = fmaf(A.tl, A.s[i] / pr, xv);
          out[i] = xv / ((1.0f / pr) * A.tl + 1.0f);
        } else {
          out[i] = A.accumulate ? out[i] + tv : tv;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < TV_RY + 2; ++r) c[r] = n[r];
    ch = nh;
    vz = vn;
    z = zn;
  }
}

// Slices per wave: each wave evaluates one slice more than it writes, so as
// many as leave TV_WAVES waves, 1 to 32 (256^3: 8192 waves 71 us, 16384 64).
constexpr size_t TV_WAVES = 16384;
void launch_tv(TVArgs A, int nvol, const float *x, float *out, bool update, hipStream_t s) {
  const dim3 tiles(ceil_div(A.nx, 64), ceil_div(A.ny, 4 * TV_RY));
  const size_t per_slice = (size_t)tiles.x * ceil_div(A.ny, TV_RY) * nvol;
  const size_t want = (size_t)A.nz * per_slice / TV_WAVES;
  A.zchunk = (int)(want < 1 ? 1 : want > 32 ? 32 : want);
  A.nchunks = (int)ceil_div(A.nz, A.zchunk);
  const dim3 grid(tiles.x, tiles.y, (unsigned)A.nchunks * nvol);
  if (update) hipLaunchKernelGGL(k_tv<true>, grid, dim3(256), 0, s, A, x, out);
  else hipLaunchKernelGGL(k_tv<false>, grid, dim3(256), 0, s, A, x, out);
}

}  // namespace

extern "C" {

int cbct_tv_primal_dual(cbct_ctx ctx, int nx, int ny, int nz, int nvol, const float *x, float *out,
                        float sigma, float alpha, float weight, int accumulate, void *stream) {
  if (!ctx) return CBCT_ERR_ARG;
  if (!x || !out)
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_tv_primal_dual: illegal array pointer provided");
  if (nx <= 0 || ny <= 0 || nz <= 0 || nvol <= 0)
    return cbct_fail(ctx, CBCT_ERR_ARG, "Input and reference dimensions must agree");
  if (x == out)
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_tv_primal_dual: input and output must not alias");
  if ((size_t)nz * nvol > 65535u)
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_tv_primal_dual: too many slices");
  int rc = cbct_set_device(ctx);
  if (rc) return rc;
  TVArgs A{};
  A.nx = nx;
  A.ny = ny;
  A.nz = nz;
  const float wsig = weight * sigma, omega = sigma * alpha;
  A.scale = wsig / (1.0f + omega);
  A.weight = weight;
  A.accumulate = accumulate;
  launch_tv(A, nvol, x, out, false, as_stream(stream));
  CBCT_LAUNCH_CHECK(ctx, "k_tv");
  return CBCT_OK;
}

int cbct_tv_update_g(cbct_ctx ctx, int nx, int ny, int nz, int nvol, const float *x_in,
                     float *x_out, const float *s, const float *precon, float sigma, float alpha,
                     float weight, float tau, float avg_lambda, void *stream) {
  if (!ctx) return CBCT_ERR_ARG;
  if (!x_in || !x_out || !s || !precon)
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_tv_update_g: illegal array pointer provided");
  if (nx <= 0 || ny <= 0 || nz <= 0 || nvol <= 0)
    return cbct_fail(ctx, CBCT_ERR_ARG, "Input and reference dimensions must agree");
  if (x_in == x_out)
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_tv_update_g: x_out must not alias x_in");
  if ((size_t)nz * nvol > 65535u)
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_tv_update_g: too many slices");
  if (!(avg_lambda != 0.0f))
    return cbct_fail(ctx, CBCT_ERR_ARG, "cbct_tv_update_g: avg_lambda must be non-zero");
  int rc = cbct_set_device(ctx);
  if (rc) return rc;
  TVArgs A{};
  A.nx = nx;
  A.ny = ny;
  A.nz = nz;
  const float wsig = weight * sigma, omega = sigma * alpha;
  A.scale = wsig / (1.0f + omega);
  A.weight = weight;
  A.s = s;
  A.p = precon;
  A.tau = tau;
  A.tl = tau / avg_lambda;
  launch_tv(A, nvol, x_in, x_out, true, as_stream(stream));
  CBCT_LAUNCH_CHECK(ctx, "k_tv");
  return CBCT_OK;
}

}  // extern "C"
