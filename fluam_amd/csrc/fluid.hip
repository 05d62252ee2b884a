// fluid.hip -- the staggered-grid right-hand side W of each solve (fluam's kernelConstructW
// family) with the stochastic stress generated in registers.
//
// One workgroup owns a 16 x 16 column of cells and ZC planes of it (ZC = 1, 2 or 4), one cell per
// lane.  The velocities of its stencil are loaded first; under those loads the stress normals of the
// ZC + 2 planes (with the one-cell ring the divergence needs) are drawn into LDS, spread over all
// lanes; one barrier; then every lane takes its stencil.  Bound by the generator's instructions: at
// ZC = 4 each normal is drawn 1.9 times.  A column of 256 lanes that marched up the planes, drawing
// one plane per barrier with 62% of its lanes, took 10.1 us at 32^3 and 14.0 us at 64^3 per launch.
// The second solve of an incompressible step has the same noise, so the first pass keeps the terms
// both share and the second only adds its advection.
//
// Restates: kernelConstructW_1/_2 (src/kernelConstructW.cu:32-521), the QNB variants
// (src/kernelConstructWQuasiNeutrallyBuoyant.cu:26-705,1366-2025) and
// kernelConstructWstokesLimit/_2 (src/stokesLimitFunctions.cu:2281-2378,3922-4069).
#include "fhd_device.h"
#include "fhd_kernels.h"

namespace fhd {

constexpr int TX = 16, TY = 16;
constexpr int PX = TX + 2, PY = TY + 2;
constexpr int PLANE = PX * PY;

// Draws the stress of items [0, ntot) of the planes zs - 1 .. zs + ZC: per plane the tile's cells and
// its ring without corners.  Stress components: 0 sXX, 1 XY, 2 XZ, 3 sYY, 4 YZ, 5 sZZ.
template <int ZC>
FHD_DEV void draw_planes(const FluidWArgs& a, const Key& key, float (*nbuf)[6 * PLANE], int x0, int y0, int zs) {
  const GridDev& g = a.g;
  constexpr int NOWN = TX * TY, NPL = NOWN + 2 * TX + 2 * TY;
  for (int e = threadIdx.x; e < (ZC + 2) * NPL; e += 256 * ZC) {
    const int pl = e / NPL, i = e - pl * NPL;
    int lx, ly;
    if (i < NOWN) { lx = i % TX; ly = i / TX; }
    else {
      const int r = i - NOWN;
      if (r < TY) { lx = -1; ly = r; }
      else if (r < 2 * TY) { lx = TX; ly = r - TY; }
      else if (r < 2 * TY + TX) { lx = r - 2 * TY; ly = -1; }
      else { lx = r - 2 * TY - TX; ly = TY; }
    }
    // one conditional wrap each, except in the planes above the box (not used) of a short last chunk
    int x = x0 + lx, y = y0 + ly, z = zs - 1 + pl;
    x = x < 0 ? x + g.mx : (x >= g.mx ? x - g.mx : x);
    y = y < 0 ? y + g.my : (y >= g.my ? y - g.my : y);
    z = z < 0 ? z + g.mz : (z >= g.mz ? z - g.mz : z);
    const uint32_t cell = (uint32_t)(x + g.mx * (y + g.my * z));
    float s[8];
    draw_normals4(key, cell, FHD_STREAM_FLUID, 0, &s[0]);
    draw_normals4(key, cell, FHD_STREAM_FLUID, 1, &s[4]);
    if (a.trace_free) {
      const float tr = (s[0] + s[3] + s[5]) * (1.0f / 3.0f);
      s[0] -= tr;
      s[3] -= tr;
      s[5] -= tr;
    }
    const int p = (lx + 1) + PX * (ly + 1);
#pragma unroll
    for (int c = 0; c < 6; ++c) nbuf[pl][c * PLANE + p] = s[c];
  }
}

// The seven values of a component around a cell: itself, x - 1, x + 1, y - 1, y + 1, z - 1, z + 1.
FHD_DEV void load7(const float* f, const int n[7], float v[7]) {
#pragma unroll
  for (int k = 0; k < 7; ++k) v[k] = f[n[k]];
}

template <int ZC>
FHD_BODY void body_fluid_w(const FluidWArgs& a, const Blk& b) {
  __shared__ float nbuf[ZC + 2][6 * PLANE];
  const GridDev& g = a.g;
  const Key key = resolve_key(a.key);
  const int x0 = b.x * TX, y0 = b.y * TY, zs = b.z * ZC;
  const int lx = threadIdx.x % TX, ly = threadIdx.x / TX % TY, lz = threadIdx.x / (TX * TY);
  const int x = x0 + lx, y = y0 + ly, z = zs + lz;
  const bool own = x < g.mx && y < g.my && z < g.mz;
  const int N = g.N;
  const int xm = x == 0 ? g.mx - 1 : x - 1, xp = x == g.mx - 1 ? 0 : x + 1;
  const int ym = y == 0 ? g.my - 1 : y - 1, yp = y == g.my - 1 ? 0 : y + 1;
  const int zm = z == 0 ? g.mz - 1 : z - 1, zp = z == g.mz - 1 ? 0 : z + 1;
  const auto at = [&](int i, int j, int k) { return i + g.mx * (j + g.my * k); };
  const int n[7] = {at(x, y, z), at(xm, y, z), at(xp, y, z), at(x, ym, z), at(x, yp, z), at(x, y, zm), at(x, y, zp)};
  const int i = n[0];
  float V[3][7], pxmy, pxmz, mxpy, pymz, mxpz, mypz, w[3] = {0.0f, 0.0f, 0.0f};
  if (own) {
#pragma unroll
    for (int c = 0; c < 3; ++c) load7(a.vadv + (size_t)c * N, n, V[c]);
    const float *VX = a.vadv, *VY = VX + N, *VZ = VY + N;
    pxmy = VY[at(xp, ym, z)];
    pxmz = VZ[at(xp, y, zm)];
    mxpy = VX[at(xm, yp, z)];
    pymz = VZ[at(x, yp, zm)];
    mxpz = VX[at(xm, y, zp)];
    mypz = VY[at(x, ym, zp)];
    if (a.base_in) {
#pragma unroll
      for (int c = 0; c < 3; ++c) w[c] = a.base_in[i + (size_t)c * N];
    }
  }
  if (a.noise) {
    draw_planes<ZC>(a, key, nbuf, x0, y0, zs);
    __syncthreads();
  }
  if (!own) return;
  if (a.noise) {
    const float *cur = nbuf[lz + 1], *prv = nbuf[lz], *nxt = nbuf[lz + 2];
    const int p = (lx + 1) + PX * (ly + 1);
    const float f1 = a.f1, f4 = a.f4;
    w[0] = g.idx * f1 * (cur[0 * PLANE + p + 1] - cur[0 * PLANE + p]) +
           g.idy * f4 * (cur[1 * PLANE + p] - cur[1 * PLANE + p - PX]) +
           g.idz * f4 * (cur[2 * PLANE + p] - prv[2 * PLANE + p]);
    w[1] = g.idy * f1 * (cur[3 * PLANE + p + PX] - cur[3 * PLANE + p]) +
           g.idx * f4 * (cur[1 * PLANE + p] - cur[1 * PLANE + p - 1]) +
           g.idz * f4 * (cur[4 * PLANE + p] - prv[4 * PLANE + p]);
    w[2] = g.idz * f1 * (nxt[5 * PLANE + p] - cur[5 * PLANE + p]) +
           g.idx * f4 * (cur[2 * PLANE + p] - cur[2 * PLANE + p - 1]) +
           g.idy * f4 * (cur[4 * PLANE + p] - cur[4 * PLANE + p - PX]);
  }
  if (a.v) {
    const float ax = g.idx * g.idx, ay = g.idy * g.idy, az = g.idz * g.idz;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      float f[7];
      if (a.v == a.vadv) {
#pragma unroll
        for (int k = 0; k < 7; ++k) f[k] = V[c][k];
      } else {
        load7(a.v + (size_t)c * N, n, f);
      }
      const float L = ax * (f[2] - 2.0f * f[0] + f[1]) + ay * (f[4] - 2.0f * f[0] + f[3]) +
                      az * (f[6] - 2.0f * f[0] + f[5]);
      w[c] += a.v_coef * f[0] + a.lap_coef * L;
    }
  }
  if (a.base_out) {
#pragma unroll
    for (int c = 0; c < 3; ++c) a.base_out[i + (size_t)c * N] = w[c];
  }
  // advection (1/4) sum_b D_b[(v_a + v_a')(v_b + v_b')], src/kernelConstructW.cu:120-136; the dt
  // factor is folded into adv_coef by the caller
  const float *vx = V[0], *vy = V[1], *vz = V[2];
  const float Ax = g.idx * ((vx[2] + vx[0]) * (vx[2] + vx[0]) - (vx[0] + vx[1]) * (vx[0] + vx[1])) +
                   g.idy * ((vx[4] + vx[0]) * (vy[2] + vy[0]) - (vx[0] + vx[3]) * (pxmy + vy[3])) +
                   g.idz * ((vx[6] + vx[0]) * (vz[2] + vz[0]) - (vx[0] + vx[5]) * (pxmz + vz[5]));
  const float Ay = g.idx * ((vy[2] + vy[0]) * (vx[4] + vx[0]) - (vy[0] + vy[1]) * (mxpy + vx[1])) +
                   g.idy * ((vy[4] + vy[0]) * (vy[4] + vy[0]) - (vy[0] + vy[3]) * (vy[0] + vy[3])) +
                   g.idz * ((vy[6] + vy[0]) * (vz[4] + vz[0]) - (vy[0] + vy[5]) * (pymz + vz[5]));
  const float Az = g.idx * ((vz[2] + vz[0]) * (vx[6] + vx[0]) - (vz[0] + vz[1]) * (mxpz + vx[1])) +
                   g.idy * ((vz[4] + vz[0]) * (vy[6] + vy[0]) - (vz[0] + vz[3]) * (mypz + vy[3])) +
                   g.idz * ((vz[6] + vz[0]) * (vz[6] + vz[0]) - (vz[0] + vz[5]) * (vz[0] + vz[5]));
  const float A[3] = {0.25f * Ax, 0.25f * Ay, 0.25f * Az};
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const size_t at_c = i + (size_t)c * N;
    w[c] += a.adv_coef * A[c];
    if (a.adv_prev) w[c] += a.adv_prev_coef * a.adv_prev[at_c];
    if (a.adv_store) a.adv_store[at_c] = A[c];
    a.W[at_c] = w[c];
  }
}
FHD_KERNEL_PAIR((template <int ZC>), 256 * ZC, k_fluid_w, FluidWArgs, body_fluid_w<ZC>(a, b))

// Discrete staggered divergence (diagnostic), src/kernelUpdateVIncompressible.cu invariant.
__global__ void k_divergence(GridDev g, const float* __restrict__ v, float* __restrict__ div) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.N) return;
  int x = i % g.mx, y = (i / g.mx) % g.my, z = i / (g.mx * g.my);
  int xm = wrapi(x - 1, g.mx), ym = wrapi(y - 1, g.my), zm = wrapi(z - 1, g.mz);
  const float* VX = v;
  const float* VY = v + g.N;
  const float* VZ = v + 2 * (size_t)g.N;
  div[i] = (VX[i] - VX[xm + g.mx * (y + g.my * z)]) * g.idx + (VY[i] - VY[x + g.mx * (ym + g.my * z)]) * g.idy +
           (VZ[i] - VZ[x + g.mx * (y + g.my * zm)]) * g.idz;
}

// Excess-mass fluid update: lap = coef L dv (seven-point staggered Laplacian per component,
// laplacianDeltaV, src/quasiNeutrallyBuoyantFunctions.cu:5294-5386) and v2 = al v + be v2 + ga dv
// (calculateVelocityAtHalfTimeStep / updateFluidQuasiNeutrallyBuoyantSemiImplicit).
FHD_BODY void body_mass_fluid(const MassFluidArgs& a, const Blk& b) {
  const GridDev& g = a.g;
  const size_t e = (size_t)b.x * blockDim.x + threadIdx.x;
  if (e >= 3 * (size_t)g.N) return;
  const int C = (int)(e / g.N);
  const int i = (int)(e - (size_t)C * g.N);
  const int x = i % g.mx, y = (i / g.mx) % g.my, z = i / (g.mx * g.my);
  const float* f = a.dv + (size_t)C * g.N;
  auto at = [&](int xx, int yy, int zz) { return f[wrapi(xx, g.mx) + g.mx * (wrapi(yy, g.my) + g.my * wrapi(zz, g.mz))]; };
  const float c0 = f[i];
  const float L = g.idx * g.idx * (at(x + 1, y, z) - 2.0f * c0 + at(x - 1, y, z)) +
                  g.idy * g.idy * (at(x, y + 1, z) - 2.0f * c0 + at(x, y - 1, z)) +
                  g.idz * g.idz * (at(x, y, z + 1) - 2.0f * c0 + at(x, y, z - 1));
  a.lap[e] = a.coef * L;
  if (a.v2) a.v2[e] = a.al * a.v[e] + a.be * a.v2[e] + a.ga * c0;
}
FHD_KERNEL_PAIR((), 256, k_mass_fluid, MassFluidArgs, body_mass_fluid(a, b))

void launch_mass_fluid(const MassFluidArgs& a, hipStream_t s) {
  launch(k_mass_fluid, k_mass_fluid_b, FAM_MASS_FLUID, dim3((unsigned)((3 * (size_t)a.g.N + 255) / 256)), 256, a, s);
}

// Normals of the shared generator, for parity tests: out[4 i + k] = draw(index i)[k].
__global__ void k_normals(Key key, int stream, int sub, int n, float* out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float v[4];
  draw_normals4(key, (uint32_t)i, (uint32_t)stream, (uint32_t)sub, v);
  for (int k = 0; k < 4; ++k) out[4 * i + k] = v[k];
}

FHD_BODY void body_zero_f(const FillArgs& a, const Blk& b) {
  const size_t i = (size_t)b.x * blockDim.x + threadIdx.x;
  if (i < a.n) a.p[i] = 0.0f;
}
FHD_KERNEL_PAIR((), 256, k_zero_f, FillArgs, body_zero_f(a, b))

void launch_normals(const Key& key, int stream, int sub, int n, float* out, hipStream_t s) {
  hipLaunchKernelGGL(k_normals, dim3((n + 255) / 256), dim3(256), 0, s, key, stream, sub, n, out);
}

void launch_zero_f(float* p, size_t n, hipStream_t s) {
  const FillArgs a{p, n};
  launch(k_zero_f, k_zero_f_b, FAM_ZERO, dim3((unsigned)((n + 255) / 256)), 256, a, s);
}

// Advances the device-side step counter that graph-replayed steps key their noise with.
FHD_BODY void body_advance_step(const StepArgs& a) {
  if (threadIdx.x == 0) *a.step += 1ull;
}
FHD_KERNEL_PAIR((), 64, k_advance_step, StepArgs, body_advance_step(a))
void launch_advance_step(unsigned long long* step, hipStream_t s) {
  const StepArgs a{step};
  launch(k_advance_step, k_advance_step_b, FAM_STEP, dim3(1), 64, a, s);
}

void launch_fluid_w(const FluidWArgs& a, hipStream_t s) {
  const int want = t_recorder && a.zchunk_b > 0 ? a.zchunk_b : a.zchunk;
  const int zc = want >= 4 ? 4 : want >= 2 ? 2 : 1;
  const dim3 grid((a.g.mx + TX - 1) / TX, (a.g.my + TY - 1) / TY, (a.g.mz + zc - 1) / zc);
  if (zc == 4) launch(k_fluid_w<4>, k_fluid_w_b<4>, FAM_FLUID_W, grid, 1024, a, s);
  else if (zc == 2) launch(k_fluid_w<2>, k_fluid_w_b<2>, FAM_FLUID_W, grid, 512, a, s);
  else launch(k_fluid_w<1>, k_fluid_w_b<1>, FAM_FLUID_W, grid, 256, a, s);
}

void launch_divergence(const GridDev& g, const float* v, float* div, hipStream_t s) {
  hipLaunchKernelGGL(k_divergence, dim3((g.N + 255) / 256), dim3(256), 0, s, g, v, div);
}

// Equal-time structure factor sample: acc[i] += |spec[i]|^2 in FP64 over the half spectrum of
// the three velocity components (the in-situ counterpart of the HydroGrid static structure
// factor that fluam's analysis hook feeds, src/hydroAnalysisIncompressible.cu:35-92).  The
// phase of the staggering shift drops out of |.|^2, so the plain transform of each component
// is used.  HBM-bound: 8 B read + 16 B read-modify-write per spectral entry.
__global__ __launch_bounds__(256) void k_sk_accum(const float2* __restrict__ spec, double* __restrict__ acc,
                                                 long long n) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const float2 v = spec[i];
    acc[i] += (double)v.x * (double)v.x + (double)v.y * (double)v.y;
  }
}
void launch_sk_accum(const float2* spec, double* acc, size_t n, hipStream_t s) {
  if (n == 0) return;
  long long blocks = ((long long)n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_sk_accum, dim3((unsigned)blocks), dim3(256), 0, s, spec, acc, (long long)n);
}

}  // namespace fhd
