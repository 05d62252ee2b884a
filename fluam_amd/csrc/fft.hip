// fft.hip -- batched, LDS-staged mixed-radix Stockham 3D real FFT for gfx950, with the
// Fourier-space viscous / Stokes solve fused into the z-pencil pass: the runtime-size kernels,
// for every grid whose lengths are 2^a 3^b (fft_fast.hip holds the size-specialised ones).
//
// Replaces the cufftExecZ2Z calls + kernelShift + kernelUpdateV* chain of fluam
// (src/runSchemeIncompressible.cu:111-138, src/runSchemeStokesLimit.cu:198-259,
//  src/realToComplex.cu:263-303, src/kernelUpdateVIncompressible.cu:21-72,
//  src/stokesLimitFunctions.cu:2399-2451).
//
// Three passes per solve, each one read + one write of the field:
//   A  xy-forward : one workgroup per (z-plane, component): real plane -> R2C along x (an
//                   mx/2-point complex FFT plus the even/odd split) -> complex FFT along y.
//   B  z-solve    : one workgroup per (ky, tile of kx) for all three components: FFT along z,
//                   staggering shifts + projection + viscous / Stokes operator, inverse FFT.
//   C  xy-inverse : inverse of A, with an epilogue that blends the result with another field.
// Half-spectrum layout in HBM: spec[c][ky][z][kx], kx in [0, mx/2], row pitch P = mx/2 + 1, so
// a pass-B tile (fixed ky, a run of kx, every z) is one compact block of rows.
//
// The workgroup is sized to its data: 256, 512 or 1024 lanes for up to 2112, 4224 or 8448 complex
// elements in LDS, so a lane never holds more than 9 elements (64 VGPRs, the CU full of waves in
// every class), every load of a lane is in flight at once, and the butterflies a lane may hold in
// a stage are a constant per radix.  The radices go up to 16 (at most three stages for any length
// up to 256), the divisions by runtime extents are multiplications by host-made reciprocals, and the
// y transform's last stage (the inverse's first) works on the modes in global memory.  Bound by LDS
// and barrier latency, like the size-specialised passes.  Per launch (HIP events, which add about
// 4 us), with 256 lanes, radices up to 8 and a load-wait-store loop per element at first, then with
// every stage through LDS, and now: 108 x 54 x 72 forward 33.6, 13.5, 12.8, inverse 34.8, 13.0, 12.9 us;
// 128 x 64 x 32 inverse 13.8, now 13.3, 96 x 48 x 64 13.1, now 12.5.  Where a size-specialised instance
// exists it stays ahead (128^3 forward and inverse 20.7 / 19.2 against 23.6 / 23.2 us; 64^3 9.6 / 8.9
// against 13.8 / 13.3), so those shapes keep it; the z pass is fft_z.hip's but for a few lengths.
// The runtime-size and the size-specialised FFT kernels have to give the same bits (a replica runs
// on the one alone and on the other in a merged batch), so the compiler must not choose which
// products become fused multiply-adds: the fused ones are written out.
#pragma clang fp contract(off)
#include "fhd_device.h"
#include "fhd_kernels.h"
#include "fft_common.h"
#include "plane_spread.h"

namespace fhd {

constexpr int kClassElems[3] = {2112, 4224, 8448};  // complex elements of a 256-, 512-, 1024-lane workgroup
constexpr int kPerLane = 9;                          // ceil(8448 / 1024)
constexpr int kmax_for(int R) { return (2112 + R * 256 - 1) / (R * 256); }

// Lines of one transform in LDS: line l at l * ls, element stride es; ml = fast_div's reciprocal
// of the line count.
struct Lines {
  int count;
  uint32_t ml;
  int ls, es;
};

// One radix-R Stockham stage over all lines (Govindaraju et al., SC'08 formulation):
// butterfly j of a line reads x[j + r n/R], twiddles by w^{(j mod Ns) r}, w = e^{-2 pi i/(Ns R)},
// and writes to (j / Ns) Ns R + (j mod Ns) + r Ns.  In place: every lane reads its butterflies
// into registers, the workgroup synchronises, then writes.  Consecutive lanes take butterfly j of
// consecutive lines, which lie an odd number of elements apart or next to each other, so the
// lanes of a wave use different LDS banks and share one twiddle.  INV: the adjoint stage of the
// inverse transform.  GIO: the modes lie in global memory, element e of line l at m.g[l + e m.gs], and
// a transform of two stages runs the first one in place (all as in fft_stages.h).
struct Modes {
  float2* g;
  int gs;
};
struct NotReady {
  FHD_DEV void operator()() const {}
};
template <int R, int NT, bool INV, bool GIO, class Ready>
FHD_DEV void stockham_stage(float2* buf, const Lines& ln, const LinePlan& p, int Ns, uint32_t mns, const float2* tw,
                            int twmul, const Modes& m, const Ready& ready) {
  constexpr int KMAX = kmax_for(R);
  constexpr float s = INV ? 1.0f : -1.0f;
  const int n = p.n, nbl = n / R;
  const int total = ln.count * nbl;
  const int twstep = n / (Ns * R) * twmul;
  const bool last = Ns * R == n, glob = GIO && last, inpl = GIO && p.nst == 2;
  // opaque to the compiler, which otherwise hoists the lane indices of every radix's stage out of
  // the stage loop and spills them (150 VGPRs)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int in_j = inpl && last ? R : 1, in_r = inpl && last ? ln.es : nbl * ln.es;
  const int out_r = inpl && !last ? in_r : Ns * ln.es;
  float2 v[KMAX][R];
  int to[KMAX], t1[KMAX];  // first element of the butterfly's outputs (-1: none), twiddle step
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int b = tid + k * NT;
    to[k] = -1;
    if (b < total) {
      const int j = fast_div(b, ln.ml), l = b - j * ln.count;
      const int base = l * ln.ls;
      const int jn = Ns == 1 ? j : fast_div(j, mns), kk = j - jn * Ns;
      t1[k] = kk * twstep;
      const int in = base + j * in_j * ln.es, out = inpl && !last ? in : base + (jn * Ns * R + kk) * ln.es;
      if (GIO && INV && last) {
        int at = l + j * m.gs;
#pragma unroll
        for (int r = 0; r < R; ++r, at += nbl * m.gs) v[k][r] = m.g[at];
      } else {
        int at = INV ? out : in;
        const int step = INV ? out_r : in_r;
#pragma unroll
        for (int r = 0; r < R; ++r, at += step) v[k][r] = buf[at];
      }
      to[k] = GIO && !INV && last ? l + j * m.gs : INV ? in : out;
    }
  }
  if (GIO && INV && last) ready();
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    if (to[k] >= 0) {
      if (!INV && Ns > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) v[k][r] = cmul(v[k][r], tw[r * t1[k]]);
      }
      Dft<R>::run(v[k], s);
      if (INV && Ns > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) v[k][r] = cmul(v[k][r], cconj(tw[r * t1[k]]));
      }
    }
  }
  if (!last && !inpl) __syncthreads();
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    if (to[k] >= 0) {
      int at = to[k];
      if (GIO && !INV && last) {
#pragma unroll
        for (int r = 0; r < R; ++r, at += nbl * m.gs) m.g[at] = v[k][r];
      } else {
        const int step = INV ? in_r : out_r;
#pragma unroll
        for (int r = 0; r < R; ++r, at += step) buf[at] = v[k][r];
      }
    }
  }
  if (!glob || INV) __syncthreads();
}

// Full FFT of every line: at most three stages, undone in reverse order by the inverse.
template <int NT, bool INV, bool GIO, class Ready>
FHD_DEV void lds_fft(float2* buf, const Lines& ln, const LinePlan& p, const float2* tw, int twmul, const Modes& m,
                     const Ready& ready) {
  int Ns = INV ? p.n : 1;
  for (int k = 0; k < p.nst; ++k) {
    const int st = INV ? p.nst - 1 - k : k;
    const int R = p.radix[st];
    const uint32_t mns = p.mns[st];
    if (INV) Ns /= R;
    switch (R) {
#define FHD_STAGE(r) stockham_stage<r, NT, INV, GIO>(buf, ln, p, Ns, mns, tw, twmul, m, ready); break
      case 16: FHD_STAGE(16);
      case 9: FHD_STAGE(9);
      case 8: FHD_STAGE(8);
      case 6: FHD_STAGE(6);
      case 4: FHD_STAGE(4);
      case 3: FHD_STAGE(3);
      default: FHD_STAGE(2);
#undef FHD_STAGE
    }
    if (!INV) Ns *= R;
  }
}
template <int NT, bool INV>
FHD_DEV void lds_fft(float2* buf, const Lines& ln, const LinePlan& p, const float2* tw, int twmul) {
  lds_fft<NT, INV, false>(buf, ln, p, tw, twmul, Modes{nullptr, 0}, NotReady{});
}

// ---------------------------------------------------------------------------------------
// Pass A: real plane -> half spectrum along x -> FFT along y.  LDS rows of PS = P | 1 elements
// (odd, so that the rows of an x stage start in different banks).
// ---------------------------------------------------------------------------------------
// SP: the plane is the sources' spread field (plane_spread.h) plus `in` (null: none).
template <int NT, int ELEMS, bool SP>
FHD_BODY void body_fft_xy_fwd(const FftArgs& a, const float* __restrict__ in, float2* __restrict__ spec,
                              const Blk& b, const PlaneSrc* src_sp) {
  __shared__ __align__(16) float2 buf[ELEMS];  // plane_spread clears it 16 bytes at a time
  // the twiddles of both transforms; before they are stored, plane_spread's lists (whose scales lie beyond
  // the twiddles)
  constexpr int kTw = 2 * kMaxFftLen * sizeof(float2);
  static_assert(offsetof(PlaneLds, scale) >= kTw, "the scales are read while the twiddles are stored");
  __shared__ __align__(16) unsigned char side[SP && (int)sizeof(PlaneLds) > kTw ? (int)sizeof(PlaneLds) : kTw];
  float2* const twx = reinterpret_cast<float2*>(side);
  float2* const twy = twx + kMaxFftLen;
  // with spreading, the three components and the neighbouring planes, which read the same sources,
  // are kept on one XCD
  const int item = SP ? xcd_item(b.x + b.nx * b.y, b.nx * b.ny) : 0;
  const int z = SP ? item / b.ny : b.x, c = SP ? item - z * b.ny : b.y;
  const int mx = a.g.mx, my = a.g.my, mz = a.g.mz, P = a.g.P, h = mx / 2, PS = P | 1;
  const float2* src = reinterpret_cast<const float2*>(in + ((size_t)c * mz + z) * (size_t)my * mx);
  if constexpr (!SP) {
    float2 v[kPerLane];
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < h * my) v[k] = src[e];
    }
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < h * my) buf[e + fast_div(e, a.mdh) * (PS - h)] = v[k];
    }
  } else {
    PlaneLds& pl = *reinterpret_cast<PlaneLds*>(side);
    // the integers become the plane in place; between two sweeps the first sums wait in this
    // workgroup's own rows of the spectrum (at least mx floats each), written later
    float* part = reinterpret_cast<float*>(spec + ((size_t)c * my * mz + z) * P);
    int* acc = reinterpret_cast<int*>(buf);
    const bool more = plane_spread<NT, false>(acc, 2 * my * PS, 2 * PS, a.g, *src_sp, z, c, pl);
    const PlaneUnit unit = plane_unit(pl, *src_sp, a.g);
    if (more) {
      for (int e = threadIdx.x; e < h * my; e += NT) {
        const int y = fast_div(e, a.mdh), x = e - y * h;
        const int2 q = *reinterpret_cast<const int2*>(&buf[x + y * PS]);
        const float f = unit.at(pl, 2 * x, y);
        float* at = part + (size_t)y * mz * 2 * P + 2 * x;
        at[0] = f * (float)q.x;
        at[1] = f * (float)q.y;
      }
      __syncthreads();
      plane_spread<NT, true>(acc, 2 * my * PS, 2 * PS, a.g, *src_sp, z, c, pl);
    }
    for (int e = threadIdx.x; e < h * my; e += NT) {
      const int y = fast_div(e, a.mdh), x = e - y * h;
      float2* at_e = &buf[x + y * PS];
      const int2 q = *reinterpret_cast<const int2*>(at_e);
      const float f = unit.at(pl, 2 * x, y) * (more ? unit.rest : 1.0f);
      float2 r = make_float2(f * (float)q.x, f * (float)q.y);
      if (more) {
        const float* at = part + (size_t)y * mz * 2 * P + 2 * x;
        r = cadd(r, make_float2(at[0], at[1]));
      }
      *at_e = in ? cadd(r, src[e]) : r;
    }
  }
  for (int i = threadIdx.x; i < mx; i += NT) twx[i] = a.twx[i];
  for (int i = threadIdx.x; i < my; i += NT) twy[i] = a.twy[i];
  __syncthreads();
  // x: h-point complex FFT of the even/odd-packed rows
  lds_fft<NT, false>(buf, Lines{my, a.mdy, PS, 1}, a.lx, twx, 2);
  // even/odd split: X[k] = E + w^k O, X[h-k] = conj(E - w^k O)
  const int npair = h / 2 + 1;
  for (int e = threadIdx.x; e < my * npair; e += NT) {
    const int k = fast_div(e, a.mdy), y = e - k * my;
    float2* row = buf + y * PS;
    const float2 A = row[k];
    const float2 B = cconj(row[k == 0 ? 0 : h - k]);
    const float2 E = cscale(cadd(A, B), 0.5f);
    const float2 D = csub(A, B);
    const float2 O = make_float2(0.5f * D.y, -0.5f * D.x);  // (A - B) / (2i)
    const float2 wO = cmul(twx[k], O);
    if (k == 0) {
      row[0] = make_float2(E.x + O.x, 0.0f);
      row[h] = make_float2(E.x - O.x, 0.0f);
    } else {
      row[k] = cadd(E, wO);
      if (h - k != k) row[h - k] = cconj(csub(E, wO));
    }
  }
  __syncthreads();
  // y: columns kx = 0..P-1
  float2* dst = spec + ((size_t)c * my * mz + z) * P;
  if (my > 1) {
    lds_fft<NT, false, true>(buf, Lines{P, a.mdp, 1, PS}, a.ly, twy, 1, Modes{dst, mz * P}, NotReady{});
  } else if ((int)threadIdx.x < P) {
    dst[threadIdx.x] = buf[threadIdx.x];
  }
}
FHD_KERNEL_PAIR_OCC((template <int NT, int ELEMS>), NT, 8, k_fft_xy_fwd, FftPass,
                    body_fft_xy_fwd<NT, ELEMS, false>(a.f, a.in, a.spec, b, nullptr))
FHD_KERNEL_PAIR_OCC((template <int NT, int ELEMS>), NT, 8, k_fft_spread_xy_fwd, FftSpread,
                    body_fft_xy_fwd<NT, ELEMS, true>(a.p.f, a.p.in, a.p.spec, b, &a.s))

// ---------------------------------------------------------------------------------------
// Pass B: FFT along z, Fourier-space operator, inverse FFT along z, for all three components.
// The P columns of a ky row are cut into b.nx tiles whose widths differ by at most one; a tile's
// columns lie on a grid of T (the widest tile) per component, lines of LS = mz | 1 elements.
// ---------------------------------------------------------------------------------------
template <int NT, int ELEMS>
FHD_BODY void body_fft_z_solve(const FftArgs& a, float2* __restrict__ spec, int T, const Blk& b) {
  __shared__ float2 buf[ELEMS];
  __shared__ float2 twz[kMaxFftLen], ezs[kMaxFftLen];
  __shared__ float gzs[kMaxFftLen];
  const int my = a.g.my, mz = a.g.mz, P = a.g.P, LS = mz | 1;
  // neighbouring column tiles share the 128-byte lines of each z row: keep them on one XCD
  const int item = xcd_item(b.x + b.nx * b.y, b.nx * b.ny);
  const int ky = item / b.nx, tile = item - ky * b.nx;
  const int wide = P / b.nx, rem = P - wide * b.nx;
  const int kx0 = tile * wide + min(tile, rem), w = wide + (tile < rem ? 1 : 0);
  const uint32_t mt = fast_div_magic(T), mlz = fast_div_magic(mz);
  const int tot = a.ncomp * mz * T;
  const size_t cstride = (size_t)my * mz * P;
  float2* base = spec + (size_t)ky * mz * P + kx0;
  float2 v[kPerLane];
#pragma unroll
  for (int k = 0; k < kPerLane; ++k) {
    const int e = threadIdx.x + k * NT;
    const int r = fast_div(e, mt), t = e - r * T, c = fast_div(r, mlz), z = r - c * mz;
    if (e < tot && t < w) v[k] = base[c * cstride + z * P + t];
  }
  for (int i = threadIdx.x; i < mz; i += NT) {
    twz[i] = a.twz[i];
    ezs[i] = a.ez[i];
    gzs[i] = a.gz[i];
  }
#pragma unroll
  for (int k = 0; k < kPerLane; ++k) {
    const int e = threadIdx.x + k * NT;
    const int r = fast_div(e, mt), t = e - r * T, c = fast_div(r, mlz), z = r - c * mz;
    if (e < tot && t < w) buf[(c * T + t) * LS + z] = v[k];
  }
  __syncthreads();
  const Lines zl{a.ncomp * T, fast_div_magic(a.ncomp * T), LS, 1};
  if (a.zmode != 2) lds_fft<NT, false>(buf, zl, a.lz, twz, 1);
  if (a.zmode == 0) {
    // Fourier-space operator in the staggered (shifted) basis; 1/N normalisation folded in.
    const float gy = a.gy[ky];
    const float2 ey = a.ey[ky];
    const Key key = a.knoise ? resolve_key(a.key) : a.key;
    for (int e = threadIdx.x; e < mz * w; e += NT) {
      const int t = fast_div(e, mlz), z = e - t * mz, kx = kx0 + t;
      const float gx = a.gx[kx];
      const float2 ex = a.ex[kx];
      const float gz = gzs[z];
      const float2 ez = ezs[z];
      const int i0 = t * LS + z, i1 = i0 + T * LS, i2 = i1 + T * LS;
      float2 b0 = buf[i0], b1 = buf[i1], b2 = buf[i2];
      solve_mode(a, key, kx, ky, z, gx, gy, gz, ex, ey, ez, b0, b1, b2);
      buf[i0] = b0;
      buf[i1] = b1;
      buf[i2] = b2;
    }
    __syncthreads();
  }
  if (a.zmode != 1) lds_fft<NT, true>(buf, zl, a.lz, twz, 1);
  // the lane index, opaque to the compiler: the store indices are recomputed here rather than
  // kept live in registers from the loads through both transforms
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
#pragma unroll
  for (int k = 0; k < kPerLane; ++k) {
    const int e = tid + k * NT;
    const int r = fast_div(e, mt), t = e - r * T, c = fast_div(r, mlz), z = r - c * mz;
    if (e < tot && t < w) base[c * cstride + z * P + t] = buf[(c * T + t) * LS + z];
  }
}
FHD_KERNEL_PAIR_OCC((template <int NT, int ELEMS>), NT, 8, k_fft_z_solve, FftPass,
                    body_fft_z_solve<NT, ELEMS>(a.f, a.spec, a.T, b))

// ---------------------------------------------------------------------------------------
// Pass C: inverse FFT along y, C2R along x; out = alpha * result + beta * aux.
// ---------------------------------------------------------------------------------------
template <int NT, int ELEMS>
FHD_BODY void body_fft_xy_inv(const FftArgs& a, const float2* __restrict__ spec, float* out,
                              const float* aux, float alpha, float beta, const Blk& b) {
  __shared__ float2 buf[ELEMS];
  __shared__ float2 twx[kMaxFftLen];
  __shared__ float2 twy[kMaxFftLen];
  const int z = b.x, c = b.y;
  const int mx = a.g.mx, my = a.g.my, mz = a.g.mz, P = a.g.P, h = mx / 2, PS = P | 1;
  float2* src = const_cast<float2*>(spec) + ((size_t)c * my * mz + z) * P;
  const auto tables = [&] {
    for (int i = threadIdx.x; i < mx; i += NT) twx[i] = a.twx[i];
    for (int i = threadIdx.x; i < my; i += NT) twy[i] = a.twy[i];
    __syncthreads();
  };
  if (my > 1) {
    lds_fft<NT, true, true>(buf, Lines{P, a.mdp, 1, PS}, a.ly, twy, 1, Modes{src, mz * P}, tables);
  } else {
    if ((int)threadIdx.x < P) buf[threadIdx.x] = src[threadIdx.x];
    tables();
  }
  // C2R packing: Z[k] = (X[k] + conj X[h-k]) + i (X[k] - conj X[h-k]) e^{+2 pi i k / mx}
  const int npair = h / 2 + 1;
  for (int e = threadIdx.x; e < my * npair; e += NT) {
    const int k = fast_div(e, a.mdy), y = e - k * my;
    float2* row = buf + y * PS;
    const float2 Xk = row[k], Xh = row[h - k];
    const float2 wk = cconj(twx[k]);  // e^{+2 pi i k / mx}
    const float2 B = cconj(Xh);
    const float2 Zk = cadd(cadd(Xk, B), cmul_si(cmul(csub(Xk, B), wk), 1.0f));
    if (k != 0 && h - k != k) {
      const float2 B2 = cconj(Xk);
      const float2 wk2 = make_float2(-wk.x, wk.y);  // e^{+2 pi i (h-k)/mx} = -conj(e^{+2 pi i k/mx})
      row[h - k] = cadd(cadd(Xh, B2), cmul_si(cmul(csub(Xh, B2), wk2), 1.0f));
    }
    row[k] = Zk;
  }
  __syncthreads();
  lds_fft<NT, true>(buf, Lines{my, a.mdy, PS, 1}, a.lx, twx, 2);
  const size_t off = ((size_t)c * mz + z) * (size_t)my * mx;
  float2* dst = reinterpret_cast<float2*>(out + off);
  const float2* ax = reinterpret_cast<const float2*>(aux + off);
  float2 q[kPerLane];
  if (aux) {
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < h * my) q[k] = ax[e];
    }
  }
#pragma unroll
  for (int k = 0; k < kPerLane; ++k) {
    const int e = threadIdx.x + k * NT;
    if (e < h * my) {
      const int y = fast_div(e, a.mdh);
      const float2 p = buf[e + y * (PS - h)];
      float2 r = make_float2(alpha * p.x, alpha * p.y);
      if (aux) {
        r.x = fmaf(beta, q[k].x, r.x);
        r.y = fmaf(beta, q[k].y, r.y);
      }
      dst[e] = r;
    }
  }
}
FHD_KERNEL_PAIR_OCC((template <int NT, int ELEMS>), NT, 8, k_fft_xy_inv, FftPass,
                    body_fft_xy_inv<NT, ELEMS>(a.f, a.spec, a.out, a.aux, a.alpha, a.beta, b))

// Workgroup class of a pass that holds `elems` complex elements.
static int lds_class(int elems) { return elems <= kClassElems[0] ? 0 : elems <= kClassElems[1] ? 1 : 2; }

#define FHD_LAUNCH_CLASS(cls, kern, fam, grid, x, s)                                                     \
  do {                                                                                                   \
    if ((cls) == 0) launch(kern<256, kClassElems[0]>, kern##_b<256, kClassElems[0]>, fam, grid, 256, x, s); \
    else if ((cls) == 1) launch(kern<512, kClassElems[1]>, kern##_b<512, kClassElems[1]>, fam, grid, 512, x, s); \
    else launch(kern<1024, kClassElems[2]>, kern##_b<1024, kClassElems[2]>, fam, grid, 1024, x, s);      \
  } while (0)

// A merged batch takes the runtime-size passes also where size-specialised ones exist (planes with
// edges up to 64): its replicas' shapes then share one dispatch per workgroup class instead of one
// per shape (32 boxes with edges 16-64: 22 dispatches of a few planes each per pass and round, four
// at a time).
static bool merged_plane(const FftArgs& a) { return t_recorder && fast_edge(a.g.mx) && fast_edge(a.g.my); }

void launch_fft_xy_fwd(const FftArgs& a, const float* in, float2* spec, hipStream_t s) {
  if (!a.generic && !merged_plane(a) && fast_fft_xy_fwd(a, in, spec, s)) return;
  const FftPass x{a, in, spec, nullptr, nullptr, 0.0f, 0.0f, 0};
  FHD_LAUNCH_CLASS(lds_class(a.g.my * (a.g.P | 1)), k_fft_xy_fwd, FAM_FFT_XY_FWD, dim3(a.g.mz, a.ncomp), x, s);
}
void launch_fft_spread_xy_fwd(const FftArgs& a, const float* in, const PlaneSrc& src, float2* spec, hipStream_t s) {
  if (!a.generic && !merged_plane(a) && fast_fft_spread_xy_fwd(a, in, src, spec, s)) return;
  const FftSpread x{{a, in, spec, nullptr, nullptr, 0.0f, 0.0f, 0}, src};
  FHD_LAUNCH_CLASS(lds_class(a.g.my * (a.g.P | 1)), k_fft_spread_xy_fwd, FAM_FFT_XY_FWD, dim3(a.g.mz, a.ncomp), x, s);
}
// Lengths without an instance in fft_z.hip, or all of them when the runtime-size kernels are forced.
// Columns per workgroup: the schedule's tile, as far as the largest class holds it.
int z_columns(const FftArgs& a, int want) {
  const int fast = a.generic ? 0 : fast_z_columns(a.g.mz, want);
  const int most = kClassElems[2] / (3 * (a.g.mz | 1));  // >= 10: mz is at most 256
  return fast ? fast : want < most ? want : most;
}
void launch_fft_z_solve(const FftArgs& a, float2* spec, hipStream_t s) {
  if (!a.generic && fast_fft_z_solve(a, spec, s)) return;
  const int LS = a.g.mz | 1, want = z_columns(a, a.btile);
  const int ntile = (a.g.P + want - 1) / want, T = (a.g.P + ntile - 1) / ntile;
  const FftPass x{a, nullptr, spec, nullptr, nullptr, 0.0f, 0.0f, T};
  FHD_LAUNCH_CLASS(lds_class(3 * T * LS), k_fft_z_solve, FAM_FFT_Z, dim3(ntile, a.g.my), x, s);
}
void launch_fft_xy_inv(const FftArgs& a, const float2* spec, float* out, const float* aux, float alpha, float beta,
                       hipStream_t s) {
  if (!a.generic && !merged_plane(a) && fast_fft_xy_inv(a, spec, out, aux, alpha, beta, s)) return;
  const FftPass x{a, nullptr, const_cast<float2*>(spec), out, aux, alpha, beta, 0};
  FHD_LAUNCH_CLASS(lds_class(a.g.my * (a.g.P | 1)), k_fft_xy_inv, FAM_FFT_XY_INV, dim3(a.g.mz, a.ncomp), x, s);
}

}  // namespace fhd
