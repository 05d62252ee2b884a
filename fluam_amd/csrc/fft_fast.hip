// fft_fast.hip -- size-specialised versions of the xy passes (see fft.hip for the algorithm).  Transform lengths, radix plans and LDS extents are template parameters, so every
// index division in the Stockham stages is by a constant and the register arrays are sized for
// the actual plane instead of the worst case.  Instantiated for xy planes mx x my with both
// lengths in {16, 24, 32, 48, 64} or mx = my in {96, 128}; other shapes use the generic kernels,
// which share the spectrum layout spec[c][ky][z][kx].
// The runtime-size and the size-specialised FFT kernels have to give the same bits (a replica runs
// on the one alone and on the other in a merged batch), so the compiler must not choose which
// products become fused multiply-adds: the fused ones are written out.
#pragma clang fp contract(off)
#include "fhd_device.h"
#include "fhd_kernels.h"
#include "fft_common.h"
#include "fft_stages.h"


namespace fhd {

// ---------------- pass A ----------------
FHD_KERNEL_PAIR((template <int MX, int MY, int NT, int PX, int PY>), NT, k_fftA, FftPass,
                body_fftA<MX, MY, NT, PX, PY, false>(a.f, a.in, a.spec, b, nullptr))

// ---------------- pass C: FFT along y (inverse) -> C2R along x -> out = alpha r + beta aux ----
template <int MX, int MY, int NT, int PX = 0, int PY = 0>
FHD_BODY void body_fftC(const FftArgs& a, const float2* __restrict__ spec, float* out,
                        const float* aux, float alpha, float beta, const Blk& b) {
  constexpr int H = MX / 2, P = H + 1;
  __shared__ float2 buf[MY * P];
  __shared__ float2 twx[MX];
  __shared__ float2 twy[MY];
  const int z = b.x, c = b.y, mz = a.g.mz;
  float2* src = const_cast<float2*>(spec) + (size_t)c * MY * mz * P + (size_t)z * P;
  ffft_modes<MY, P, NT, P, 1, true, plan_choice(MY, PY)>(buf, P, 1, twy, src, mz * P, [&] {
    for (int i = threadIdx.x; i < MX; i += NT) twx[i] = a.twx[i];
    for (int i = threadIdx.x; i < MY; i += NT) twy[i] = a.twy[i];
    __syncthreads();
  });
  constexpr int NP = H / 2 + 1;
  for (int e = threadIdx.x; e < MY * NP; e += NT) {
    const int y = e / NP, k = e - y * NP;
    float2* row = buf + y * P;
    const float2 Xk = row[k], Xh = row[H - k];
    const float2 wk = cconj(twx[k]);
    const float2 B = cconj(Xh);
    const float2 Zk = cadd(cadd(Xk, B), cmul_si(cmul(csub(Xk, B), wk), 1.0f));
    if (k != 0 && H - k != k) {
      const float2 B2 = cconj(Xk);
      const float2 wk2 = make_float2(-wk.x, wk.y);
      row[H - k] = cadd(cadd(Xh, B2), cmul_si(cmul(csub(Xh, B2), wk2), 1.0f));
    }
    row[k] = Zk;
  }
  __syncthreads();
  ffft<H, 1, NT, MY, 2, true, plan_choice(H, PX)>(buf, MY, P, twx);
  const size_t off = ((size_t)c * mz + z) * (size_t)(MX * MY);
  float4* dst = reinterpret_cast<float4*>(out + off);
  const float4* ax = aux ? reinterpret_cast<const float4*>(aux + off) : nullptr;
  constexpr int Q = MX / 4;
  constexpr int NS = (MY * Q + NT - 1) / NT;
  float4 q[NS];
  if (ax) {
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < MY * Q) q[k] = ax[e];
    }
  }
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    const int e = threadIdx.x + k * NT;
    if (e < MY * Q) {
      const int y = e / Q, x4 = e - y * Q;
      const float2 p0 = buf[y * P + 2 * x4], p1 = buf[y * P + 2 * x4 + 1];
      float4 r = make_float4(alpha * p0.x, alpha * p0.y, alpha * p1.x, alpha * p1.y);
      if (ax) {
        r.x = fmaf(beta, q[k].x, r.x);
        r.y = fmaf(beta, q[k].y, r.y);
        r.z = fmaf(beta, q[k].z, r.z);
        r.w = fmaf(beta, q[k].w, r.w);
      }
      dst[e] = r;
    }
  }
}
FHD_KERNEL_PAIR((template <int MX, int MY, int NT, int PX, int PY>), NT, k_fftC, FftPass,
                body_fftC<MX, MY, NT, PX, PY>(a.f, a.spec, a.out, a.aux, a.alpha, a.beta, b))

// ---------------- dispatch ----------------
template <int MX, int MY, int NT, int PX, int PY>
static void launch_AC_plan(const FftPass& x, int which, int mz, hipStream_t s) {
  // merged batches hold the smaller planes as runtime-size passes (merged_plane)
  BatchedFn ba = nullptr, bc = nullptr;
  if constexpr (MX > 64) {
    ba = k_fftA_b<MX, MY, NT, PX, PY>;
    bc = k_fftC_b<MX, MY, NT, PX, PY>;
  }
  if (which == 0) launch(k_fftA<MX, MY, NT, PX, PY>, ba, FAM_FFT_XY_FWD, dim3(mz, x.f.ncomp), NT, x, s);
  else launch(k_fftC<MX, MY, NT, PX, PY>, bc, FAM_FFT_XY_INV, dim3(mz, x.f.ncomp), NT, x, s);
}
// The radix plans of the x and y transforms (plan_choice indices, px + 3 py) are square_plan's and can
// be forced for 96 x 96 and 128 x 128 planes (128 x 128 also has 9: the register-transform kernels of
// fft128.hip); every other plane has plan 0.
template <int MX, int MY, int NT>
static void launch_AC_nt(const FftPass& x, int which, int mz, hipStream_t s) {
  if constexpr ((MX == 128 && MY == 128) || (MX == 96 && MY == 96)) {
    switch (which == 0 ? x.f.plan_xy : x.f.plan_xy_inv) {
      case 1: launch_AC_plan<MX, MY, NT, 1, 0>(x, which, mz, s); return;
      case 2: launch_AC_plan<MX, MY, NT, 2, 0>(x, which, mz, s); return;
      case 3: launch_AC_plan<MX, MY, NT, 0, 1>(x, which, mz, s); return;
      case 4: launch_AC_plan<MX, MY, NT, 1, 1>(x, which, mz, s); return;
      case 5: launch_AC_plan<MX, MY, NT, 2, 1>(x, which, mz, s); return;
      case 6: launch_AC_plan<MX, MY, NT, 0, 2>(x, which, mz, s); return;
      case 7: launch_AC_plan<MX, MY, NT, 1, 2>(x, which, mz, s); return;
      case 8: launch_AC_plan<MX, MY, NT, 2, 2>(x, which, mz, s); return;
      case 9:
        if constexpr (MX == 128) {
          launch_fft128_xy(x, which, mz, s);  // transforms in registers (fft128.hip)
          return;
        }
        break;
      default: break;
    }
  }
  launch_AC_plan<MX, MY, NT, 0, 0>(x, which, mz, s);
}
// Lanes per plane workgroup.  A single context's pass has only 3 mz plane workgroups, and more
// lanes per plane cover more of the plane load and store latency: 1024 from 64^2 up (128^3:
// 25.4 vs 26.1 / 27.3 us per pass with 512; 58-60 VGPRs, two workgroups per CU by LDS).  A
// batched dispatch already holds the planes of many contexts, and 96^2 planes pack better there as
// 512-lane workgroups.
template <int MX, int MY>
static bool launch_AC(const FftArgs& a, int which, const float* in, float2* spec, float* out, const float* aux,
                      float alpha, float beta, hipStream_t s) {
  const FftPass x{a, in, spec, out, aux, alpha, beta, 0};
  if constexpr (MX == 96) {
    if (t_recorder) {
      launch_AC_nt<MX, MY, 512>(x, which, a.g.mz, s);
      return true;
    }
  }
  launch_AC_nt<MX, MY, MX * MY >= 64 * 64 ? 1024 : 256>(x, which, a.g.mz, s);
  return true;
}

// Rectangular planes mx x my with both lengths in {16, 24, 32, 48, 64}.
template <int MX>
static bool launch_AC_rect(const FftArgs& a, int which, const float* in, float2* spec, float* out, const float* aux,
                           float alpha, float beta, hipStream_t s) {
  switch (a.g.my) {
    case 16: return launch_AC<MX, 16>(a, which, in, spec, out, aux, alpha, beta, s);
    case 24: return launch_AC<MX, 24>(a, which, in, spec, out, aux, alpha, beta, s);
    case 32: return launch_AC<MX, 32>(a, which, in, spec, out, aux, alpha, beta, s);
    case 48: return launch_AC<MX, 48>(a, which, in, spec, out, aux, alpha, beta, s);
    case 64: return launch_AC<MX, 64>(a, which, in, spec, out, aux, alpha, beta, s);
    default: return false;
  }
}

static bool fast_AC(const FftArgs& a, int which, const float* in, float2* spec, float* out, const float* aux,
                    float alpha, float beta, hipStream_t s) {
  if (a.g.mx == a.g.my) {
    if (a.g.mx == 96) return launch_AC<96, 96>(a, which, in, spec, out, aux, alpha, beta, s);
    if (a.g.mx == 128) return launch_AC<128, 128>(a, which, in, spec, out, aux, alpha, beta, s);
  }
  switch (a.g.mx) {
    case 16: return launch_AC_rect<16>(a, which, in, spec, out, aux, alpha, beta, s);
    case 24: return launch_AC_rect<24>(a, which, in, spec, out, aux, alpha, beta, s);
    case 32: return launch_AC_rect<32>(a, which, in, spec, out, aux, alpha, beta, s);
    case 48: return launch_AC_rect<48>(a, which, in, spec, out, aux, alpha, beta, s);
    case 64: return launch_AC_rect<64>(a, which, in, spec, out, aux, alpha, beta, s);
    default: return false;
  }
}

bool fast_fft_xy_fwd(const FftArgs& a, const float* in, float2* spec, hipStream_t s) {
  return fast_AC(a, 0, in, spec, nullptr, nullptr, 0.0f, 0.0f, s);
}
bool fast_fft_spread_xy_fwd(const FftArgs& a, const float* in, const PlaneSrc& src, float2* spec, hipStream_t s) {
  const FftSpread x{{a, in, spec, nullptr, nullptr, 0.0f, 0.0f, 0}, src};
  switch (a.g.mx) {
#define FHD_SPREAD(mx) case mx: return launch_spread_rect<mx>(x, s)
    FHD_SPREAD(16);
    FHD_SPREAD(24);
    FHD_SPREAD(32);
    FHD_SPREAD(48);
    FHD_SPREAD(64);
    FHD_SPREAD(96);
    FHD_SPREAD(128);
#undef FHD_SPREAD
    default: return false;
  }
}
bool fast_fft_xy_inv(const FftArgs& a, const float2* spec, float* out, const float* aux, float alpha, float beta,
                     hipStream_t s) {
  return fast_AC(a, 1, nullptr, const_cast<float2*>(spec), out, aux, alpha, beta, s);
}

}  // namespace fhd
