// fft_stages.h -- the Stockham stages and the forward xy pass of the size-specialised FFT kernels,
// shared by the plain passes (fft_fast.hip) and the passes with spreading (fft_spread.hip).
// Bound by LDS crossings and barriers: a plane crosses LDS ten times with six barriers.  Twelve and
// ten, with every stage written, waited for and read back on both sides, took 20.0 us per inverse
// launch at 128^3 (HIP events, which add about 4 us; now 18.3), 14.7 at 96^3 (14.1); 100 steps of
// 128^3 Stokes 22.8 ms (now 22.0).
#pragma once
#include "fhd_device.h"
#include "fhd_kernels.h"
#include "fft_common.h"
#include "plane_spread.h"

namespace fhd {

// One radix-R Stockham stage, lines l = 0..lines-1 (lines <= MAXL) at base l * LS, element
// stride ES.  Consecutive lanes take butterfly j of consecutive lines: the lines are either
// adjacent elements (ES > 1, LS = 1) or an odd number of elements apart (ES = 1), so the lanes
// of a wave read and write different LDS banks in every stage, and share one twiddle.  (Taking
// consecutive butterflies of one line instead makes the writes of the early stages R-way bank
// conflicts.)
// INV: the stage of the inverse transform, which undoes the forward stages in reverse order (reads
// where the forward stage writes, twiddles after the butterfly, writes where it reads).  The
// inverse is then the exact adjoint of the forward transform with the table's rounded twiddles, so
// their phase errors cancel over the round trip of a solve instead of adding up over the steps.
// The last stage (the inverse's first) reads and writes the same elements, so nothing waits between.
// GIO: it leaves LDS out on the side of the modes, which lie in global memory (`g`: element e of line
// l at g[l + e gs]; of consecutive lines in consecutive words).  A transform of two stages then also
// runs its first one in place: element j R1 + r stays at j + r R2, so the second stage's butterfly j
// finds its elements at j R2 + r.  `ready` is called once the global loads are under way and ends with
// a barrier.
template <int N, int R, int NS, int ES, int NT, int MAXL, int TWM, bool INV, bool GIO, bool INPL, class Ready>
FHD_DEV void fstage(float2* buf, int lines, int LS, const float2* tw, float2* g, int gs, const Ready& ready) {
  constexpr int NBL = N / R;
  constexpr int KMAX = (MAXL * NBL + NT - 1) / NT;
  constexpr int STRIDE = N / (NS * R);
  constexpr bool LAST = NS * R == N, GLOB = GIO && LAST;
  constexpr float s = INV ? 1.0f : -1.0f;
  // elements of butterfly j on the input side of the forward stage (NBL apart) and on its output side
  // (NS apart in the sub-transform's block)
  constexpr int IN_J = INPL && LAST ? R : 1, IN_R = INPL && LAST ? 1 : NBL;
  constexpr bool OUT_IN = INPL && !LAST;
  const auto in_at = [&](int j) { return j * IN_J; };
  const auto out_at = [&](int j) { return OUT_IN ? in_at(j) : (j / NS) * NS * R + j % NS; };
  constexpr int OUT_R = OUT_IN ? IN_R : NS;
  float2 v[KMAX][R];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int b = threadIdx.x + k * NT;
    const int j = b / MAXL, l = b - j * MAXL;
    if (j < NBL && l < lines) {
      const int base = l * LS + (INV ? out_at(j) : in_at(j)) * ES;
#pragma unroll
      for (int r = 0; r < R; ++r) v[k][r] = GLOB && INV ? g[l + (j + r * NBL) * gs] : buf[base + r * (INV ? OUT_R : IN_R) * ES];
    }
  }
  if (GLOB && INV) ready();
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int b = threadIdx.x + k * NT;
    const int j = b / MAXL, l = b - j * MAXL;
    if (j < NBL && l < lines) {
      const int kk = j % NS;
      if (!INV && NS > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) v[k][r] = cmul(v[k][r], tw[(kk * r * STRIDE) * TWM]);
      }
      Dft<R>::run(v[k], s);
      if (INV && NS > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) v[k][r] = cmul(v[k][r], cconj(tw[(kk * r * STRIDE) * TWM]));
      }
    }
  }
  if (!LAST && !INPL) __syncthreads();
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int b = threadIdx.x + k * NT;
    const int j = b / MAXL, l = b - j * MAXL;
    if (j < NBL && l < lines) {
      const int base = l * LS + (INV ? in_at(j) : out_at(j)) * ES;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (GLOB && !INV) g[l + (j + r * NBL) * gs] = v[k][r];
        else buf[base + r * (INV ? IN_R : OUT_R) * ES] = v[k][r];
      }
    }
  }
  if (!GLOB || INV) __syncthreads();
}

struct NotReady {
  FHD_DEV void operator()() const {}
};
constexpr int plan_stages(uint32_t plan, int n) {
  int st = 0;
  for (int done = 1; done < n; ++st) done *= plan_at(plan, n, st);
  return st;
}

template <int N, int ST, int NS, int ES, int NT, int MAXL, int TWM, uint32_t PLAN, bool INV, bool GIO, class Ready>
struct FStages {
  static FHD_DEV void run(float2* buf, int lines, int LS, const float2* tw, float2* g, int gs, const Ready& ready) {
    constexpr int R = NS >= N ? 1 : plan_at(PLAN, N, ST);
    constexpr bool INPL = GIO && plan_stages(PLAN, N) == 2;
    if constexpr (R > 1) {
      if constexpr (!INV) fstage<N, R, NS, ES, NT, MAXL, TWM, INV, GIO, INPL>(buf, lines, LS, tw, g, gs, ready);
      FStages<N, ST + 1, NS * R, ES, NT, MAXL, TWM, PLAN, INV, GIO, Ready>::run(buf, lines, LS, tw, g, gs, ready);
      if constexpr (INV) fstage<N, R, NS, ES, NT, MAXL, TWM, INV, GIO, INPL>(buf, lines, LS, tw, g, gs, ready);
    }
  }
};

template <int N, int ES, int NT, int MAXL, int TWM, bool INV, uint32_t PLAN>
FHD_DEV void ffft(float2* buf, int lines, int LS, const float2* tw) {
  FStages<N, 0, 1, ES, NT, MAXL, TWM, PLAN, INV, false, NotReady>::run(buf, lines, LS, tw, nullptr, 0, NotReady{});
}
// The same with the modes in global memory (fstage's GIO).
template <int N, int ES, int NT, int MAXL, int TWM, bool INV, uint32_t PLAN, class Ready = NotReady>
FHD_DEV void ffft_modes(float2* buf, int lines, int LS, const float2* tw, float2* g, int gs, const Ready& ready = Ready{}) {
  FStages<N, 0, 1, ES, NT, MAXL, TWM, PLAN, INV, true, Ready>::run(buf, lines, LS, tw, g, gs, ready);
}

// ---------------- pass A: real plane -> half spectrum (x) -> FFT along y ----------------
// SP: the plane is the sources' spread field (plane_spread.h) plus `in` (null: none).
template <int MX, int MY, int NT, int PX, int PY, bool SP>
FHD_BODY void body_fftA(const FftArgs& a, const float* __restrict__ in, float2* __restrict__ spec, const Blk& b,
                        const PlaneSrc* src_sp) {
  constexpr int H = MX / 2, P = H + 1;
  __shared__ __align__(16) float2 buf[MY * P];  // plane_spread clears it 16 bytes at a time
  // the twiddles; before they are stored, plane_spread's lists (whose scales lie beyond the twiddles)
  constexpr int kTw = (MX + MY) * sizeof(float2);
  static_assert(offsetof(PlaneLds, scale) >= kTw, "the scales are read while the twiddles are stored");
  __shared__ __align__(16) unsigned char side[SP && (int)sizeof(PlaneLds) > kTw ? (int)sizeof(PlaneLds) : kTw];
  float2* const twx = reinterpret_cast<float2*>(side);
  float2* const twy = twx + MX;
  const int mz = a.g.mz;
  // with spreading, the three components and the neighbouring planes, which read the same sources,
  // are kept on one XCD
  const int item = SP ? xcd_item(b.x + b.nx * b.y, b.nx * b.ny) : 0;
  const int z = SP ? item / b.ny : b.x, c = SP ? item - z * b.ny : b.y;
  const float4* src = reinterpret_cast<const float4*>(in + ((size_t)c * mz + z) * (size_t)(MX * MY));
  constexpr int Q = MX / 4;
  // every load of this lane in flight at once, then into LDS (a load-store loop would wait out
  // one HBM round trip per element)
  constexpr int NL = (MY * Q + NT - 1) / NT;
  if constexpr (!SP) {
    float4 v[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < MY * Q) v[k] = src[e];
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < MY * Q) {
        const int y = e / Q, x4 = e - y * Q;
        buf[y * P + 2 * x4] = make_float2(v[k].x, v[k].y);
        buf[y * P + 2 * x4 + 1] = make_float2(v[k].z, v[k].w);
      }
    }
  } else {
    PlaneLds& pl = *reinterpret_cast<PlaneLds*>(side);
    // the integers become the plane in place; between two sweeps the first sums wait in this
    // workgroup's own rows of the spectrum (at least MX floats each), written later
    float* part = reinterpret_cast<float*>(spec + (size_t)c * MY * mz * P + (size_t)z * P);
    const auto at = [&](int e) { return (size_t)(e / (MX / 2)) * mz * 2 * P + 2 * (e % (MX / 2)); };
    int* acc = reinterpret_cast<int*>(buf);
    const float2* src2 = reinterpret_cast<const float2*>(src);
    const bool more = plane_spread<NT, false>(acc, 2 * MY * P, 2 * P, a.g, *src_sp, z, c, pl);
    const PlaneUnit unit = plane_unit(pl, *src_sp, a.g);
    if (more) {
      for (int e = threadIdx.x; e < MY * H; e += NT) {
        const int2 q = *reinterpret_cast<const int2*>(&buf[e / H * P + e % H]);
        const float f = unit.at(pl, 2 * (e % H), e / H);
        part[at(e)] = f * (float)q.x;
        part[at(e) + 1] = f * (float)q.y;
      }
      __syncthreads();
      plane_spread<NT, true>(acc, 2 * MY * P, 2 * P, a.g, *src_sp, z, c, pl);
    }
#pragma unroll 2
    for (int e = threadIdx.x; e < MY * H; e += NT) {
      float2* at_e = &buf[e / H * P + e % H];
      const int2 q = *reinterpret_cast<const int2*>(at_e);
      const float f = unit.at(pl, 2 * (e % H), e / H) * (more ? unit.rest : 1.0f);
      float2 r = make_float2(f * (float)q.x, f * (float)q.y);
      if (more) r = cadd(r, make_float2(part[at(e)], part[at(e) + 1]));
      *at_e = in ? cadd(r, src2[e]) : r;
    }
  }
  for (int i = threadIdx.x; i < MX; i += NT) twx[i] = a.twx[i];
  for (int i = threadIdx.x; i < MY; i += NT) twy[i] = a.twy[i];
  __syncthreads();
  ffft<H, 1, NT, MY, 2, false, plan_choice(H, PX)>(buf, MY, P, twx);
  constexpr int NP = H / 2 + 1;
  for (int e = threadIdx.x; e < MY * NP; e += NT) {
    const int y = e / NP, k = e - y * NP;
    float2* row = buf + y * P;
    const float2 A = row[k];
    const float2 B = cconj(row[k == 0 ? 0 : H - k]);
    const float2 E = cscale(cadd(A, B), 0.5f);
    const float2 D = csub(A, B);
    const float2 O = make_float2(0.5f * D.y, -0.5f * D.x);
    const float2 wO = cmul(twx[k], O);
    if (k == 0) {
      row[0] = make_float2(E.x + O.x, 0.0f);
      row[H] = make_float2(E.x - O.x, 0.0f);
    } else {
      row[k] = cadd(E, wO);
      if (H - k != k) row[H - k] = cconj(csub(E, wO));
    }
  }
  __syncthreads();
  ffft_modes<MY, P, NT, P, 1, false, plan_choice(MY, PY)>(buf, P, 1, twy, spec + (size_t)c * MY * mz * P + (size_t)z * P,
                                                          mz * P);
}

}  // namespace fhd
