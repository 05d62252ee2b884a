// plane_spread.h -- spreading S F fused into the forward xy transform: the workgroup that
// transforms plane z of component C first adds, in its LDS plane, every stencil row that lies on
// the plane, so the spread field never goes through memory and no separate spreading launch or
// stencil record exists.
//
// Replaces the 27-slot scatter + per-cell gather of src/stokesLimitFunctions.cu:659-1158,1198-1681
// and src/kernelSpreadParticles.cu:3012-4082.
//
// The contributions are added as 32-bit fixed-point integers by LDS atomics: integer addition is
// associative, so the field is bit-identical whatever order they arrive in.  The scale comes from
// the plane's largest source value and from the largest number of sources whose stencils can meet
// at one node (counted in blocks of 4 x 4 columns), so that no node's sum reaches 2^31; with more
// than kOneLimb of them a second sweep adds what the first one's rounding left over.
//
// Bound by the latency of its dependent phases and, for the pairs, by the vector instructions of
// the rows; a plane is one workgroup, so at 128^3 half the CUs hold two of the 384 planes and half
// one.  Per launch at 128^3 with 65,536 particles (rocprof): first solve (vector values, most of
// them zero) 34 us, second (values and pairs) 50 us, where the transform alone takes 17.7 us; a
// separate record pass, a spread of 8^3 tiles and the transform took 44 and 69 us.  64^3 with 16,384
// particles: 16 and 23 us against 22 and 37; 32^3 with 1,024: 12 and 16 us against 16 and 21.
//
//  1. scan: the sources sorted into the tile layers that can reach the plane are tested by a 4-byte
//     key (their half cell along z and their 4 x 4 block of columns); the hits enter the plane's
//     count and a list in LDS (ballot compaction).
//  2. values: vector values are read for the bound, and the hits with a zero component (a particle
//     with no WCA neighbour) leave the list.
//  3. add: one lane per listed source computes its weights along x and y and its weight on this
//     plane, and adds the 9 or 16 nodes of the row.  The two rows of a random-finite-difference
//     pair have the same nodes but for the few particles within the displacement of a half cell's
//     face, so their difference is added at once.
#pragma once
#include "fhd_device.h"
#include "fhd_kernels.h"

namespace fhd {

constexpr int kListCap = 6144;     // hits listed at once (also the sources scanned per chunk when more)
constexpr int kOneLimb = 255;      // most sources per node for a single 32-bit sum

// The key of a sorted slot: bits 0-8 its half cell along z (wrapped cell, sign of the offset), bit
// 9 set when a displacement below `margin` may change it, bits 16 up its block of 4 x 4 columns.
FHD_DEV unsigned plane_key(const GridDev& g, int cx, int cy, int cz, float dz, float margin) {
  const float a = fabsf(dz);
  const unsigned edge = a < margin || a > 0.5f * g.dz - margin ? 1u << 9 : 0u;
  return (unsigned)(2 * cz + (dz >= 0.0f ? 1 : 0)) | edge | ((unsigned)((cx >> 2) + ((g.mx + 3) >> 2) * (cy >> 2)) << 16);
}

// Weights of one axis at an explicit node base (the reference-quirk RFD variant): node k sits at
// integer position base + k in node units, the particle at c + frac - stag/2.
template <int NPTS>
FHD_DEV void axis_weights_at(int base, int c, float frac, int stag, AxisWeights& aw) {
  aw.base = base;
  float f = (float)(c - base) + frac - 0.5f * (float)stag;
#pragma unroll
  for (int k = 0; k < 4; ++k) aw.w[k] = (k < NPTS) ? (NPTS == 3 ? phi3(f - (float)k) : phi4(f - (float)k)) : 0.0f;
}

// A cell index wrapped into [0, m): usually at most one box away.
FHD_DEV int wrap_near(int c, int m) {
  c += c < 0 ? m : 0;
  c -= c >= m ? m : 0;
  return (unsigned)c < (unsigned)m ? c : wrapi(c, m);
}

// Largest value over the wave, in every lane.  (An LDS atomicMax with per-lane values compiles to
// a 64-iteration scalar read-lane loop, so each wave reduces first.)
FHD_DEV int wave_max_i32(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const int t = __shfl_xor(v, o);
    v = v > t ? v : t;
  }
  return v;
}

// The sources of one group that can reach a plane: up to three runs of sorted slots.
struct PlaneRuns {
  int s[3], n[3];
  FHD_DEV int total() const { return n[0] + n[1] + n[2]; }
  FHD_DEV int slot(int i) const {
    return i < n[0] ? s[0] + i : i < n[0] + n[1] ? s[1] + (i - n[0]) : s[2] + (i - n[0] - n[1]);
  }
};

// Boundary k (0-5: first and last slot of three runs) of group G's runs for plane z.
FHD_DEV int run_bound(const Tiles& t, const SpreadGroup& G, int z, int k) {
  const int own = z / t.tz, lz = z - own * t.tz, which = k >> 1;
  // a source stays within one cell of its layer (the sort's skin is at most half a cell); its
  // stencil reaches two cells, plus its displacement.  Along an axis of one or two tiles sources
  // are listed in any of them.
  const int reach = 3 + ((G.wide + 1) >> 1);
  int lay = own;
  bool on = which == 0;
  if (which == 1) {
    on = t.ntz == 2 || (t.ntz >= 3 && lz < reach);
    lay = own == 0 ? t.ntz - 1 : own - 1;
  } else if (which == 2) {
    on = t.ntz >= 3 && lz >= t.tz - reach;
    lay = own == t.ntz - 1 ? 0 : own + 1;
  }
  return on ? G.set.start[(lay + (k & 1)) * t.ntx * t.nty] : 0;
}

// Whether the stencil of a source with half cell h2 along z has a node on plane z for component C
// (never false for one that has: `wide` half cells of displacement either way are allowed for).
FHD_DEV bool row_hits(int h2, int wide, int z, int mz, int npts, bool stag) {
  const int off = (npts == 4) != stag ? 1 : 0, back = npts == 3 && !stag ? 1 : 2;
  const int lo = ((h2 - wide + off) >> 1) - back, hi = ((h2 + wide + off) >> 1) - back + npts - 1;
  int t = z - lo;
  t += t < 0 ? mz : 0;
  t -= t >= mz ? mz : 0;
  return t <= hi - lo || hi - lo >= mz - 1;
}

// Weights along one axis of a source at cell c, offset d, displaced by `disp`, first node folded into
// the box.  quirk: the nodes come from the displaced position, the weights from the undisplaced one.
// drift: weights become val x weight + drift x derivative weight (the force and the thermal drift
// share their nodes).
template <int NPTS>
FHD_DEV AxisWeights src_axis(int c, float d, float disp, float h, float ih, int m, int stag, bool quirk, float val,
                             float drift) {
  float x = d + disp;
  int cc = c;
  if (!(fabsf(x) < 0.5f * h)) {
    renorm_axis(cc, x, h, ih);
    cc = wrap_near(cc, m);
  }
  AxisWeights w;
  axis_weights<NPTS>(cc, x * ih, stag, w);
  if (quirk) axis_weights_at<NPTS>(w.base, c, d * ih, stag, w);
  if (drift != 0.0f) {
    AxisWeights dw;
    axis_dweights<NPTS>(cc, x * ih, 1, dw);
#pragma unroll
    for (int k = 0; k < NPTS; ++k) w.w[k] = fmaf(val, w.w[k], drift * dw.w[k]);
  }
  w.base = fold(w.base, m);
  return w;
}

// The weight on plane z (zero when the stencil misses it).
template <int NPTS>
FHD_DEV float row_weight(const AxisWeights& w, int z, int mz) {
  float r = 0.0f;
  if (mz >= NPTS) {
    int t = z - w.base;
    t += t < 0 ? mz : 0;
#pragma unroll
    for (int k = 0; k < NPTS; ++k) r = t == k ? w.w[k] : r;
  } else {  // a stencil that meets the plane more than once
    for (int k = 0; k < NPTS; ++k) r += fold(w.base + k, mz) == z ? w.w[k] : 0.0f;
  }
  return r;
}

// Node k along an axis from the folded first node b.
FHD_DEV int node_at(int b, int k, int m) {
  int n = b + k;
  n -= n >= m ? m : 0;
  if (m < 4) n %= m;
  return n;
}

// Adds the nodes of a row (weights wx and wy times r), or of the difference of two rows on the same
// nodes (PAIR: minus vx and vy times s).
template <int NPTS, bool PAIR>
FHD_DEV void add_nodes(int* acc, int pitch, const GridDev& g, const AxisWeights& wx, const AxisWeights& wy, float r,
                       const AxisWeights& vx, const AxisWeights& vy, float s, float scale2) {
  int xs[NPTS];
#pragma unroll
  for (int k = 0; k < NPTS; ++k) xs[k] = node_at(wx.base, k, g.mx);
#pragma unroll
  for (int ky = 0; ky < NPTS; ++ky) {
    const int row = node_at(wy.base, ky, g.my) * pitch;
    const float wyz = wy.w[ky] * r, vyz = PAIR ? vy.w[ky] * s : 0.0f;
#pragma unroll
    for (int kx = 0; kx < NPTS; ++kx) {
      float v = wx.w[kx] * wyz;
      if (PAIR) v = fmaf(-vx.w[kx], vyz, v);
      // rounded: truncation would shift every sum toward zero (it tripled the velocity's error)
      int n = (int)rintf(v);
      if (scale2 != 0.0f) n = (int)rintf((v - (float)n) * scale2);
      atomicAdd(&acc[row + xs[kx]], n);
    }
  }
}

// Most that an axis of m cells contributes to what a source adds to a node, per unit of its value: one
// weight (1/2 of 4 points, 2/3 of 3), or the sum of those that a narrow axis folds onto the node, which is
// more only on an axis of one cell, where it is all of them.  deriv: derivative weights may take the
// place of the plain ones (thermal drift: 1/2 and 1; folded onto one cell they cancel).
template <int NPTS>
FHD_DEV float axis_most(int m, bool deriv) {
  return m == 1 ? 1.0f : NPTS == 4 ? 0.5f : deriv ? 1.0f : 2.0f / 3.0f;
}

struct PlaneLds {
  unsigned short list[kListCap];  // group 0's hits from the front, group 1's from the back
  int runs[2][6];
  int n[2];   // the groups' hit counts
  int kept;   // group 0's hits with a value
  int bound;  // largest value (float bits)
  int most;   // most sources that can meet at a node
};

FHD_DEV int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Appends the kept entries of a wave's lanes to the front of the list.
FHD_DEV void list_keep(PlaneLds& L, bool keep, int entry) {
  const int lane = threadIdx.x & 63;
  const unsigned long long bal = __ballot(keep);
  if (bal == 0) return;
  int at = 0;
  if (lane == 0) at = atomicAdd(&L.kept, __popcll(bal));
  at = __shfl(at, 0) + __popcll(bal & ((1ull << lane) - 1ull));
  if (keep) L.list[at] = (unsigned short)entry;
}

FHD_DEV PlaneRuns plane_runs(const PlaneLds& L, int gi) {
  PlaneRuns r;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    r.s[k] = uniform(L.runs[gi][2 * k]);
    r.n[k] = uniform(L.runs[gi][2 * k + 1]) - r.s[k];
  }
  return r;
}

// Lists the hits among sources [i0, i1) of group gi (entries relative to i0); `count`: also counts
// them by block.  K keys of a lane are in flight at once.
template <int NT, int K>
FHD_DEV void plane_keys(const SpreadGroup& G, const PlaneRuns& runs, int b, int i1, unsigned key[K]) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = b + k * NT + (int)threadIdx.x;
    key[k] = i < i1 ? G.key[runs.slot(i)] : ~0u;
  }
}
template <int NT, int K>
FHD_DEV void plane_test(const GridDev& g, const PlaneSrc& P, int gi, const unsigned key[K], int b, int i0, int z, int C,
                        PlaneLds& L, int* blocks, bool count) {
  const SpreadGroup& G = P.grp[gi];
  const int lane = threadIdx.x & 63;
  unsigned long long bal[K];
  int total = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const bool hit = key[k] != ~0u && row_hits(key[k] & 511, key[k] & 512 ? G.wide : 0, z, g.mz, P.kernel_points, C == 2);
    if (hit && count) atomicAdd(&blocks[key[k] >> 16], G.mode == SRC_RFD ? 2 : 1);
    bal[k] = __ballot(hit);
    total += __popcll(bal[k]);
  }
  if (total == 0) return;
  int at = 0;
  if (lane == 0) at = atomicAdd(&L.n[gi], total);
  at = __shfl(at, 0);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int mine = at + __popcll(bal[k] & ((1ull << lane) - 1ull));
    if ((bal[k] >> lane & 1) && mine < kListCap)
      L.list[gi == 0 ? mine : kListCap - 1 - mine] = (unsigned short)(b + k * NT + (int)threadIdx.x - i0);
    at += __popcll(bal[k]);
  }
}
// from: the first source scanned (i0 or later).
template <int NT>
FHD_DEV void plane_scan(const GridDev& g, const PlaneSrc& P, int gi, const PlaneRuns& runs, int i0, int from, int i1,
                        int z, int C, PlaneLds& L, int* blocks, bool count) {
  constexpr int K = 4;
  for (int b = from; b < i1; b += K * NT) {
    unsigned key[K];
    plane_keys<NT, K>(P.grp[gi], runs, b, i1, key);
    plane_test<NT, K>(g, P, gi, key, b, i0, z, C, L, blocks, count);
  }
}

// Component C of source j's value.
FHD_DEV float src_value(const SpreadGroup& G, int j, int C) {
  return G.coef * reinterpret_cast<const float*>(G.val + G.set.id[j])[C];
}

// Adds source j's row to the plane.
template <int NPTS>
FHD_DEV void plane_add(int* acc, int pitch, const GridDev& g, const SpreadGroup& G, int j, int z, int C, float scale,
                       float scale2) {
  float v = src_value(G, j, C);
  v = fabsf(v) <= 3.0e38f ? v : 0.0f;  // the plane is marked already
  const int4 c = G.set.cell[j];
  const float4 d = G.set.off[j];
  const float drift = G.drift * (C == 0 ? g.idx : C == 1 ? g.idy : g.idz);
  const auto axis = [&](int a, int ca, float da, float h, float ih, int m) {
    const bool face = a == C;
    return src_axis<NPTS>(ca, da, 0.0f, h, ih, m, face, false, v, face ? drift : 0.0f);
  };
  float r = row_weight<NPTS>(axis(2, c.z, d.z, g.dz, g.idz, g.mz), z, g.mz) * scale;
  if (drift == 0.0f) r *= v;
  const AxisWeights wx = axis(0, c.x, d.x, g.dx, g.idx, g.mx), wy = axis(1, c.y, d.y, g.dy, g.idy, g.my);
  add_nodes<NPTS, false>(acc, pitch, g, wx, wy, r, wx, wy, 0.0f, scale2);
}

// Adds the difference of both rows of RFD pair j.
template <int NPTS>
FHD_DEV void plane_add_pair(int* acc, int pitch, const GridDev& g, const SpreadGroup& G, int j, int z, int C, float scale,
                            float scale2) {
  const int4 c = G.set.cell[j];
  const float4 d = G.set.off[j];
  const float4 w = G.val[j];
  const float v = (C == 0 ? w.x : C == 1 ? w.y : w.z) * G.coef * scale;
  const bool quirk = G.rfd_quirk;
  const auto zw = [&](float s) {
    return v * row_weight<NPTS>(src_axis<NPTS>(c.z, d.z, s * w.z, g.dz, g.idz, g.mz, C == 2, quirk, 0.0f, 0.0f), z, g.mz);
  };
  const float r0 = zw(G.disp), r1 = zw(-G.disp);
  const AxisWeights x0 = src_axis<NPTS>(c.x, d.x, G.disp * w.x, g.dx, g.idx, g.mx, C == 0, quirk, 0.0f, 0.0f);
  const AxisWeights x1 = src_axis<NPTS>(c.x, d.x, -G.disp * w.x, g.dx, g.idx, g.mx, C == 0, quirk, 0.0f, 0.0f);
  const AxisWeights y0 = src_axis<NPTS>(c.y, d.y, G.disp * w.y, g.dy, g.idy, g.my, C == 1, quirk, 0.0f, 0.0f);
  const AxisWeights y1 = src_axis<NPTS>(c.y, d.y, -G.disp * w.y, g.dy, g.idy, g.my, C == 1, quirk, 0.0f, 0.0f);
  if (x0.base == x1.base && y0.base == y1.base) {
    add_nodes<NPTS, true>(acc, pitch, g, x0, y0, r0, x1, y1, r1, scale2);
  } else {
    add_nodes<NPTS, false>(acc, pitch, g, x0, y0, r0, x0, y0, 0.0f, scale2);
    add_nodes<NPTS, false>(acc, pitch, g, x1, y1, -r1, x1, y1, 0.0f, scale2);
  }
}
template <int NPTS, int NT>
FHD_DEV void plane_add_list(int* acc, int pitch, const GridDev& g, const SpreadGroup& G, int gi, const PlaneRuns& runs,
                            int i0, int nh, int z, int C, const PlaneLds& L, float scale, float scale2) {
  for (int k = threadIdx.x; k < nh; k += NT) {
    const int j = runs.slot(i0 + L.list[gi == 0 ? k : kListCap - 1 - k]);
    if (G.mode == SRC_RFD) plane_add_pair<NPTS>(acc, pitch, g, G, j, z, C, scale, scale2);
    else plane_add<NPTS>(acc, pitch, g, G, j, z, C, scale, scale2);
  }
}

// Accumulates the plane into acc (`words` words, row pitch `pitch`, cleared here) and returns what
// the integers are to be multiplied by; *inv2 != 0: the caller takes these sums (times the returned
// factor) and calls again with sweep 1 for the remainders, to be multiplied by *inv2.  Every lane
// of the workgroup calls it; the plane is complete (barrier passed) on return.
template <int NPTS, int NT>
FHD_DEV float plane_spread(int* acc, int words, int pitch, const GridDev& g, const PlaneSrc& P, int z, int C,
                           PlaneLds& L, int sweep, float* inv2) {
  int* const blocks = acc;  // the block counts, until the plane is cleared
  const int tid = threadIdx.x, lane = tid & 63;
  const int bx = (g.mx + 3) >> 2, by = (g.my + 3) >> 2;
  if (tid < 12 && tid < 6 * P.ngroups) L.runs[tid >= 6][tid % 6] = run_bound(P.t, P.grp[tid >= 6], z, tid % 6);
  if (sweep == 0)
    for (int e = tid; e < bx * by; e += NT) blocks[e] = 0;
  if (tid < 2) L.n[tid] = 0;
  if (tid == 0) L.kept = 0;
  if (sweep == 0 && tid == 0) L.bound = L.most = 0;
  __syncthreads();
  const bool two = P.ngroups > 1;
  bool one;  // every group's sources have 16-bit indices
  {
    const PlaneRuns r0 = plane_runs(L, 0);
    const int n0 = r0.total();
    // the first keys of both groups are in flight at once
    constexpr int K = 4;
    unsigned k0[K], k1[K];
    plane_keys<NT, K>(P.grp[0], r0, 0, n0, k0);
    PlaneRuns r1 = r0;
    int n1 = 0;
    if (two) {
      r1 = plane_runs(L, 1);
      n1 = r1.total();
      plane_keys<NT, K>(P.grp[1], r1, 0, n1, k1);
    }
    plane_test<NT, K>(g, P, 0, k0, 0, 0, z, C, L, blocks, sweep == 0);
    if (n0 > K * NT) plane_scan<NT>(g, P, 0, r0, 0, K * NT, n0, z, C, L, blocks, sweep == 0);
    if (two) {
      plane_test<NT, K>(g, P, 1, k1, 0, 0, z, C, L, blocks, sweep == 0);
      if (n1 > K * NT) plane_scan<NT>(g, P, 1, r1, 0, K * NT, n1, z, C, L, blocks, sweep == 0);
    }
    one = n0 <= 65536 && n1 <= 65536;
  }
  __syncthreads();
  int nhit0 = uniform(L.n[0]);
  const int nhit1 = uniform(L.n[1]);
  one = one && nhit0 + nhit1 <= kListCap;
  // most sources at a node: its stencils come from cells at most 3 away, so from the blocks of 4 around
  // its own, unless a pair is displaced by more than a cell along x or y
  const auto count_and_clear = [&] {
    if (sweep == 0) {
      int most = 0;
      if (P.near) {
        for (int e = tid; e < bx * by; e += NT) {
          const int y = e / bx, x = e - y * bx;
          int s = 0;
          for (int dy = -1; dy <= min(1, by - 2); ++dy) {
            const int yy = y + dy < 0 ? by - 1 : y + dy >= by ? 0 : y + dy;
            for (int dx = -1; dx <= min(1, bx - 2); ++dx) {
              const int xx = x + dx < 0 ? bx - 1 : x + dx >= bx ? 0 : x + dx;
              s += blocks[xx + bx * yy];
            }
          }
          most = max(most, s);
        }
      } else {
        most = nhit0 + 2 * nhit1;
      }
      most = wave_max_i32(most);
      if (lane == 0) atomicMax(&L.most, most);
    }
    __syncthreads();
    int4* acc4 = reinterpret_cast<int4*>(acc);
    for (int e = tid; e < words / 4; e += NT) acc4[e] = make_int4(0, 0, 0, 0);
    if (tid < (words & 3)) acc[(words & ~3) + tid] = 0;
  };
  // bound of the values: a pair's normals are below 5.8 (24-bit uniforms), vector values are read
  // (under the count).  Group 0 holds vector values; its listed hits without one leave the list.
  {
    const SpreadGroup& G = P.grp[0];
    const PlaneRuns r = plane_runs(L, 0);
    const float drift = fabsf(G.drift) * (C == 0 ? g.idx : C == 1 ? g.idy : g.idz);
    float m = two ? 5.8f * fabsf(P.grp[1].coef) : 0.0f;
    if (one) {
      constexpr int K = (kListCap + NT - 1) / NT;
      constexpr int KF = 3;  // values of a lane in flight at once
      unsigned short e[KF];
      float v[KF];
      // rounds of KF x NT entries, each read in full before the shorter list overwrites it
      for (int k0 = 0; k0 < K * NT && (k0 == 0 || k0 < nhit0); k0 += KF * NT) {
#pragma unroll
        for (int k = 0; k < KF; ++k) {
          const int i = k0 + tid + k * NT;
          v[k] = 0.0f;
          if (i < nhit0) {
            e[k] = L.list[i];
            v[k] = src_value(G, r.slot(e[k]), C);
          }
        }
        if (k0 == 0) count_and_clear();
        else __syncthreads();
#pragma unroll
        for (int k = 0; k < KF; ++k) {
          const bool in = k0 + tid + k * NT < nhit0;
          const float a = fabsf(v[k]) + drift;
          if (in) m = fmaxf(m, a <= 3.0e38f ? a : 3.4e38f);  // overflowed or NaN: marks the plane
          list_keep(L, in && (v[k] != 0.0f || drift != 0.0f), e[k]);
        }
      }
    } else {
      count_and_clear();
      for (int i = tid; i < r.total(); i += NT) {
        const float a = fabsf(src_value(G, r.slot(i), C)) + drift;
        m = fmaxf(m, a <= 3.0e38f ? a : 3.4e38f);
      }
    }
    const int w = wave_max_i32(__float_as_int(m));
    if (lane == 0) atomicMax(&L.bound, w);
  }
  __syncthreads();
  if (one) nhit0 = uniform(L.kept);
  // what a source adds to a node is below value x the product of its axes' most (axis_most)
  const float top = __int_as_float(uniform(L.bound));
  const bool bad = top > 3.0e38f;
  const bool drift = P.grp[0].drift != 0.0f;
  const float most = axis_most<NPTS>(g.mx, drift && C == 0) * axis_most<NPTS>(g.my, drift && C == 1) *
                     axis_most<NPTS>(g.mz, drift && C == 2);
  const float m = bad ? 0.0f : 1.001f * top * most;
  const int n = max(uniform(L.most), 1);
  int e2 = -90;
  if (m > 0.0f) {
    int e;
    frexpf(m, &e);  // m < 2^e
    e2 = max(e, -90);
  }
  // n 2^S <= 2^31; a source's up to eight additions to a node round by half a unit each, which the
  // thousandth above covers while S >= 13
  const int S = 30 - (31 - __clz(n)) - (n > 65536 ? 1 : 0);
  const float scale = ldexpf(1.0f, S - e2);
  const float scale2 = sweep == 0 ? 0.0f : ldexpf(1.0f, S);
  for (int gi = 0; gi < P.ngroups; ++gi) {
    const SpreadGroup& G = P.grp[gi];
    const PlaneRuns r = plane_runs(L, gi);
    // more hits than the list holds: chunks of as many sources
    const int all = one ? 1 : r.total(), step = one ? 1 : kListCap;
    for (int i0 = 0; i0 < all; i0 += step) {
      int nh = gi == 0 ? nhit0 : nhit1;
      if (!one) {
        __syncthreads();  // the previous chunk's list consumed
        if (tid == 0) L.n[gi] = 0;
        __syncthreads();
        plane_scan<NT>(g, P, gi, r, i0, i0, min(all, i0 + step), z, C, L, blocks, false);
        __syncthreads();
        nh = uniform(L.n[gi]);
      }
      plane_add_list<NPTS, NT>(acc, pitch, g, G, gi, r, one ? 0 : i0, nh, z, C, L, scale, scale2);
    }
  }
  __syncthreads();
  // an overflowed or NaN source: the plane is written non-finite, which the interpolation flags
  const float inv = bad ? __builtin_inff() : ldexpf(1.0f, e2 - S) * P.out_coef;
  *inv2 = n > kOneLimb && !bad ? ldexpf(inv, -S) : 0.0f;
  return inv;
}
template <int NT>
FHD_DEV float plane_spread(int* acc, int words, int pitch, const GridDev& g, const PlaneSrc& P, int z, int C,
                           PlaneLds& L, int sweep, float* inv2) {
  return P.kernel_points == 4 ? plane_spread<4, NT>(acc, words, pitch, g, P, z, C, L, sweep, inv2)
                              : plane_spread<3, NT>(acc, words, pitch, g, P, z, C, L, sweep, inv2);
}

}  // namespace fhd
