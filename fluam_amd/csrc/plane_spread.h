// plane_spread.h -- spreading S F fused into the forward xy transform: the workgroup that
// transforms plane z of component C first adds, in its LDS plane, every stencil row that lies on
// the plane, so the spread field never goes through memory and no separate spreading launch or
// stencil record exists.
//
// Replaces the 27-slot scatter + per-cell gather of src/stokesLimitFunctions.cu:659-1158,1198-1681
// and src/kernelSpreadParticles.cu:3012-4082.
//
// The contributions are added as 32-bit fixed-point integers by LDS atomics: integer addition is
// associative, so the field is bit-identical whatever order they arrive in.  Every 4 x 4 block of columns
// has its own scale, from the largest value among the sources that can reach it and from their number, so
// that no node's sum reaches 2^31 and a weak force is rounded by its own neighbourhood's measure, not by
// the plane's strongest; where that leaves a row less than 23 bits (255 forces or some 15,000 pairs in
// reach of a block) a second sweep adds what the first one's rounding left over.
//
// Bound by the latency of its dependent phases and, for the pairs, by the vector instructions of
// the rows; a plane is one workgroup, so at 128^3 half the CUs hold two of the 384 planes and half
// one.  Per launch at 128^3 with 65,536 particles (rocprof): first solve (vector values, most of
// them zero) 32 us, second (values and pairs) 52 us, where the transform alone takes 16 us; a
// separate record pass, a spread of 8^3 tiles and the transform took 44 and 69 us.  64^3 with 16,384
// particles: 16 and 24 us against 22 and 37; 32^3 with 1,024: 10 and 14 us against 16 and 21.  At the
// 64 registers that let two planes share a CU the 128 x 128 kernel spills 11 VGPRs, smaller ones none.
//
//  1. scan: the sources sorted into the tile layers that can reach the plane are tested by a 4-byte
//     key (their half cell along z and their 4 x 4 block of columns); the hits enter a list in LDS
//     (ballot compaction), pairs their block's count.
//  2. values: vector values are read for the blocks' counts and bounds, and the hits with a zero component
//     (a particle with no WCA neighbour) leave the list.
//  3. scales: each block's, from the counts and bounds of the blocks around it.
//  4. add: one lane per listed source computes its weights along x and y and its weight on this
//     plane, and adds the 9 or 16 nodes of the row.  The two rows of a random-finite-difference
//     pair have the same nodes but for the few particles within the displacement of a half cell's
//     face, so their difference is added at once.
// Planes with more hits than the list holds do without it: they read the values of all sources in
// reach, and each wave then collects the hits of its own share of the keys and adds a row per lane.  128^3
// with 524,288 particles: 300 us per launch (their average), where listing them piece by piece took 384,
// and the record pass, the spread and the transform 297; 64^3 with 131,072: 147, 179 and 157 us.
#pragma once
#include <stddef.h>
#include "fhd_device.h"
#include "fhd_kernels.h"

namespace fhd {

constexpr int kListCap = 6144;     // most hits listed
constexpr int kPlaneBlocks = 1024; // 4 x 4 blocks of the largest plane that can hold particles

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

// Most that an axis of m cells contributes to what a source adds to a node, per unit of its value: one
// weight (1/2 of 4 points, 2/3 of 3), or the sum of those that a narrow axis folds onto the node, which is
// more only on an axis of one cell, where it is all of them.  deriv: derivative weights may take the
// place of the plain ones (thermal drift: 1/2 and 1; folded onto one cell they cancel).
template <int NPTS>
FHD_DEV float axis_most(int m, bool deriv) {
  return m == 1 ? 1.0f : NPTS == 4 ? 0.5f : deriv ? 1.0f : 2.0f / 3.0f;
}

struct PlaneLds {
  union {
    unsigned short list[kListCap];  // group 0's hits from the front, group 1's from the back
    int slots[kListCap / 2];        // without a list: a share of each wave for its next hits
  };
  int runs[2][6];
  int n[2];   // the groups' hit counts
  int kept;   // group 0's hits with a value (without a list: whether there are any)
  int most;   // most additions that can meet at a node
  int top;    // largest value (float bits)
  int more;   // the remainders are to be summed as well
  int bad;    // an overflowed or NaN source
  signed char scale[kPlaneBlocks];  // binary exponent of each 4 x 4 block's fixed-point scale
};

// Bounds per plane and component: what a source adds to a node is below its value times `most`; one row of
// a pair below `row`, and the two rows' difference, their weights being Lipschitz, below `diff` (a hundredth
// of it at the default displacement).
struct PlaneBounds {
  float most, row, diff;
};
template <int NPTS>
FHD_DEV PlaneBounds plane_bounds(const GridDev& g, const PlaneSrc& P, int C) {
  const int m[3] = {g.mx, g.my, g.mz};
  const float ih[3] = {g.idx, g.idy, g.idz};
  const bool two = P.ngroups > 1, drift = P.grp[0].drift != 0.0f;
  PlaneBounds b{1.0f, 0.0f, 0.0f};
  // a pair's normals are below 5.8 (24-bit uniforms)
  const float apart = two ? 2.0f * 5.8f * fabsf(P.grp[1].disp) : 0.0f;
  float w[3], d[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    w[a] = axis_most<NPTS>(m[a], drift && a == C);
    // slopes are at most 1/2 and 1; a narrow axis folds two weights onto a node
    d[a] = m[a] == 1 ? 0.0f : fminf(w[a], (NPTS == 4 ? 0.5f : 1.0f) * (m[a] < NPTS ? 2.0f : 1.0f) * apart * ih[a]);
    b.most *= w[a];
  }
  if (two) {
    const float v = fminf(5.8f * fabsf(P.grp[1].coef), 3.0e38f);
    b.row = v * b.most;
    b.diff = v * fminf(b.most, d[0] * w[1] * w[2] + w[0] * d[1] * w[2] + w[0] * w[1] * d[2]);
  }
  return b;
}
// Binary exponent x of the fixed-point scale of nodes that `nf` values of at most t and `np` pairs reach:
// no node's sum passes 2^31, no single row's value 2^30.  A hundredth is left for what the additions round,
// at most eight of them from a source.  more: the largest row keeps less than 23 bits, so the remainders
// are to be summed as well.
FHD_DEV int block_scale(const PlaneBounds& b, int nf, int np, float t, bool& more) {
  const float down = 9.31322575e-10f;  // 2^-30: counts times values stay finite
  const float value = t * b.most * down;
  const float row = 1.01f * fmaxf(value, np ? b.row * down : 0.0f);
  const float sum = 1.01f * fmaf((float)nf, value, (float)np * (b.diff * down));
  int er = -200, es = -200;
  if (row > 0.0f) frexpf(row, &er);  // row < 2^er
  if (sum > 0.0f) frexpf(sum, &es);
  er = max(er + 30, -90);
  const int x = min(30 - er, 1 - es) - (nf + np > 1 << 18 ? 1 : 0);
  more |= x < 23 - er;
  return x;
}
// Binary exponent of the scale of the remainders, which are at most half a unit each.
FHD_DEV int rest_exp(int most) { return 27 - (31 - __clz(max(most, 1))); }

// Adds the nodes of a row (weights wx and wy times r), or of the difference of two rows on the same
// nodes (PAIR: minus vx and vy times s).  Four nodes lie in at most two blocks along an axis.
template <int NPTS, bool PAIR>
FHD_DEV void add_nodes(int* acc, int pitch, const GridDev& g, const PlaneLds& L, const AxisWeights& wx,
                       const AxisWeights& wy, float r, const AxisWeights& vx, const AxisWeights& vy, float s,
                       float scale2) {
  const int nbx = (g.mx + 3) >> 2, nby = (g.my + 3) >> 2;
  const int xa = wx.base >> 2, xb = xa + 1 == nbx ? 0 : xa + 1;
  const int ya = wy.base >> 2, yb = ya + 1 == nby ? 0 : ya + 1;
  const int aa = L.scale[xa + nbx * ya], ba = L.scale[xb + nbx * ya];
  const int ab = L.scale[xa + nbx * yb], bb = L.scale[xb + nbx * yb];
  int xs[NPTS];
#pragma unroll
  for (int k = 0; k < NPTS; ++k) xs[k] = node_at(wx.base, k, g.mx);
#pragma unroll
  for (int ky = 0; ky < NPTS; ++ky) {
    const int y = node_at(wy.base, ky, g.my), row = y * pitch;
    const bool own = y >> 2 == ya;
    const int ea = own ? aa : ab, eb = own ? ba : bb;
    const float wyz = wy.w[ky] * r, vyz = PAIR ? vy.w[ky] * s : 0.0f;
#pragma unroll
    for (int kx = 0; kx < NPTS; ++kx) {
      float v = wx.w[kx] * wyz;
      if (PAIR) v = fmaf(-vx.w[kx], vyz, v);
      v = ldexpf(v, xs[kx] >> 2 == xa ? ea : eb);
      // rounded: truncation would shift every sum toward zero (it tripled the velocity's error)
      int n = (int)rintf(v);
      if (scale2 != 0.0f) n = (int)rintf((v - (float)n) * scale2);
      atomicAdd(&acc[row + xs[kx]], n);
    }
  }
}

FHD_DEV int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Appends the kept entries of a wave's lanes to the front of the list.
FHD_DEV void list_keep(PlaneLds& L, int lane, bool keep, int entry) {
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

// Component C of source j's value.
FHD_DEV float src_value(const SpreadGroup& G, int j, int C) {
  return G.coef * reinterpret_cast<const float*>(G.val + G.set.id[j])[C];
}

// The keys of sources [b, b + K NT) of a group, K of a lane in flight at once.
template <int NT, int K>
FHD_DEV void plane_keys(const SpreadGroup& G, const PlaneRuns& runs, int tid, int b, int i1, unsigned key[K]) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = b + k * NT + tid;
    key[k] = i < i1 ? G.key[runs.slot(i)] : ~0u;
  }
}
FHD_DEV bool key_hits(unsigned key, const SpreadGroup& G, int z, int mz, int npts, bool stag) {
  return key != ~0u && row_hits(key & 511, key & 512 ? G.wide : 0, z, mz, npts, stag);
}
// Lists the marked sources.
template <int NT, int K>
FHD_DEV void plane_list(PlaneLds& L, int gi, int tid, const bool hit[K], int b) {
  const int lane = tid & 63;
  unsigned long long bal[K];
  int total = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    bal[k] = __ballot(hit[k]);
    total += __popcll(bal[k]);
  }
  if (total == 0) return;
  int at = 0;
  if (lane == 0) at = atomicAdd(&L.n[gi], total);
  at = __shfl(at, 0);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int mine = at + __popcll(bal[k] & ((1ull << lane) - 1ull));
    if (hit[k] && mine < kListCap) L.list[gi == 0 ? mine : kListCap - 1 - mine] = (unsigned short)(b + k * NT + tid);
    at += __popcll(bal[k]);
  }
}
// Lists the hits among the keys, and counts pairs by block (block null: not).
template <int NT, int K>
FHD_DEV void plane_test(const GridDev& g, const PlaneSrc& P, int gi, int tid, const unsigned key[K], int b, int z,
                        int C, PlaneLds& L, int4* block) {
  bool hit[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    hit[k] = key_hits(key[k], P.grp[gi], z, g.mz, P.kernel_points, C == 2);
    if (hit[k] && gi == 1 && block) atomicAdd(&block[key[k] >> 16].y, 1);
  }
  plane_list<NT, K>(L, gi, tid, hit, b);
}
template <int NT>
FHD_DEV void plane_scan(const GridDev& g, const PlaneSrc& P, int gi, int tid, const PlaneRuns& runs, int from, int i1,
                        int z, int C, PlaneLds& L, int4* block) {
  constexpr int K = 4;
  for (int b = from; b < i1; b += K * NT) {
    unsigned key[K];
    plane_keys<NT, K>(P.grp[gi], runs, tid, b, i1, key);
    plane_test<NT, K>(g, P, gi, tid, key, b, z, C, L, block);
  }
}

// Adds source j's row to the plane.
template <int NPTS>
FHD_DEV void plane_add(int* acc, int pitch, const GridDev& g, const PlaneLds& L, const SpreadGroup& G, int j, int z,
                       int C, float scale2) {
  float v = src_value(G, j, C);
  v = fabsf(v) <= 3.0e38f ? v : 0.0f;  // the plane is marked already
  const int4 c = G.set.cell[j];
  const float4 d = G.set.off[j];
  const float drift = G.drift * (C == 0 ? g.idx : C == 1 ? g.idy : g.idz);
  const auto axis = [&](int a, int ca, float da, float h, float ih, int m) {
    const bool face = a == C;
    return src_axis<NPTS>(ca, da, 0.0f, h, ih, m, face, false, v, face ? drift : 0.0f);
  };
  float r = row_weight<NPTS>(axis(2, c.z, d.z, g.dz, g.idz, g.mz), z, g.mz);
  if (drift == 0.0f) r *= v;
  const AxisWeights wx = axis(0, c.x, d.x, g.dx, g.idx, g.mx), wy = axis(1, c.y, d.y, g.dy, g.idy, g.my);
  add_nodes<NPTS, false>(acc, pitch, g, L, wx, wy, r, wx, wy, 0.0f, scale2);
}

// Adds the difference of both rows of RFD pair j.
template <int NPTS>
FHD_DEV void plane_add_pair(int* acc, int pitch, const GridDev& g, const PlaneLds& L, const SpreadGroup& G, int j, int z,
                            int C, float scale2) {
  const int4 c = G.set.cell[j];
  const float4 d = G.set.off[j];
  const float4 w = G.val[j];
  const float v = (C == 0 ? w.x : C == 1 ? w.y : w.z) * G.coef;
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
    add_nodes<NPTS, true>(acc, pitch, g, L, x0, y0, r0, x1, y1, r1, scale2);
  } else {
    add_nodes<NPTS, false>(acc, pitch, g, L, x0, y0, r0, x0, y0, 0.0f, scale2);
    add_nodes<NPTS, false>(acc, pitch, g, L, x1, y1, -r1, x1, y1, 0.0f, scale2);
  }
}
// The next source for this lane (-1: none) of those of a group that hit the plane, gathered without the list:
// each wave takes its share of the keys (from b on), collects their hits (of group 0 those with a value) in
// LDS (n of them) and hands them out whenever it has one for every lane.  No barrier, so the waves cover each
// other's loads.  False when nothing is left.
template <int NPTS, int NT, bool PAIRS>
FHD_DEV bool plane_gather(const SpreadGroup& G, const PlaneRuns& r, int all, int lane, int* slots, int mz, int z, int C,
                          int& b, int& n, int& j) {
  constexpr int K = 2;
  static_assert(64 * K + 63 <= kListCap / 2 / (NT / 64), "a wave's share holds what it collects");
  while (n < 64 && b < all) {
    int slot[K];
    unsigned key[K];
    float v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = b + k * 64 + lane;
      slot[k] = r.slot(i);
      key[k] = i < all ? G.key[slot[k]] : ~0u;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (!key_hits(key[k], G, z, mz, NPTS, C == 2)) key[k] = ~0u;
      if (!PAIRS) v[k] = key[k] != ~0u ? src_value(G, slot[k], C) : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const bool hit = key[k] != ~0u && (PAIRS || v[k] != 0.0f || G.drift != 0.0f);
      const unsigned long long bal = __ballot(hit);
      if (hit) slots[n + __popcll(bal & ((1ull << lane) - 1ull))] = slot[k];
      n += __popcll(bal);
    }
    b += NT * K;
  }
  if (n == 0) return false;
  const int take = min(n, 64);
  n -= take;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  j = lane < take ? slots[n + lane] : -1;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  return true;
}

// Adds the rows of group 0 (vector values) or 1 (pairs): `nh` listed sources, or (`one` false) all that hit.
template <int NPTS, int NT, bool PAIRS>
FHD_DEV void plane_add_group(int* acc, int pitch, const GridDev& g, const PlaneSrc& P, int tid, int z, int C, PlaneLds& L,
                             bool one, int nh, float scale2) {
  const SpreadGroup& G = P.grp[PAIRS];
  const PlaneRuns r = plane_runs(L, PAIRS);
  const int all = r.total(), lane = tid & 63, wave = uniform(tid >> 6);
  int n = 0, b = one ? wave * 64 : wave * 128;
  for (;;) {
    int j = -1;
    if (one) {
      if (b >= nh) break;
      if (b + lane < nh) j = r.slot(L.list[PAIRS ? kListCap - 1 - b - lane : b + lane]);
      b += NT;
    } else if (!plane_gather<NPTS, NT, PAIRS>(G, r, all, lane, L.slots + wave * (kListCap / 2 / (NT / 64)), g.mz, z, C, b, n, j)) {
      break;
    }
    if (j >= 0) {
      if (PAIRS) plane_add_pair<NPTS>(acc, pitch, g, L, G, j, z, C, scale2);
      else plane_add<NPTS>(acc, pitch, g, L, G, j, z, C, scale2);
    }
  }
}

// Accumulates the plane into acc (`words` words, row pitch `pitch`, cleared here) and returns whether a
// second call (REST) is to follow, for what the rounding of this one's integers left over: the caller
// adds the sums of both, times plane_unit.  Every lane of the workgroup calls it; the plane is complete
// (barrier passed) on return.
template <int NPTS, int NT, bool REST>
FHD_DEV bool plane_spread(int* acc, int words, int pitch, const GridDev& g, const PlaneSrc& P, int z, int C,
                          PlaneLds& L) {
  int tid = threadIdx.x;

  const int lane = tid & 63;
  const int bx = (g.mx + 3) >> 2, by = (g.my + 3) >> 2;
  // each block's values (x), pairs (y) and largest value (z, float bits), until the scales are known
  int4* const block = reinterpret_cast<int4*>(acc);
  const int head = !REST ? 4 * bx * by : 0;  // a block has four words of the plane at least
  if (tid < 12 && tid < 6 * P.ngroups) L.runs[tid >= 6][tid % 6] = run_bound(P.t, P.grp[tid >= 6], z, tid % 6);
  for (int e = tid; e < head; e += NT) acc[e] = 0;
  if (tid < 2) L.n[tid] = 0;
  if (tid == 0) L.kept = 0;
  if (!REST && tid == 0) L.most = L.top = L.more = L.bad = 0;
  __syncthreads();
  const bool two = P.ngroups > 1;
  // sources in reach, of which the plane is hit by about five in fourteen (five planes of the one or two
  // layers of eight): with three times what the list holds they are not listed
  const int n0 = plane_runs(L, 0).total(), n1 = two ? plane_runs(L, 1).total() : 0;
  const bool listed = n0 + n1 <= 3 * kListCap;
  int4* const pairs = !REST ? block : nullptr;
  if (listed) {
    const PlaneRuns r0 = plane_runs(L, 0);
    // the first keys of both groups are in flight at once
    constexpr int K = 4;
    unsigned k0[K], k1[K];
    plane_keys<NT, K>(P.grp[0], r0, tid, 0, n0, k0);
    PlaneRuns r1 = r0;
    if (two) {
      r1 = plane_runs(L, 1);
      plane_keys<NT, K>(P.grp[1], r1, tid, 0, n1, k1);
    }
    plane_test<NT, K>(g, P, 0, tid, k0, 0, z, C, L, nullptr);
    if (n0 > K * NT) plane_scan<NT>(g, P, 0, tid, r0, K * NT, n0, z, C, L, nullptr);
    if (two) {
      plane_test<NT, K>(g, P, 1, tid, k1, 0, z, C, L, pairs);
      if (n1 > K * NT) plane_scan<NT>(g, P, 1, tid, r1, K * NT, n1, z, C, L, pairs);
    }
  }
  __syncthreads();
  const int nhit0 = listed ? uniform(L.n[0]) : n0, nhit1 = listed ? uniform(L.n[1]) : n1;  // at most
  const bool one = listed && nhit0 + nhit1 <= kListCap;
  const auto clear = [&](int from, int to) {  // both multiples of 4, or the plane's end
    int4* acc4 = reinterpret_cast<int4*>(acc);
    for (int e = from / 4 + tid; e < to / 4; e += NT) acc4[e] = make_int4(0, 0, 0, 0);
    if (tid < (to & 3)) acc[(to & ~3) + tid] = 0;
  };
  // Group 0 holds vector values: those of its hits enter their blocks' counts and bounds, and the listed
  // hits without one leave the list.
  {
    const SpreadGroup& G = P.grp[0];
    const PlaneRuns r = plane_runs(L, 0);
    const float drift = fabsf(G.drift) * (C == 0 ? g.idx : C == 1 ? g.idy : g.idz);
    const auto enter = [&](float v, unsigned key) {
      const float a = fabsf(v) + drift;
      const bool fine = a <= 3.0e38f;
      if (!fine) L.bad = 1;
      if (!REST) {
        atomicAdd(&block[key >> 16].x, 1);
        atomicMax(&block[key >> 16].z, __float_as_int(fine ? a : 3.0e38f));
      }
    };
    if (one) {
      constexpr int K = (kListCap + NT - 1) / NT;
      constexpr int KF = 3;  // values of a lane in flight at once
      unsigned short e[KF];
      unsigned key[KF];
      float v[KF];
      // rounds of KF x NT entries, each read in full before the shorter list overwrites it
      for (int k0 = 0; k0 < K * NT && (k0 == 0 || k0 < nhit0); k0 += KF * NT) {
#pragma unroll
        for (int k = 0; k < KF; ++k) {
          const int i = k0 + tid + k * NT;
          v[k] = 0.0f;
          if (i < nhit0) {
            e[k] = L.list[i];
            const int j = r.slot(e[k]);
            key[k] = G.key[j];
            v[k] = src_value(G, j, C);
          }
        }
        if (k0 == 0) clear(head, words);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < KF; ++k) {
          const bool keep = k0 + tid + k * NT < nhit0 && (v[k] != 0.0f || drift != 0.0f);
          if (keep) enter(v[k], key[k]);
          list_keep(L, lane, keep, e[k]);
        }
      }
    } else {
      clear(head, words);
      constexpr int K = 4;
      for (int b = 0; b < n0; b += K * NT) {
        unsigned key[K];
        float v[K];
        plane_keys<NT, K>(G, r, tid, b, n0, key);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          if (!key_hits(key[k], G, z, g.mz, NPTS, C == 2)) key[k] = ~0u;
          v[k] = key[k] != ~0u ? src_value(G, r.slot(b + k * NT + tid), C) : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
          if (key[k] != ~0u && (v[k] != 0.0f || drift != 0.0f)) {
            enter(v[k], key[k]);
            L.kept = 1;
          }
      }
      if (two && !listed && !REST) {
        const SpreadGroup& G1 = P.grp[1];
        const PlaneRuns r1 = plane_runs(L, 1);
        for (int b = 0; b < n1; b += K * NT) {
          unsigned key[K];
          plane_keys<NT, K>(G1, r1, tid, b, n1, key);
#pragma unroll
          for (int k = 0; k < K; ++k)
            if (key_hits(key[k], G1, z, g.mz, NPTS, C == 2)) atomicAdd(&block[key[k] >> 16].y, 1);
        }
      }
    }
  }
  __syncthreads();
  const int nval = uniform(L.kept);
  if (!REST) {
    // The scale of a block's nodes: their sources lie in cells at most 3 away, so in the blocks around it,
    // unless a pair is displaced by more than a cell along x or y (then the plane has one scale).
    const PlaneBounds bounds = plane_bounds<NPTS>(g, P, C);
    if (tid == 0 && two && !(5.8f * fabsf(P.grp[1].coef) <= 3.0e38f)) L.bad = 1;
    bool more = false;
    int n_most = 0, t_most = 0;
    for (int e = tid; e < bx * by; e += NT) {
      const int y = e / bx, x = e - y * bx;
      // the rows and columns around it, each once: of two there is no third, of one no second
      const int ys[3] = {y, y == 0 ? by - 1 : y - 1, y == by - 1 ? 0 : y + 1};
      const int xs[3] = {x, x == 0 ? bx - 1 : x - 1, x == bx - 1 ? 0 : x + 1};
      int4 around[3][3];
#pragma unroll
      for (int dy = 0; dy < 3; ++dy)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) around[dy][dx] = block[xs[dx] + bx * ys[dy]];
      int nf = 0, np = 0, t = 0;
#pragma unroll
      for (int dy = 0; dy < 3; ++dy)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          const bool in = dy < by && dx < bx;
          nf += in ? around[dy][dx].x : 0;
          np += in ? around[dy][dx].y : 0;
          t = max(t, around[dy][dx].z);
        }
      if (P.near) L.scale[e] = (signed char)block_scale(bounds, nf, np, __int_as_float(t), more);
      n_most = max(n_most, nf + 2 * np);
      t_most = max(t_most, t);
    }
    n_most = wave_max_i32(P.near ? n_most : nhit0 + 2 * nhit1);
    if (lane == 0) atomicMax(&L.most, n_most);
    if (!P.near) {
      t_most = wave_max_i32(t_most);
      if (lane == 0) atomicMax(&L.top, t_most);
    }
    if (more) L.more = 1;
    __syncthreads();
    clear(0, head);
    if (!P.near) {
      const int x = block_scale(bounds, nval ? nhit0 : 0, nhit1, __int_as_float(L.top), more);
      for (int e = tid; e < bx * by; e += NT) L.scale[e] = (signed char)x;
      if (more) L.more = 1;
    }
    __syncthreads();
  }
  const float scale2 = !REST ? 0.0f : ldexpf(1.0f, rest_exp(uniform(L.most)));
  if (nval) plane_add_group<NPTS, NT, false>(acc, pitch, g, P, tid, z, C, L, one, nval, scale2);
  if (two) plane_add_group<NPTS, NT, true>(acc, pitch, g, P, tid, z, C, L, one, nhit1, scale2);
  __syncthreads();
  return !REST && uniform(L.more) != 0 && uniform(L.bad) == 0;
}
template <int NT, bool REST>
FHD_DEV bool plane_spread(int* acc, int words, int pitch, const GridDev& g, const PlaneSrc& P, int z, int C,
                          PlaneLds& L) {
  return P.kernel_points == 4 ? plane_spread<4, NT, REST>(acc, words, pitch, g, P, z, C, L)
                              : plane_spread<3, NT, REST>(acc, words, pitch, g, P, z, C, L);
}

// What the integers at node (x, y) are to be multiplied by, those of the second call by `rest` times as much.  A plane
// with an overflowed or NaN source is written non-finite, which the interpolation flags.
struct PlaneUnit {
  float coef, rest;
  int nbx;
  FHD_DEV float at(const PlaneLds& L, int x, int y) const { return ldexpf(coef, -L.scale[(x >> 2) + nbx * (y >> 2)]); }
};
FHD_DEV PlaneUnit plane_unit(const PlaneLds& L, const PlaneSrc& P, const GridDev& g) {
  return PlaneUnit{uniform(L.bad) ? __builtin_inff() : P.out_coef, ldexpf(1.0f, -rest_exp(uniform(L.most))), (g.mx + 3) >> 2};
}

}  // namespace fhd
