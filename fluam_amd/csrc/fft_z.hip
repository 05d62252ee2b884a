// fft_z.hip -- the z pass for column lengths that are a product of two radices (every 2^a 3^b from
// 16 to 256 but 162, 216 and 243, which take fft.hip's z pass, like the lengths below 16).
//
// FFT along z, operator, inverse FFT.  With N = R1 R2 the transform is two Stockham stages: the first
// takes its elements straight from global memory, the last of the inverse stores straight to it, and
// the second stages of both directions read and write the same elements, so a column crosses LDS
// eight times with four barriers (twelve and ten when load, stages, operator and store each staged
// through LDS).  Every phase spreads its own work over all lanes.  The operator is one rolled loop:
// keeping the modes in registers between the stages instead needs it unrolled R2 times, and fetching
// 25 KB of straight-line code that no wave has run before took longer than the LDS crossings
// (128^3 Stokes 36 us per launch, this form 26.4).  Bound by the LDS crossings and, with noise, by the
// Philox and Box-Muller arithmetic, with the memory round trips of the ends under other workgroups.
// Per launch (HIP events, which add about 4 us), staged through LDS and now: Stokes 128^3 31 -> 26.4,
// 128 x 128 x 256 69 -> 46.6, 128 x 64 x 32 13 -> 10.0, 32^3 9.6 -> 8.0; 108 x 54 x 72 19 -> 11.0.
#pragma clang fp contract(off)  // same bits from every instance (fft_fast.hip)
#include "fhd_device.h"
#include "fhd_kernels.h"
#include "fft_common.h"

namespace fhd {

// First radix, the larger one; the second is n / zr1(n).  0: not a product of two.
constexpr int zr1(int n) {
  switch (n) {
    case 16: return 4;
    case 18: case 24: case 36: return 6;
    case 32: case 48: case 64: return 8;
    case 27: case 54: case 72: case 81: return 9;
    case 96: case 108: case 144: return 12;
    case 128: case 192: case 256: return 16;
    default: return 0;
  }
}
// The lanes of a wave take consecutive lines in the first stage and consecutive butterflies of a
// line in the second: odd line strides that are R1 + 1 (or 2) past a multiple of the 32 banks of
// 8 bytes keep both free of conflicts but for the odd pair.
constexpr int zstride(int n) {
  const int want = (zr1(n) + 1) | 1;
  int ls = n;
  while (ls % 32 != want % 32) ++ls;
  return ls;
}
template <int N, int LINES> struct ZLds {
  float2 buf[LINES * zstride(N)];
  float2 tw[N], ez[N];
  float gz[N];
};

template <int N, int NT, int LINES>
FHD_DEV void body_fftz(const FftPass& x, const Blk& b, ZLds<N, LINES>& L) {
  constexpr int R1 = zr1(N), R2 = N / R1, LS = zstride(N);
  static_assert(LINES * R2 <= NT, "one butterfly per lane in the first stage");
  const FftArgs& a = x.f;
  const int T = x.T, P = a.g.P, my = a.g.my;
  // neighbouring column tiles share the 128-byte lines of each z row: keep them on one XCD
  const int item = xcd_item(b.x + b.nx * b.y, b.nx * b.ny);
  const int ky = item / b.nx, tile = item - ky * b.nx;
  const int wide = P / b.nx, rem = P - wide * b.nx;
  const int kx0 = tile * wide + min(tile, rem), w = wide + (tile < rem ? 1 : 0);
  const int cs = my * N * P;  // 3 cs: far below 2^31 at every size
  float2* const base = x.spec + (size_t)ky * N * P + kx0;
  const int tid = threadIdx.x, lines = a.ncomp * T;
  {
    // first stage: butterfly j of line l = (component c, column t), elements z = j + r R2
    const int j = fast_div(tid, x.ml), l = tid - j * lines, c = fast_div(l, x.mt), t = l - c * T;
    const bool on = j < R2 && t < w;
    const float2* const col = base + c * cs + j * P + t;
    float2* const line = L.buf + l * LS + j * R1;
    float2 v[R1];
    if (a.zmode != 2 && on) {
#pragma unroll
      for (int r = 0; r < R1; ++r) v[r] = col[r * (R2 * P)];
    }
    for (int i = tid; i < N; i += NT) {
      L.tw[i] = a.twz[i];
      L.ez[i] = a.ez[i];
      L.gz[i] = a.gz[i];
    }
    if (a.zmode != 2 && on) {
      Dft<R1>::run(v, -1.0f);
#pragma unroll
      for (int r = 0; r < R1; ++r) line[r] = v[r];
    }
  }
  __syncthreads();
  // second stage: butterfly j of line l, elements and modes j + r R1
  if (a.zmode == 0) {
    for (int i = tid; i < lines * R1; i += NT) {
      const int l = i / R1, j = i - l * R1;
      float2* const row = L.buf + l * LS + j;
      float2 v[R2];
#pragma unroll
      for (int r = 0; r < R2; ++r) v[r] = r ? cmul(row[r * R1], L.tw[j * r]) : row[0];
      Dft<R2>::run(v, -1.0f);
#pragma unroll
      for (int r = 0; r < R2; ++r) row[r * R1] = v[r];
    }
    __syncthreads();
    const float gy = a.gy[ky];
    const float2 ey = a.ey[ky];
    const Key key = a.knoise ? resolve_key(a.key) : a.key;
#pragma unroll 1
    for (int i = tid; i < N * w; i += NT) {
      const int t = i / N, z = i - t * N, kx = kx0 + t;
      float2* const m = L.buf + t * LS + z;
      float2 b0 = m[0], b1 = m[T * LS], b2 = m[2 * T * LS];
      solve_mode(a, key, kx, ky, z, a.gx[kx], gy, L.gz[z], a.ex[kx], ey, L.ez[z], b0, b1, b2);
      m[0] = b0;
      m[T * LS] = b1;
      m[2 * T * LS] = b2;
    }
    __syncthreads();
    for (int i = tid; i < lines * R1; i += NT) {
      const int l = i / R1, j = i - l * R1;
      float2* const row = L.buf + l * LS + j;
      float2 v[R2];
#pragma unroll
      for (int r = 0; r < R2; ++r) v[r] = row[r * R1];
      Dft<R2>::run(v, 1.0f);
#pragma unroll
      for (int r = 0; r < R2; ++r) row[r * R1] = r ? cmul(v[r], cconj(L.tw[j * r])) : v[r];
    }
    __syncthreads();
  } else {
    // one direction alone: the modes lie in global memory, consecutive lanes take consecutive columns
    for (int i = tid; i < lines * R1; i += NT) {
      const int j = fast_div(i, x.ml), l = i - j * lines, c = fast_div(l, x.mt), t = l - c * T;
      if (t >= w) continue;
      float2* const row = L.buf + l * LS + j;
      float2* const modes = base + c * cs + j * P + t;
      float2 v[R2];
      if (a.zmode == 1) {
#pragma unroll
        for (int r = 0; r < R2; ++r) v[r] = r ? cmul(row[r * R1], L.tw[j * r]) : row[0];
        Dft<R2>::run(v, -1.0f);
#pragma unroll
        for (int r = 0; r < R2; ++r) modes[r * (R1 * P)] = v[r];
      } else {
#pragma unroll
        for (int r = 0; r < R2; ++r) v[r] = modes[r * (R1 * P)];
        Dft<R2>::run(v, 1.0f);
#pragma unroll
        for (int r = 0; r < R2; ++r) row[r * R1] = r ? cmul(v[r], cconj(L.tw[j * r])) : v[r];
      }
    }
    if (a.zmode == 1) return;
    __syncthreads();
  }
  // the lane index, opaque to the compiler: the first stage's addresses are computed again rather than
  // kept in registers (64 of them let the CU hold all its waves)
  int again = threadIdx.x;
  asm volatile("" : "+v"(again));
  const int j = fast_div(again, x.ml), l = again - j * lines, c = fast_div(l, x.mt), t = l - c * T;
  if (j < R2 && t < w) {
    float2* const col = base + c * cs + j * P + t;
    const float2* const line = L.buf + l * LS + j * R1;
    float2 v[R1];
#pragma unroll
    for (int r = 0; r < R1; ++r) v[r] = line[r];
    Dft<R1>::run(v, 1.0f);
#pragma unroll
    for (int r = 0; r < R1; ++r) col[r * (R2 * P)] = v[r];
  }
}

// Lanes of a workgroup with 3 T lines: a butterfly of the second stage each.
constexpr int zlanes(int n, int T) { return (3 * T * zr1(n) + 63) / 64 * 64; }
template <int N, int T>
FHD_BODY void body_z(const FftPass& x, const Blk& b) {
  __shared__ ZLds<N, 3 * T> L;
  body_fftz<N, zlanes(N, T), 3 * T>(x, b, L);
}
FHD_KERNEL_PAIR_OCC((template <int N, int T>), zlanes(N, T), 8, k_fftz, FftPass, body_z<N, T>(a, b))

// Merged batches: one kernel for the lengths of their usual boxes, so that replicas of different
// lengths share a dispatch; every workgroup runs the code of its length.
constexpr int kMergedLanes = 256;
constexpr bool zmerged(int n) { return n == 16 || n == 24 || n == 32 || n == 48 || n == 64; }
template <int N> using ZMerged = ZLds<N, kMergedLanes / zr1(N)>;
constexpr size_t zmost() {
  size_t m = 0;
  for (size_t n : {sizeof(ZMerged<16>), sizeof(ZMerged<24>), sizeof(ZMerged<32>), sizeof(ZMerged<48>), sizeof(ZMerged<64>)})
    if (n > m) m = n;
  return m;
}
FHD_BODY void body_z_merged(const FftPass& x, const Blk& b) {
  __shared__ __align__(16) unsigned char raw[zmost()];
  switch (x.f.g.mz) {
#define FHD_Z(n) case n: body_fftz<n, kMergedLanes, kMergedLanes / zr1(n)>(x, b, *reinterpret_cast<ZMerged<n>*>(raw)); break
    FHD_Z(16);
    FHD_Z(24);
    FHD_Z(32);
    FHD_Z(48);
    FHD_Z(64);
#undef FHD_Z
  }
}
FHD_KERNEL_PAIR_OCC((), kMergedLanes, 8, k_fftz_merged, FftPass, body_z_merged(a, b))

// The lengths of the merged kernel have no batched form of their own.
template <int N, int T>
static BatchedFn z_batched() {
  if constexpr (zmerged(N)) return nullptr;
  else return k_fftz_b<N, T>;
}

int fast_z_columns(int mz, int want) {
  if (mz > 256 || !zr1(mz)) return 0;
  return want <= 2 ? 2 : want <= 4 ? 4 : 8;  // beyond 8 the workgroups are too few and too large
}

template <int N>
static bool launch_z(const FftArgs& a, float2* spec, hipStream_t s) {
  const bool merged = t_recorder && zmerged(N);
  const int tile = fast_z_columns(N, a.btile);
  const int most = merged ? kMergedLanes / zr1(N) / a.ncomp : tile * 3 / a.ncomp;
  const int ntile = (a.g.P + most - 1) / most, T = (a.g.P + ntile - 1) / ntile;
  const FftPass x{a, nullptr, spec, nullptr, nullptr, 0.0f, 0.0f, T, fast_div_magic(T), fast_div_magic(a.ncomp * T)};
  const dim3 grid(ntile, a.g.my);
  if constexpr (zmerged(N)) {
    if (merged) {
      launch(k_fftz_merged, k_fftz_merged_b, FAM_FFT_Z, grid, kMergedLanes, x, s);
      return true;
    }
  }
#define FHD_Z(t) launch(k_fftz<N, t>, z_batched<N, t>(), FAM_FFT_Z, grid, zlanes(N, t), x, s)
  if (tile == 2) FHD_Z(2);
  else if (tile == 4) FHD_Z(4);
  else FHD_Z(8);
#undef FHD_Z
  return true;
}

bool fast_fft_z_solve(const FftArgs& a, float2* spec, hipStream_t s) {
  switch (a.g.mz) {
#define FHD_Z(n) case n: return launch_z<n>(a, spec, s)
    FHD_Z(16); FHD_Z(18); FHD_Z(24); FHD_Z(27); FHD_Z(32); FHD_Z(36); FHD_Z(48); FHD_Z(54); FHD_Z(64);
    FHD_Z(72); FHD_Z(81); FHD_Z(96); FHD_Z(108); FHD_Z(128); FHD_Z(144); FHD_Z(192); FHD_Z(256);
#undef FHD_Z
    default: return false;
  }
}

}  // namespace fhd
