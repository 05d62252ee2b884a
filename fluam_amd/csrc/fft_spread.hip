// fft_spread.hip -- the forward xy pass with spreading for the plane shapes of fft_fast.hip: mx x my
// with both lengths in {16, 24, 32, 48, 64} or mx = my in {96, 128}.  Compiled once per mx
// (FHD_SPREAD_MX): these are the largest kernels of the library.
// The runtime-size and the size-specialised FFT kernels have to give the same bits (a replica runs
// on the one alone and on the other in a merged batch), so the compiler must not choose which
// products become fused multiply-adds: the fused ones are written out.
#pragma clang fp contract(off)
#include "fft_stages.h"

namespace fhd {

FHD_KERNEL_PAIR_OCC((template <int MX, int MY, int NT>), NT, 8, k_spread_fftA, FftSpread,
                    body_fftA<MX, MY, NT, MX == MY ? square_plan(MX) % 3 : 0, MX == MY ? square_plan(MX) / 3 : 0, true>(
                        a.p.f, a.p.in, a.p.spec, b, &a.s))

// Lanes per plane workgroup as in the plain pass of a context launched alone.  Merged batches hold the planes
// with both edges in the list above as runtime-size passes (merged_plane; the same radices and written-out
// fused operations give the same bits), so only the larger squares have a batched form.
template <int MX, int MY>
static bool launch_plane(const FftSpread& x, hipStream_t s) {
  constexpr int NT = MX * MY >= 64 * 64 ? 1024 : 256;
  BatchedFn batched = nullptr;
  if constexpr (MX > 64) batched = k_spread_fftA_b<MX, MY, NT>;
  launch(k_spread_fftA<MX, MY, NT>, batched, FAM_FFT_XY_FWD, dim3(x.p.f.g.mz, x.p.f.ncomp), NT, x, s);
  return true;
}
template <int MX>
bool launch_spread_rect(const FftSpread& x, hipStream_t s) {
  if constexpr (MX > 64) {
    return x.p.f.g.my == MX && launch_plane<MX, MX>(x, s);
  } else {
    switch (x.p.f.g.my) {
      case 16: return launch_plane<MX, 16>(x, s);
      case 24: return launch_plane<MX, 24>(x, s);
      case 32: return launch_plane<MX, 32>(x, s);
      case 48: return launch_plane<MX, 48>(x, s);
      case 64: return launch_plane<MX, 64>(x, s);
      default: return false;
    }
  }
}
template bool launch_spread_rect<FHD_SPREAD_MX>(const FftSpread&, hipStream_t);

}  // namespace fhd
