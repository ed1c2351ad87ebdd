// Row and pencil kernels for the other axis lengths: every length from 32 to
// 1024 without a prime factor above 7 that KW_FAST_SIZES does not list
// (KW_LEN_SIZES).  They are the templates of kw_xrow.inc and kw_pencil.inc at one
// workgroup size and radix plan 4, without the batched wrappers and the variants
// that the autotuner tries.  The runtime-radix kernels of kw_kernels.hip, which
// ran these lengths before and still run shorter and longer axes, index every
// butterfly input and output by runtime division, copy a tile in and out of LDS
// around the transform and hold two or three LDS buffers: a step of 216x150x189
// took 1773 us, with these 502; 105x63x81 340 -> 106; 2-D 270x180 254 -> 59.
//
// Compiled once for each length, with KW_LENGTH defined: the runtime loads a
// translation unit's device code as a whole when one of its kernels is first
// launched, about 10 ms for 14 lengths and 2 ms for one, and a run has up to three
// of them (a whole process of the executable, 14 lengths a unit -> one: 270x180,
// 50 steps 124 -> 93 ms; 216x150x189, 10 steps 201 -> 157; with the runtime-radix
// kernels 99 and 162).
#ifndef KW_LENGTH
#error "KW_LENGTH: one of KW_LEN_SIZES"
#endif
#include "kw_axisym.inc"
#include "kw_pencil.inc"
#include "kw_xrow.inc"

namespace kw {

// Pencil workgroup sizes by the rules of the tuned lengths.  Last axis: 512 threads
// from 384 points up and 1024, whose tile is the CU's, from 512 up; us a launch at
// 128x128xN with 256 / 512 / 1024 threads: 189 points 21.7 / 19.5 / 24.8, 252 30.5 /
// 29.4 / 26.3, 350 39.2 / 39.9 / 40.3, 448 53.7 / 42.7 / 42.2, 525 75.9 / 63.8 / 69.3,
// 640 97 / 85 / 76, 1000 284 / 182 / 120; below 512 some lengths would run up to a
// third faster with more threads (270 38.2 / 26.2 / 30.4, 392 68.8 / 50.8 / 39.4).
// Y pass: 512 from 256 up, and 1024 where no two workgroups of 512 with their
// tables fit a CU; at 128xNx128: 189 15.8 / 14.8 / 16.9, 252 21.1 / 18.6 / 19.4, 270
// 21.4 / 18.4 / 20.7, 392 34.6 / 26.6 / 27.1, 525 51.7 / 41.6 / 37.3, 640 61.5 / 53.0 /
// 48.7, 1000 105 / 79 / 80.
constexpr int len_last_nt(int n) { return n >= 512 ? 1024 : n >= 384 ? 512 : 256; }
template <int N>
constexpr int len_y_nt() {
  return N < 256 ? 256 : PencilCfg<N, 512, 4>::lds(2) <= 81920 ? 512 : 1024;
}

template <int N>
constexpr RadialFn len_radial() {
  if constexpr (N % 2 == 0)
    return &radial_t<N>;
  else
    return nullptr;
}

static const LenKernels* len_entry() {
  constexpr int N = KW_LENGTH, RNT = 256, YNT = len_y_nt<N>(), LNT = len_last_nt(N);
  static const LenKernels k{&xvel<N, RNT>, &xdens<N, RNT>, &xpres<N, RNT>, &xinit<N, RNT>, &xsrc<N, RNT>,
                            &xc2r<N, RNT>, &ypass_t<N, YNT, 4>, &ygrad_t<N, YNT, 4>, &last_t<N, LNT, 4>,
                            &last_launch<N, narrow_nt(N), 4, false, kNarrowTX>, len_radial<N>(), RNT, YNT, LNT};
  return &k;
}

#define KW_LEN_NAME(n) len_kernels_##n
#define KW_LEN_ENTRY(n) KW_LEN_NAME(n)
const LenKernels* KW_LEN_ENTRY(KW_LENGTH)() { return len_entry(); }

}  // namespace kw
