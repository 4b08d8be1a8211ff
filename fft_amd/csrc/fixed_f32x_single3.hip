// fixed_f32x_single3.hip -- compile-time plans, FP32 storage under FP64
// arithmetic, single pass: part 4 of 4 of the fast lengths other than powers
// of two.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// median 1.44x over the runtime-planned pass (7500 178 -> 128 us); 300, 360, 450,
// 675 and 768 lose 3-21 %.
// (Half-size blocks, a twiddle choice, the seventh Sched value, or kPersist: lengths
// that one group per block had slowed; figures at the top of fixed.h.)
#include "fixed.h"

namespace sfft {
namespace {
using X = Stored<StoreF32>;
const FixedC2C<X, 80, 6, 43, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5> c80;
const FixedC2C<X, 100, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10> c100;
const FixedC2C<X, 128, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8> c128;
const FixedC2C<X, 160, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 10> c160;
const FixedC2C<X, 200, 14, 18, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 8, 5, 5> c200;
const FixedC2C<X, 243, 27, 9, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 3> c243;
const FixedC2C<X, 320, 22, 12, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5, 4> c320;
const FixedC2C<X, 400, 27, 9, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5, 5> c400;
const FixedC2C<X, 486, 54, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 6> c486;
const FixedC2C<X, 600, 40, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 5> c600;
const FixedC2C<X, 720, 48, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 3> c720;
const FixedC2C<X, 810, 90, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9, 9> c810;
const FixedC2C<X, 972, 108, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 9> c972;
const FixedC2C<X, 1152, 96, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 6> c1152;
const FixedC2C<X, 1280, 86, 2, Sched<0, 0, 0, 0, kLdsPadShift, 0, 1>, 0, 16, 16, 5> c1280;
const FixedC2C<X, 1458, 162, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 2> c1458;
const FixedC2C<X, 1620, 180, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 9> c1620;
const FixedC2C<X, 1920, 128, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 8> c1920;
const FixedC2C<X, 2160, 180, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 12> c2160;
const FixedC2C<X, 2400, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 10> c2400;
const FixedC2C<X, 2592, 216, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6, 6, 6> c2592;
const FixedC2C<X, 3000, 200, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 5, 5> c3000;
const FixedC2C<X, 3240, 270, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 6> c3240;
const FixedC2C<X, 3645, 405, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 5> c3645;
const FixedC2C<X, 4000, 400, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10, 4> c4000;
const FixedC2C<X, 4500, 300, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5, 4> c4500;
const FixedC2C<X, 5000, 500, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10, 5> c5000;
const FixedC2C<X, 5625, 375, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5, 5> c5625;
const FixedC2C<X, 6075, 405, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3, 3, 3> c6075;
const FixedC2C<X, 6480, 432, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 3, 3, 3> c6480;
const FixedC2C<X, 7200, 480, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15, 2> c7200;
}  // namespace
}  // namespace sfft
