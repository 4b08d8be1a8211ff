// fixed_f32x_single2.hip -- compile-time plans, FP32 storage under FP64
// arithmetic, single pass: part 3 of 4 of the fast lengths other than powers
// of two.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// median 1.44x over the runtime-planned pass (7500 178 -> 128 us); 300, 360, 450,
// 675 and 768 lose 3-21 %.
#include "fixed.h"

namespace sfft {
namespace {
using X = Stored<StoreF32>;
const FixedC2C<X, 75, 5, 51, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5> c75;
const FixedC2C<X, 96, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6> c96;
const FixedC2C<X, 125, 9, 28, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5> c125;
const FixedC2C<X, 150, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10> c150;
const FixedC2C<X, 192, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12> c192;
const FixedC2C<X, 240, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15> c240;
const FixedC2C<X, 288, 24, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 2> c288;
const FixedC2C<X, 384, 26, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8, 3> c384;
const FixedC2C<X, 480, 32, 8, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 2> c480;
const FixedC2C<X, 576, 48, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6, 6> c576;
const FixedC2C<X, 648, 72, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 6> c648;
const FixedC2C<X, 800, 80, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 8> c800;
const FixedC2C<X, 960, 64, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 4> c960;
const FixedC2C<X, 1125, 75, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5> c1125;
const FixedC2C<X, 1250, 84, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5, 2> c1250;
const FixedC2C<X, 1440, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 10> c1440;
const FixedC2C<X, 1600, 160, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 10, 10> c1600;
const FixedC2C<X, 1875, 125, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5, 5> c1875;
const FixedC2C<X, 2025, 135, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3, 3> c2025;
const FixedC2C<X, 2304, 192, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 12> c2304;
const FixedC2C<X, 2560, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 10> c2560;
const FixedC2C<X, 2916, 324, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 6, 6> c2916;
const FixedC2C<X, 3200, 214, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8, 5, 5> c3200;
const FixedC2C<X, 3600, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15> c3600;
const FixedC2C<X, 3888, 432, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 6, 6> c3888;
const FixedC2C<X, 4374, 486, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 6> c4374;
const FixedC2C<X, 4860, 405, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 3, 3> c4860;
const FixedC2C<X, 5400, 360, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8, 3> c5400;
const FixedC2C<X, 6000, 400, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5, 5> c6000;
const FixedC2C<X, 6400, 427, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 5, 5> c6400;
const FixedC2C<X, 6912, 461, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 3, 3, 3> c6912;
const FixedC2C<X, 7680, 512, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15, 2> c7680;
}  // namespace
}  // namespace sfft
