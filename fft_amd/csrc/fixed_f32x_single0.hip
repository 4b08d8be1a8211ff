// fixed_f32x_single0.hip -- compile-time plans, FP32 storage under FP64
// arithmetic, single pass: part 1 of 4 of the fast lengths other than powers
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
const FixedC2C<X, 64, 4, 64, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 4> c64;
const FixedC2C<X, 81, 9, 28, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9> c81;
const FixedC2C<X, 108, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9> c108;
const FixedC2C<X, 135, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 9> c135;
const FixedC2C<X, 162, 18, 14, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 2> c162;
const FixedC2C<X, 216, 18, 14, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 6, 6, 6> c216;
const FixedC2C<X, 250, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 5, 5> c250;
const FixedC2C<X, 324, 36, 7, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 6, 6> c324;
const FixedC2C<X, 405, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 5> c405;
const FixedC2C<X, 500, 50, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 5> c500;
const FixedC2C<X, 625, 42, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5> c625;
const FixedC2C<X, 729, 81, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9> c729;
const FixedC2C<X, 864, 72, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6> c864;
const FixedC2C<X, 1000, 100, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10> c1000;
const FixedC2C<X, 1200, 80, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5> c1200;
const FixedC2C<X, 1296, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 9> c1296;
const FixedC2C<X, 1500, 150, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10, 10> c1500;
const FixedC2C<X, 1728, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 12> c1728;
const FixedC2C<X, 1944, 216, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 6, 6, 6> c1944;
const FixedC2C<X, 2187, 243, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 3> c2187;
const FixedC2C<X, 2430, 270, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9, 9, 3> c2430;
const FixedC2C<X, 2700, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 12> c2700;
const FixedC2C<X, 3072, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 12> c3072;
const FixedC2C<X, 3375, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15> c3375;
const FixedC2C<X, 3750, 250, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5, 5, 2> c3750;
const FixedC2C<X, 4050, 338, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6, 3> c4050;
const FixedC2C<X, 4608, 384, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 12, 2> c4608;
const FixedC2C<X, 5120, 342, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 5, 4> c5120;
const FixedC2C<X, 5760, 384, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 8, 3> c5760;
const FixedC2C<X, 6144, 410, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 8, 3> c6144;
const FixedC2C<X, 6561, 438, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 3, 3, 3, 3, 3, 3, 3, 3> c6561;
const FixedC2C<X, 7290, 486, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 3, 3, 3, 3, 3, 2> c7290;
}  // namespace
}  // namespace sfft
