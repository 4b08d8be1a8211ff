// fixed_f32x_single1.hip -- compile-time plans, FP32 storage under FP64
// arithmetic, single pass: part 2 of 4 of the fast lengths other than powers
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
const FixedC2C<X, 72, 6, 43, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6> c72;
const FixedC2C<X, 90, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9> c90;
const FixedC2C<X, 120, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8> c120;
const FixedC2C<X, 144, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12> c144;
const FixedC2C<X, 180, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12> c180;
const FixedC2C<X, 225, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15> c225;
const FixedC2C<X, 270, 23, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 3> c270;
const FixedC2C<X, 375, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5> c375;
const FixedC2C<X, 432, 36, 7, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6, 6> c432;
const FixedC2C<X, 540, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6> c540;
const FixedC2C<X, 640, 43, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8, 5> c640;
const FixedC2C<X, 750, 75, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10, 5> c750;
const FixedC2C<X, 900, 60, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 4> c900;
const FixedC2C<X, 1080, 90, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 6> c1080;
const FixedC2C<X, 1215, 135, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 9, 9> c1215;
const FixedC2C<X, 1350, 113, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6> c1350;
const FixedC2C<X, 1536, 128, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 6> c1536;
const FixedC2C<X, 1800, 120, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8> c1800;
const FixedC2C<X, 2000, 134, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5, 5, 5> c2000;
const FixedC2C<X, 2250, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 10> c2250;
const FixedC2C<X, 2500, 250, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 5, 5> c2500;
const FixedC2C<X, 2880, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 12> c2880;
const FixedC2C<X, 3125, 209, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5, 5> c3125;
const FixedC2C<X, 3456, 288, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6, 6, 6> c3456;
const FixedC2C<X, 3840, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15> c3840;
const FixedC2C<X, 4320, 360, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6, 5> c4320;
const FixedC2C<X, 4800, 320, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5, 4> c4800;
const FixedC2C<X, 5184, 432, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6, 6> c5184;
const FixedC2C<X, 5832, 486, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 6, 6, 6, 3, 3, 3> c5832;
const FixedC2C<X, 6250, 417, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5, 5, 2> c6250;
const FixedC2C<X, 6750, 450, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 2> c6750;
const FixedC2C<X, 7500, 500, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5, 5, 4> c7500;
}  // namespace
}  // namespace sfft
