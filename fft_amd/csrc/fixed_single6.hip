// fixed_single6.hip -- compile-time plans, complex FP32, single pass:
// part 3 of 4 of the fast lengths below 16000 that the other files leave.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// median 1.22x over the runtime-planned pass (9000 120 -> 79 us, 720 64 -> 50,
// 15625 102 -> 91); 2500 lost (0.98x).
#include "fixed.h"

namespace sfft {
namespace {
const FixedC2C<float, 80, 6, 43, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5> c80;
const FixedC2C<float, 100, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10> c100;
const FixedC2C<float, 135, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 9> c135;
const FixedC2C<float, 180, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12> c180;
const FixedC2C<float, 225, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15> c225;
const FixedC2C<float, 375, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15> c375;
const FixedC2C<float, 480, 32, 8, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 2> c480;
const FixedC2C<float, 675, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3> c675;
const FixedC2C<float, 900, 60, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 4> c900;
const FixedC2C<float, 1200, 80, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5> c1200;
const FixedC2C<float, 1800, 120, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8> c1800;
const FixedC2C<float, 3200, 200, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 8> c3200;
const FixedC2C<float, 3840, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15> c3840;
const FixedC2C<float, 9000, 600, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8, 5> c9000;
const FixedC2C<float, 12500, 834, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 5, 4> c12500;
const FixedC2C<float, 15625, 625, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 25> c15625;
}  // namespace
}  // namespace sfft
