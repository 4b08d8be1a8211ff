// fixed_single7.hip -- compile-time plans, complex FP32, single pass:
// part 4 of 4 of the fast lengths below 16000 that the other files leave.
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
const FixedC2C<float, 81, 9, 28, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9> c81;
const FixedC2C<float, 108, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9> c108;
const FixedC2C<float, 144, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12> c144;
const FixedC2C<float, 192, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12> c192;
const FixedC2C<float, 240, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15> c240;
const FixedC2C<float, 400, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16> c400;
const FixedC2C<float, 600, 40, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 5> c600;
const FixedC2C<float, 720, 48, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 3> c720;
const FixedC2C<float, 960, 64, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 4> c960;
const FixedC2C<float, 1250, 79, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 2> c1250;
const FixedC2C<float, 1875, 125, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5> c1875;
const FixedC2C<float, 3375, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15> c3375;
const FixedC2C<float, 5000, 313, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 8> c5000;
const FixedC2C<float, 9375, 625, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 15> c9375;
const FixedC2C<float, 13500, 900, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 4> c13500;
}  // namespace
}  // namespace sfft
