// fixed_single5.hip -- compile-time plans, complex FP32, single pass:
// part 2 of 4 of the fast lengths below 16000 that the other files leave.
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
const FixedC2C<float, 75, 5, 51, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5> c75;
const FixedC2C<float, 96, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6> c96;
const FixedC2C<float, 128, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8> c128;
const FixedC2C<float, 160, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 10> c160;
const FixedC2C<float, 216, 18, 14, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 6, 6, 6> c216;
const FixedC2C<float, 360, 24, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 3> c360;
const FixedC2C<float, 450, 30, 9, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 2> c450;
const FixedC2C<float, 640, 43, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8, 5> c640;
const FixedC2C<float, 768, 52, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 3> c768;
const FixedC2C<float, 1152, 96, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 6> c1152;
const FixedC2C<float, 1350, 113, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6> c1350;
const FixedC2C<float, 2304, 192, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 12> c2304;
const FixedC2C<float, 3750, 250, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5, 2> c3750;
const FixedC2C<float, 7500, 500, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5, 4> c7500;
const FixedC2C<float, 11250, 750, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 15, 2> c11250;
const FixedC2C<float, 15000, 1000, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 8, 5> c15000;
}  // namespace
}  // namespace sfft
