// fixed_single4.hip -- compile-time plans, complex FP32, single pass:
// part 1 of 4 of the fast lengths below 16000 that the other files leave.
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
const FixedC2C<float, 72, 6, 43, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6> c72;
const FixedC2C<float, 90, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9> c90;
const FixedC2C<float, 120, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8> c120;
const FixedC2C<float, 150, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10> c150;
const FixedC2C<float, 200, 13, 20, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 8> c200;
const FixedC2C<float, 320, 22, 12, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5, 4> c320;
const FixedC2C<float, 432, 36, 7, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6, 6> c432;
const FixedC2C<float, 625, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25> c625;
const FixedC2C<float, 750, 50, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 2> c750;
const FixedC2C<float, 1125, 75, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5> c1125;
const FixedC2C<float, 1280, 86, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 5> c1280;
const FixedC2C<float, 2000, 134, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 5> c2000;
const FixedC2C<float, 3600, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15> c3600;
const FixedC2C<float, 6750, 450, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 2> c6750;
const FixedC2C<float, 9720, 810, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 6, 3> c9720;
const FixedC2C<float, 13824, 922, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 3, 3, 3, 2> c13824;
}  // namespace
}  // namespace sfft
