// fixed_f64_real_single7.hip -- compile-time plans, real FP64 (real
// length 2h), single pass: part 8 of 8 of the fast half lengths h up to 8192.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// R2C forward and inverse median 1.31x, up to 2.4x (15000 133 + 142 -> 103 + 112
// us); h = 360, 384, 450, 640, 675 and 768 lose up to 22 %.
#include "fixed.h"

namespace sfft {
namespace {
const FixedReal<double, 100, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10> r200;
const FixedReal<double, 160, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 10> r320;
const FixedReal<double, 243, 27, 9, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 3> r486;
const FixedReal<double, 375, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5> r750;
const FixedReal<double, 540, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6> r1080;
const FixedReal<double, 800, 80, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 8> r1600;
const FixedReal<double, 1125, 75, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5> r2250;
const FixedReal<double, 1440, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 10> r2880;
const FixedReal<double, 1875, 125, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5, 5> r3750;
const FixedReal<double, 2304, 192, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 12> r4608;
const FixedReal<double, 2916, 324, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 6, 6> r5832;
const FixedReal<double, 3600, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15> r7200;
const FixedReal<double, 4374, 486, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 6> r8748;
const FixedReal<double, 5400, 360, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8, 3> r10800;
const FixedReal<double, 6400, 427, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 5, 5> r12800;
const FixedReal<double, 7680, 512, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15, 2> r15360;
}  // namespace
}  // namespace sfft
