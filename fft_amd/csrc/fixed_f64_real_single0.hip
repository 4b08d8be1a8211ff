// fixed_f64_real_single0.hip -- compile-time plans, real FP64 (real
// length 2h), single pass: part 1 of 8 of the fast half lengths h up to 8192.
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
const FixedReal<double, 64, 4, 64, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 4> r128;
const FixedReal<double, 108, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9> r216;
const FixedReal<double, 162, 18, 14, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 2> r324;
const FixedReal<double, 250, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 5, 5> r500;
const FixedReal<double, 400, 27, 9, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5, 5> r800;
const FixedReal<double, 576, 48, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6, 6> r1152;
const FixedReal<double, 810, 90, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9, 9> r1620;
const FixedReal<double, 1152, 96, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 6> r2304;
const FixedReal<double, 1458, 162, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 2> r2916;
const FixedReal<double, 1920, 128, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 8> r3840;
const FixedReal<double, 2400, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 10> r4800;
const FixedReal<double, 3000, 200, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 5, 5> r6000;
const FixedReal<double, 3645, 405, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 5> r7290;
const FixedReal<double, 4500, 300, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5, 4> r9000;
const FixedReal<double, 5625, 375, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5, 5> r11250;
const FixedReal<double, 6480, 432, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 3, 3, 3> r12960;
const FixedReal<double, 8192, 512, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 16, 2> r16384;
}  // namespace
}  // namespace sfft
