// fixed_f64_real_single3.hip -- compile-time plans, real FP64 (real
// length 2h), single pass: part 4 of 8 of the fast half lengths h up to 8192.
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
const FixedReal<double, 80, 6, 43, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5> r160;
const FixedReal<double, 128, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8> r256;
const FixedReal<double, 200, 14, 18, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 8, 5, 5> r400;
const FixedReal<double, 288, 24, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 2> r576;
const FixedReal<double, 480, 32, 8, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 2> r960;
const FixedReal<double, 648, 72, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 6> r1296;
const FixedReal<double, 960, 64, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 4> r1920;
const FixedReal<double, 1250, 84, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5, 2> r2500;
const FixedReal<double, 1600, 160, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 10, 10> r3200;
const FixedReal<double, 2025, 135, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3, 3> r4050;
const FixedReal<double, 2560, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 10> r5120;
const FixedReal<double, 3200, 214, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8, 5, 5> r6400;
const FixedReal<double, 3888, 432, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 6, 6> r7776;
const FixedReal<double, 4860, 405, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 3, 3> r9720;
const FixedReal<double, 6000, 400, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5, 5> r12000;
const FixedReal<double, 6912, 461, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 3, 3, 3> r13824;
}  // namespace
}  // namespace sfft
