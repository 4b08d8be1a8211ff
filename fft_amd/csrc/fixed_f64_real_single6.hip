// fixed_f64_real_single6.hip -- compile-time plans, real FP64 (real
// length 2h), single pass: part 7 of 8 of the fast half lengths h up to 8192.
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
const FixedReal<double, 96, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6> r192;
const FixedReal<double, 150, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10> r300;
const FixedReal<double, 240, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15> r480;
const FixedReal<double, 324, 36, 7, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 6, 6> r648;
const FixedReal<double, 512, 32, 8, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 2> r1024;
const FixedReal<double, 750, 75, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10, 5> r1500;
const FixedReal<double, 1080, 90, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 6> r2160;
const FixedReal<double, 1350, 113, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6> r2700;
const FixedReal<double, 1800, 120, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8> r3600;
const FixedReal<double, 2250, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 10> r4500;
const FixedReal<double, 2880, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 12> r5760;
const FixedReal<double, 3456, 288, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6, 6, 6> r6912;
const FixedReal<double, 4320, 360, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6, 5> r8640;
const FixedReal<double, 5184, 432, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6, 6> r10368;
const FixedReal<double, 6250, 417, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5, 5, 2> r12500;
const FixedReal<double, 7500, 500, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5, 5, 4> r15000;
}  // namespace
}  // namespace sfft
