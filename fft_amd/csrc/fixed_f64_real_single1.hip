// fixed_f64_real_single1.hip -- compile-time plans, real FP64 (real
// length 2h), single pass: part 2 of 8 of the fast half lengths h up to 8192.
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
const FixedReal<double, 72, 6, 43, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6> r144;
const FixedReal<double, 120, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8> r240;
const FixedReal<double, 180, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12> r360;
const FixedReal<double, 256, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16> r512;
const FixedReal<double, 405, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 5> r810;
const FixedReal<double, 600, 40, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 5> r1200;
const FixedReal<double, 864, 72, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6> r1728;
const FixedReal<double, 1200, 80, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5> r2400;
const FixedReal<double, 1500, 150, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10, 10> r3000;
const FixedReal<double, 1944, 216, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 6, 6, 6> r3888;
const FixedReal<double, 2430, 270, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9, 9, 3> r4860;
const FixedReal<double, 3072, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 12> r6144;
const FixedReal<double, 3750, 250, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5, 5, 2> r7500;
const FixedReal<double, 4608, 384, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 12, 2> r9216;
const FixedReal<double, 5760, 384, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 8, 3> r11520;
const FixedReal<double, 6561, 438, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 3, 3, 3, 3, 3, 3, 3, 3> r13122;
}  // namespace
}  // namespace sfft
