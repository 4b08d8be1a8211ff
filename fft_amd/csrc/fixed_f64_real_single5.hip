// fixed_f64_real_single5.hip -- compile-time plans, real FP64 (real
// length 2h), single pass: part 6 of 8 of the fast half lengths h up to 8192.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// R2C forward and inverse median 1.31x, up to 2.4x (15000 133 + 142 -> 103 + 112
// us); h = 360, 384, 450, 640, 675 and 768 lose up to 22 %.
// (Half-size blocks, a twiddle choice, the seventh Sched value, or kPersist: lengths
// that one group per block had slowed; figures at the top of fixed.h.)
#include "fixed.h"

namespace sfft {
namespace {
const FixedReal<double, 90, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9> r180;
const FixedReal<double, 144, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12> r288;
const FixedReal<double, 225, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15> r450;
const FixedReal<double, 320, 22, 6, Sched<0, 0, 0, 0, kLdsPadShift, 0, 1>, 0, 16, 5, 4> r640;
const FixedReal<double, 500, 50, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 5> r1000;
const FixedReal<double, 729, 81, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9> r1458;
const FixedReal<double, 1000, 100, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10> r2000;
const FixedReal<double, 1296, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 9> r2592;
const FixedReal<double, 1728, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 12> r3456;
const FixedReal<double, 2187, 243, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 3> r4374;
const FixedReal<double, 2700, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 12> r5400;
const FixedReal<double, 3375, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15> r6750;
const FixedReal<double, 4050, 338, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6, 3> r8100;
const FixedReal<double, 5120, 342, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 5, 4> r10240;
const FixedReal<double, 6144, 410, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 8, 3> r12288;
const FixedReal<double, 7290, 486, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 3, 3, 3, 3, 3, 2> r14580;
}  // namespace
}  // namespace sfft
