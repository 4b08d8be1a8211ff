// fixed_f64_real_single4.hip -- compile-time plans, real FP64 (real
// length 2h), single pass: part 5 of 8 of the fast half lengths h up to 8192.
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
const FixedReal<double, 81, 9, 28, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9> r162;
const FixedReal<double, 135, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 9> r270;
const FixedReal<double, 216, 18, 14, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 6, 6, 6> r432;
const FixedReal<double, 300, 20, 7, Sched<0, 0, 0, 0, kLdsPadShift, 0, 1>, 0, 15, 5, 4> r600;
const FixedReal<double, 486, 54, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 6> r972;
const FixedReal<double, 720, 48, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 3> r1440;
const FixedReal<double, 972, 108, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 9> r1944;
const FixedReal<double, 1280, 86, 2, Sched<0, 0, 0, 0, kLdsPadShift, 0, 1>, 0, 16, 16, 5> r2560;
const FixedReal<double, 1620, 180, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 9> r3240;
const FixedReal<double, 2160, 180, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 12> r4320;
const FixedReal<double, 2592, 216, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6, 6, 6> r5184;
const FixedReal<double, 3240, 270, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 6> r6480;
const FixedReal<double, 4000, 400, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10, 4> r8000;
const FixedReal<double, 5000, 500, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10, 5> r10000;
const FixedReal<double, 6075, 405, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3, 3, 3> r12150;
const FixedReal<double, 7200, 480, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15, 2> r14400;
}  // namespace
}  // namespace sfft
