// fixed_f64_real_single2.hip -- compile-time plans, real FP64 (real
// length 2h), single pass: part 3 of 8 of the fast half lengths h up to 8192.
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
const FixedReal<double, 75, 5, 51, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5> r150;
const FixedReal<double, 125, 9, 28, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5> r250;
const FixedReal<double, 192, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12> r384;
const FixedReal<double, 270, 23, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 3> r540;
const FixedReal<double, 432, 36, 7, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6, 6> r864;
const FixedReal<double, 625, 42, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5> r1250;
const FixedReal<double, 900, 60, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 4> r1800;
const FixedReal<double, 1215, 135, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 9, 9> r2430;
const FixedReal<double, 1536, 128, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 6> r3072;
const FixedReal<double, 2000, 134, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5, 5, 5> r4000;
const FixedReal<double, 2500, 250, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 5, 5> r5000;
const FixedReal<double, 3125, 209, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5, 5> r6250;
const FixedReal<double, 3840, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15> r7680;
const FixedReal<double, 4800, 320, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5, 4> r9600;
const FixedReal<double, 5832, 486, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 6, 6, 6, 3, 3, 3> r11664;
const FixedReal<double, 6750, 450, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 2> r13500;
}  // namespace
}  // namespace sfft
