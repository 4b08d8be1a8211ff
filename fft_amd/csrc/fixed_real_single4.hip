// fixed_real_single4.hip -- compile-time plans, real FP32 (real
// length 2h), single pass: part 1 of 8 of the fast half lengths h up to 15625
// that the other files leave.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// R2C forward and inverse median 1.24x (10800 114 + 127 -> 75 + 76 us, 31250 118
// + 121 -> 106 + 106), half-bin shifted 1.28x; h = 64, 72, 75, 80, 125, 200 and
// 2500 lose up to 18 % in one direction of one kind.
#include "fixed.h"

namespace sfft {
namespace {
const FixedReal<float, 81, 9, 28, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9> r162;
const FixedReal<float, 180, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12> r360;
const FixedReal<float, 450, 30, 9, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 2> r900;
const FixedReal<float, 1350, 113, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6> r2700;
const FixedReal<float, 2160, 180, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 12> r4320;
const FixedReal<float, 3840, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15> r7680;
const FixedReal<float, 6750, 450, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 2> r13500;
const FixedReal<float, 10125, 675, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 3> r20250;
const FixedReal<float, 14580, 972, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 4, 3, 3, 3, 3, 3> r29160;
}  // namespace
}  // namespace sfft
