// fixed_real_single5.hip -- compile-time plans, real FP32 (real
// length 2h), single pass: part 2 of 8 of the fast half lengths h up to 15625
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
const FixedReal<float, 90, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9> r180;
const FixedReal<float, 225, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15> r450;
const FixedReal<float, 600, 40, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 5> r1200;
const FixedReal<float, 1600, 100, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 4> r3200;
const FixedReal<float, 2700, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 12> r5400;
const FixedReal<float, 4374, 486, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 6> r8748;
const FixedReal<float, 7200, 480, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15, 2> r14400;
const FixedReal<float, 10935, 729, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 3, 3, 3, 3, 3, 3> r21870;
const FixedReal<float, 15000, 1000, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 8, 5> r30000;
}  // namespace
}  // namespace sfft
