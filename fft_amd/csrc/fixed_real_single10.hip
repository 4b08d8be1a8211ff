// fixed_real_single10.hip -- compile-time plans, real FP32 (real
// length 2h), single pass: part 7 of 8 of the fast half lengths h up to 15625
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
const FixedReal<float, 128, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8> r256;
const FixedReal<float, 375, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15> r750;
const FixedReal<float, 1125, 75, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5> r2250;
const FixedReal<float, 2000, 134, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 5> r4000;
const FixedReal<float, 3600, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15> r7200;
const FixedReal<float, 6250, 417, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 5, 2> r12500;
const FixedReal<float, 9375, 625, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 15> r18750;
const FixedReal<float, 13500, 900, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 4> r27000;
}  // namespace
}  // namespace sfft
