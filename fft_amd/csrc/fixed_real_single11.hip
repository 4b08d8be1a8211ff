// fixed_real_single11.hip -- compile-time plans, real FP32 (real
// length 2h), single pass: part 8 of 8 of the fast half lengths h up to 15625
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
const FixedReal<float, 144, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12> r288;
const FixedReal<float, 400, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16> r800;
const FixedReal<float, 1250, 79, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 2> r2500;
const FixedReal<float, 2025, 135, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3, 3> r4050;
const FixedReal<float, 3750, 250, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5, 2> r7500;
const FixedReal<float, 6400, 400, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 16> r12800;
const FixedReal<float, 9720, 810, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 6, 3> r19440;
const FixedReal<float, 13824, 922, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 3, 3, 3, 2> r27648;
}  // namespace
}  // namespace sfft
