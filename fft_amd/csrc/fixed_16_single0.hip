// fixed_16_single0.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 1 of 8 of the fast lengths
// other than powers of two.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// median 1.52x over the runtime-planned pass, up to 3.9x above 8192; 200, 2500
// and 15000 are no faster.
#include "fixed.h"

namespace sfft {
namespace {
template <class S>
struct One {
    using E = Stored<S>;
    const FixedC2C<E, 64, 4, 64, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 4> c64;
    const FixedC2C<E, 108, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9> c108;
    const FixedC2C<E, 162, 18, 14, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 2> c162;
    const FixedC2C<E, 270, 23, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 3> c270;
    const FixedC2C<E, 400, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16> c400;
    const FixedC2C<E, 576, 48, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6, 6> c576;
    const FixedC2C<E, 750, 50, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 2> c750;
    const FixedC2C<E, 1000, 100, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10> c1000;
    const FixedC2C<E, 1296, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 9> c1296;
    const FixedC2C<E, 1728, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 12> c1728;
    const FixedC2C<E, 2187, 243, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 3> c2187;
    const FixedC2C<E, 2880, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 12> c2880;
    const FixedC2C<E, 3456, 288, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6, 6, 6> c3456;
    const FixedC2C<E, 4320, 360, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6, 5> c4320;
    const FixedC2C<E, 5184, 432, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6, 6> c5184;
    const FixedC2C<E, 6250, 417, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 5, 2> c6250;
    const FixedC2C<E, 7500, 500, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5, 4> c7500;
    const FixedC2C<E, 9216, 768, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 6, 6> c9216;
    const FixedC2C<E, 10800, 720, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15, 3> c10800;
    const FixedC2C<E, 12500, 834, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 5, 4> c12500;
    const FixedC2C<E, 15360, 1024, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15, 4> c15360;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
