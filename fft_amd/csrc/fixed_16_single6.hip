// fixed_16_single6.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 7 of 8 of the fast lengths
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
    const FixedC2C<E, 96, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6> c96;
    const FixedC2C<E, 150, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10> c150;
    const FixedC2C<E, 243, 27, 9, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 3> c243;
    const FixedC2C<E, 375, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15> c375;
    const FixedC2C<E, 500, 50, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 5> c500;
    const FixedC2C<E, 720, 48, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 3> c720;
    const FixedC2C<E, 960, 64, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 4> c960;
    const FixedC2C<E, 1250, 79, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 2> c1250;
    const FixedC2C<E, 1600, 100, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 4> c1600;
    const FixedC2C<E, 2025, 135, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3, 3> c2025;
    const FixedC2C<E, 2592, 216, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6, 6, 6> c2592;
    const FixedC2C<E, 3240, 270, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 6> c3240;
    const FixedC2C<E, 4000, 400, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10, 4> c4000;
    const FixedC2C<E, 5000, 313, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 8> c5000;
    const FixedC2C<E, 6075, 405, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3, 3, 3> c6075;
    const FixedC2C<E, 7200, 480, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15, 2> c7200;
    const FixedC2C<E, 8748, 972, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 9, 9> c8748;
    const FixedC2C<E, 10240, 683, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 8, 5> c10240;
    const FixedC2C<E, 12150, 1013, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6, 3, 3> c12150;
    const FixedC2C<E, 14400, 960, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15, 4> c14400;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
