// fixed_16_single4.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 5 of 8 of the fast lengths
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
    const FixedC2C<E, 81, 9, 28, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9> c81;
    const FixedC2C<E, 135, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 9> c135;
    const FixedC2C<E, 225, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15> c225;
    const FixedC2C<E, 324, 36, 7, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 6, 6> c324;
    const FixedC2C<E, 480, 32, 8, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 2> c480;
    const FixedC2C<E, 648, 72, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 6> c648;
    const FixedC2C<E, 864, 72, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 6> c864;
    const FixedC2C<E, 1200, 80, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5> c1200;
    const FixedC2C<E, 1500, 150, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10, 10> c1500;
    const FixedC2C<E, 1944, 216, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 6, 6, 6> c1944;
    const FixedC2C<E, 2430, 270, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9, 9, 3> c2430;
    const FixedC2C<E, 3125, 209, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 5> c3125;
    const FixedC2C<E, 3840, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15> c3840;
    const FixedC2C<E, 4800, 320, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 5, 4> c4800;
    const FixedC2C<E, 5832, 648, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 9, 6> c5832;
    const FixedC2C<E, 6750, 450, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 2> c6750;
    const FixedC2C<E, 8100, 900, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 9, 9> c8100;
    const FixedC2C<E, 10000, 1000, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 10, 10> c10000;
    const FixedC2C<E, 11664, 972, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 6, 6, 6, 6, 3, 3> c11664;
    const FixedC2C<E, 13500, 900, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 4> c13500;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
