// fixed_16_single5.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 6 of 8 of the fast lengths
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
    const FixedC2C<E, 90, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9> c90;
    const FixedC2C<E, 144, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12> c144;
    const FixedC2C<E, 240, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15> c240;
    const FixedC2C<E, 360, 24, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 3> c360;
    const FixedC2C<E, 486, 54, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 6> c486;
    const FixedC2C<E, 675, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3> c675;
    const FixedC2C<E, 900, 60, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 4> c900;
    const FixedC2C<E, 1215, 135, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 9, 9> c1215;
    const FixedC2C<E, 1536, 128, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 6> c1536;
    const FixedC2C<E, 2000, 134, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 5> c2000;
    const FixedC2C<E, 2560, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 10> c2560;
    const FixedC2C<E, 3200, 200, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 8> c3200;
    const FixedC2C<E, 3888, 432, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 6, 6> c3888;
    const FixedC2C<E, 4860, 540, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9, 9, 6> c4860;
    const FixedC2C<E, 6000, 400, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 15> c6000;
    const FixedC2C<E, 6912, 576, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 6, 6> c6912;
    const FixedC2C<E, 8640, 720, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 12, 5> c8640;
    const FixedC2C<E, 10125, 675, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 3> c10125;
    const FixedC2C<E, 12000, 800, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 15, 2> c12000;
    const FixedC2C<E, 13824, 922, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 3, 3, 3, 2> c13824;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
