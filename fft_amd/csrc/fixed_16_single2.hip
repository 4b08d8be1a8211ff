// fixed_16_single2.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 3 of 8 of the fast lengths
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
    const FixedC2C<E, 75, 5, 51, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5> c75;
    const FixedC2C<E, 125, 9, 28, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 5> c125;
    const FixedC2C<E, 192, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12> c192;
    const FixedC2C<E, 300, 20, 13, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 4> c300;
    const FixedC2C<E, 432, 36, 7, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6, 6> c432;
    const FixedC2C<E, 625, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25> c625;
    const FixedC2C<E, 800, 50, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 2> c800;
    const FixedC2C<E, 1125, 75, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5> c1125;
    const FixedC2C<E, 1440, 144, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 10> c1440;
    const FixedC2C<E, 1875, 125, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5> c1875;
    const FixedC2C<E, 2304, 192, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 12> c2304;
    const FixedC2C<E, 3000, 200, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 8> c3000;
    const FixedC2C<E, 3645, 405, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 5> c3645;
    const FixedC2C<E, 4500, 300, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5, 4> c4500;
    const FixedC2C<E, 5625, 375, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 15> c5625;
    const FixedC2C<E, 6480, 540, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 6, 6> c6480;
    const FixedC2C<E, 7776, 864, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 9, 6> c7776;
    const FixedC2C<E, 9600, 640, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 8, 5> c9600;
    const FixedC2C<E, 11250, 750, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 15, 2> c11250;
    const FixedC2C<E, 12960, 864, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 3, 3, 3, 2> c12960;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
