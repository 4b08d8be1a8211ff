// fixed_16_single5.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 6 of 8 of the fast lengths
// other than powers of two.
// Radices are those the runtime planner's cost model chooses within the 512
// threads of a 16-bit block, so that bits and strided calls (which run the
// runtime-planned pass) stay as they were: the radices of 1024 threads made
// strided calls of 14 lengths 1.1 to 2.1x slower (both directions of 128 MB:
// 6912 267 -> 562 us, 13122 588 -> 965).  Six lengths take those all the same,
// because batches gain and strided calls do not lose (batches / strided, 512 ->
// 1024: 6561 308 / 496 -> 165 / 475, 8100 224 / 573 -> 188 / 502, 11250 243 / 646
// -> 222 / 570, 13500 249 / 569 -> 236 / 570, 14400 181 / 518 -> 174 / 521, 15360
// 182 / 478 -> 172 / 483).  Threads are free (the bits do not depend on them):
// about 256 a block, from 4860 on the multiple of the butterflies that idles least;
// one group per block (the persistent form of these kernels had lost).  Bound by
// HBM.  Listed where faster over both directions with neither 3 % slower, batches
// of 128 MB: median 1.5x over the runtime-planned pass, up to 3.5x above 7500;
// 200, 2500 and 15000 are no faster.
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
    const FixedC2C<E, 4860, 405, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 3, 3> c4860;
    const FixedC2C<E, 6000, 400, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 15> c6000;
    const FixedC2C<E, 6912, 432, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 3, 3, 3> c6912;
    const FixedC2C<E, 8640, 720, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 6, 6> c8640;
    const FixedC2C<E, 10125, 675, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 3> c10125;
    const FixedC2C<E, 12000, 800, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 10, 5> c12000;
    const FixedC2C<E, 13824, 864, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 9, 6> c13824;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
