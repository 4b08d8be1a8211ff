// fixed_16_single2.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 3 of 8 of the fast lengths
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
    const FixedC2C<E, 6480, 432, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 3, 3, 3> c6480;
    const FixedC2C<E, 7776, 486, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 9, 9, 6> c7776;
    const FixedC2C<E, 9600, 960, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 10, 10, 6> c9600;
    const FixedC2C<E, 11250, 750, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 15, 2> c11250;
    const FixedC2C<E, 12960, 810, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 10, 9, 9> c12960;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
