// fixed_16_single4.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 5 of 8 of the fast lengths
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
    const FixedC2C<E, 5832, 486, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 6, 6, 6, 3, 3, 3> c5832;
    const FixedC2C<E, 6750, 450, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 2> c6750;
    const FixedC2C<E, 8100, 900, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10, 9, 9> c8100;
    const FixedC2C<E, 10000, 625, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 16> c10000;
    const FixedC2C<E, 11664, 729, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 9, 9, 9> c11664;
    const FixedC2C<E, 13500, 900, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 4> c13500;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
