// fixed_16_single7.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 8 of 8 of the fast lengths
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
    const FixedC2C<E, 100, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10> c100;
    const FixedC2C<E, 160, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 10> c160;
    const FixedC2C<E, 250, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 10> c250;
    const FixedC2C<E, 384, 26, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8, 3> c384;
    const FixedC2C<E, 540, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6> c540;
    const FixedC2C<E, 729, 81, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9> c729;
    const FixedC2C<E, 972, 108, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 9> c972;
    const FixedC2C<E, 1280, 86, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 5> c1280;
    const FixedC2C<E, 1620, 180, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 9> c1620;
    const FixedC2C<E, 2160, 180, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 12> c2160;
    const FixedC2C<E, 2700, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 12> c2700;
    const FixedC2C<E, 3375, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15> c3375;
    const FixedC2C<E, 4050, 338, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6, 3> c4050;
    const FixedC2C<E, 5120, 342, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 5, 4> c5120;
    const FixedC2C<E, 6144, 410, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 8, 3> c6144;
    const FixedC2C<E, 7290, 729, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 3, 3, 3, 3, 3, 2> c7290;
    const FixedC2C<E, 9000, 900, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 10, 10, 6> c9000;
    const FixedC2C<E, 10368, 864, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 12, 6> c10368;
    const FixedC2C<E, 12288, 820, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 16, 3> c12288;
    const FixedC2C<E, 14580, 972, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 6, 6, 3, 3, 3> c14580;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
