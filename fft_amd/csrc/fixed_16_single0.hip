// fixed_16_single0.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 1 of 8 of the fast lengths
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
    const FixedC2C<E, 12500, 625, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 10, 2> c12500;
    const FixedC2C<E, 15360, 1024, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15, 4> c15360;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
