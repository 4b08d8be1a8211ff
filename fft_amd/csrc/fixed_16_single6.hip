// fixed_16_single6.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 7 of 8 of the fast lengths
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
    const FixedC2C<E, 10240, 640, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 10, 4> c10240;
    const FixedC2C<E, 12150, 810, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 10, 9, 9> c12150;
    const FixedC2C<E, 14400, 960, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15, 4> c14400;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
