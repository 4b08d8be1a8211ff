// fixed_16_single1.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 2 of 8 of the fast lengths
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
    const FixedC2C<E, 72, 6, 43, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 6> c72;
    const FixedC2C<E, 120, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8> c120;
    const FixedC2C<E, 180, 15, 17, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12> c180;
    const FixedC2C<E, 288, 24, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 12, 2> c288;
    const FixedC2C<E, 405, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 5> c405;
    const FixedC2C<E, 600, 40, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 5> c600;
    const FixedC2C<E, 768, 52, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 3> c768;
    const FixedC2C<E, 1080, 90, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 6> c1080;
    const FixedC2C<E, 1350, 113, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6> c1350;
    const FixedC2C<E, 1800, 120, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8> c1800;
    const FixedC2C<E, 2250, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 10> c2250;
    const FixedC2C<E, 2916, 324, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 6, 6> c2916;
    const FixedC2C<E, 3600, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 15> c3600;
    const FixedC2C<E, 4374, 486, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 6> c4374;
    const FixedC2C<E, 5400, 360, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8, 3> c5400;
    const FixedC2C<E, 6400, 400, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 16> c6400;
    const FixedC2C<E, 7680, 512, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15, 2> c7680;
    const FixedC2C<E, 9375, 625, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 15> c9375;
    const FixedC2C<E, 10935, 729, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 9, 9, 9> c10935;
    const FixedC2C<E, 12800, 800, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 10, 5> c12800;
    const FixedC2C<E, 15625, 625, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 25> c15625;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
