// fixed_16_single3.hip -- compile-time plans with 16-bit storage
// (float LDS and arithmetic), single pass: part 4 of 8 of the fast lengths
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
    const FixedC2C<E, 80, 6, 43, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5> c80;
    const FixedC2C<E, 128, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8> c128;
    const FixedC2C<E, 216, 18, 14, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 6, 6, 6> c216;
    const FixedC2C<E, 320, 22, 12, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 5, 4> c320;
    const FixedC2C<E, 450, 30, 9, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 2> c450;
    const FixedC2C<E, 640, 43, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8, 5> c640;
    const FixedC2C<E, 810, 90, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 9, 9> c810;
    const FixedC2C<E, 1152, 96, 3, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 6> c1152;
    const FixedC2C<E, 1458, 162, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 2> c1458;
    const FixedC2C<E, 1920, 128, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 8> c1920;
    const FixedC2C<E, 2400, 240, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 10> c2400;
    const FixedC2C<E, 3072, 256, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 12> c3072;
    const FixedC2C<E, 3750, 250, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5, 2> c3750;
    const FixedC2C<E, 4608, 384, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 12, 12, 2> c4608;
    const FixedC2C<E, 5760, 384, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 8, 3> c5760;
    const FixedC2C<E, 6561, 729, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 9> c6561;
    const FixedC2C<E, 8000, 800, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 10, 10, 5> c8000;
    const FixedC2C<E, 9720, 648, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 9, 9, 8> c9720;
    const FixedC2C<E, 11520, 768, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15, 3> c11520;
    const FixedC2C<E, 13122, 729, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 9, 9, 9, 9, 2> c13122;
};
const One<StoreF16> f16;
const One<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
