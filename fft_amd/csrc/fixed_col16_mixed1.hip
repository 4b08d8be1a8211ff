// fixed_col16_mixed1.hip -- compile-time column passes of two-pass
// plans with 16-bit storage, part 2 of 4 of the mixed-radix lengths of
// fixed_col_mixed.hip and fixed_col_large.hip.  Radices as the runtime planner's
// cost model chooses them at 16 elements a thread; the widest tile of up to 32
// columns of which two blocks fit a CU.  Bound by HBM; batches of 128 MB, both
// passes against runtime-planned ones: 1.1-1.9x (124416 314 -> 168 us, 388800
// 294 -> 166).
#include "fixed.h"

namespace sfft {
namespace {
template <class S>
struct Col {
    using E = Stored<S>;
    const FixedCol<E, 125, 5, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 25, 5> c125;
    const FixedCol<E, 160, 16, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 10> c160;
    const FixedCol<E, 200, 13, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 25, 8> c200;
    const FixedCol<E, 243, 27, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 9, 9, 3> c243;
    const FixedCol<E, 300, 20, 16, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 5, 4> c300;
    const FixedCol<E, 375, 25, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 25, 15> c375;
    const FixedCol<E, 432, 36, 8, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 12, 6, 6> c432;
    const FixedCol<E, 500, 50, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 10, 10, 5> c500;
    const FixedCol<E, 625, 25, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 25, 25> c625;
    const FixedCol<E, 720, 48, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 15, 3> c720;
    const FixedCol<E, 800, 50, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 25, 16, 2> c800;
    const FixedCol<E, 960, 64, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 15, 4> c960;
};
const Col<StoreF16> f16;
const Col<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
