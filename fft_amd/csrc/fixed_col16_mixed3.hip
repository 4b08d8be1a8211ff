// fixed_col16_mixed3.hip -- compile-time column passes of two-pass
// plans with 16-bit storage, part 4 of 4 of the mixed-radix lengths of
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
    const FixedCol<E, 144, 12, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 12, 12> c144;
    const FixedCol<E, 180, 15, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 12> c180;
    const FixedCol<E, 225, 15, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 15> c225;
    const FixedCol<E, 270, 23, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 6, 3> c270;
    const FixedCol<E, 324, 36, 8, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 9, 6, 6> c324;
    const FixedCol<E, 400, 25, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 25, 16> c400;
    const FixedCol<E, 480, 32, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 15, 2> c480;
    const FixedCol<E, 576, 48, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 6, 6> c576;
    const FixedCol<E, 648, 72, 4, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 12, 9, 6> c648;
    const FixedCol<E, 750, 50, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 25, 15, 2> c750;
    const FixedCol<E, 864, 72, 4, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 12, 12, 6> c864;
    const FixedCol<E, 1000, 100, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad>, 10, 10, 10> c1000;
};
const Col<StoreF16> f16;
const Col<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
