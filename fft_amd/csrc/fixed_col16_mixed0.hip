// fixed_col16_mixed0.hip -- compile-time column passes of two-pass
// plans with 16-bit storage, part 1 of 4 of the mixed-radix lengths of
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
    const FixedCol<E, 81, 9, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 9, 9> c81;
    const FixedCol<E, 150, 15, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 10> c150;
    const FixedCol<E, 192, 16, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 12> c192;
    const FixedCol<E, 240, 16, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 15> c240;
    const FixedCol<E, 288, 24, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 12, 12, 2> c288;
    const FixedCol<E, 360, 24, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 8, 3> c360;
    const FixedCol<E, 405, 45, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 9, 9, 5> c405;
    const FixedCol<E, 486, 54, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 9, 9, 6> c486;
    const FixedCol<E, 600, 40, 8, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 8, 5> c600;
    const FixedCol<E, 675, 45, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 15, 3> c675;
    const FixedCol<E, 768, 52, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 16, 3> c768;
    const FixedCol<E, 900, 60, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 15, 4> c900;
};
const Col<StoreF16> f16;
const Col<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
