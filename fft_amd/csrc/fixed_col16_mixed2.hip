// fixed_col16_mixed2.hip -- compile-time column passes of two-pass
// plans with 16-bit storage, part 3 of 4 of the mixed-radix lengths of
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
    const FixedCol<E, 135, 15, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 9> c135;
    const FixedCol<E, 162, 18, 16, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 9, 9, 2> c162;
    const FixedCol<E, 216, 18, 16, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad>, 6, 6, 6> c216;
    const FixedCol<E, 250, 25, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 25, 10> c250;
    const FixedCol<E, 320, 22, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 5, 4> c320;
    const FixedCol<E, 384, 26, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 8, 3> c384;
    const FixedCol<E, 450, 30, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 15, 2> c450;
    const FixedCol<E, 540, 45, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 15, 6, 6> c540;
    const FixedCol<E, 640, 43, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad>, 16, 8, 5> c640;
    const FixedCol<E, 729, 81, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad>, 9, 9, 9> c729;
    const FixedCol<E, 810, 90, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad>, 10, 9, 9> c810;
    const FixedCol<E, 972, 108, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad>, 12, 9, 9> c972;
};
const Col<StoreF16> f16;
const Col<StoreBF16> bf16;
}  // namespace
}  // namespace sfft
