// wide_col.hip -- wider column tiles for launches that fill the device (one
// tile per CU or more; smaller launches take the tiles of fixed_col.hip or the
// runtime-planned pass, whose bits are the same).
// WideCol<type, N, threads per column, columns per block, Sched<...>,
// radices...>: exchanged a component plane at a time.  Listed where measured
// faster (both directions): FP32 2^24 370 us against 467 without, 2^21 x 8 322
// / 372, 2^22 x 4 298 / 408; IEEE half 2^24 280 / 419, 2^20 x 16 (4096 x 256)
// 196 / 234, 2^18 x 64 (2048 x 128) 179 / 193; F32X 2^24 600 / 739.  FP32 2048
// (339 / 331 at 2^22), half 1024 and 512 (168 / 155 at 2^18), and FP64 at every
// length (577 / 522 at 2^21) are slower this way: no next tile is prefetched.
#include "wide.h"

namespace sfft {
namespace {
const WideCol<float, 4096, 64, 8, Sched<0, 0, 0, 0>, 16, 16, 16> w4096;
// 1024: 16 columns (128-byte rows) of 32 elements a thread, persistent: with
// 1024 columns a pass, 8 KB between rows, 252 us against 303 at 2^20 x 16
const FixedColWide<float, 1024, 32, 16, Sched<0, 0, 0, 0>, 16, 16, 4> w1024;
template <class S>
struct Wide16 {
    using E = Stored<S>;
    const WideCol<E, 4096, 64, 8, Sched<0, 0, 0, 0>, 16, 16, 16> w4096;
    const WideCol<E, 2048, 32, 16, Sched<0, 0, 0, 0>, 16, 16, 8> w2048;
};
const Wide16<StoreF16> w16_f16;
const Wide16<StoreBF16> w16_bf16;
const WideCol<Stored<StoreF32>, 4096, 128, 4, Sched<0, 0, 0, 0>, 16, 16, 16> w4096x;
}  // namespace
}  // namespace sfft
