// fixed_p2_mid.hip -- compile-time plans, complex FP32: 4096, 2048.
// FixedC2C<type, N, threads per transform, transforms per block,
//          Sched<prefetch stage, min waves per SIMD, pair loads, prefetch first>,
//          variant (0 = default, the fastest measured), radices...>
// 4096 loads its twiddles after the exchange: 320 transforms 7.7 -> 7.1 us (7.0
// persistent), 1536 20.4 -> 19.9 (18.9), 4096 44.0 -> 42.9 (44.6); one 5.00 -> 5.08.
// (Half-size blocks, a twiddle choice, the seventh Sched value, or kPersist: lengths
// that one group per block had slowed; figures at the top of fixed.h.)
#include "fixed.h"

namespace sfft {
namespace {
const FixedC2C<float, 4096, 256, 1, Sched<-1, 4, 0, 0, kLdsPadShift, 0, 0>, 0, 16, 16, 16> c4096a;
const FixedC2C<float, 4096, 256, 1, Sched<-2, 0, 0>, 1, 16, 16, 16> c4096b;
const FixedC2C<float, 2048, 128, 1, Sched<-1, 0, 0>, 0, 16, 16, 8> c2048a;
const FixedC2C<float, 2048, 128, 2, Sched<0, 4, 0>, 1, 16, 16, 8> c2048b;
}  // namespace
}  // namespace sfft
