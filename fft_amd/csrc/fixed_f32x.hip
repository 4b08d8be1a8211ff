// fixed_f32x.hip -- compile-time single-pass plans for FP32 storage under FP64
// arithmetic: the shapes of the FP64 powers of two (fixed_f64.hip).
#include "fixed.h"

namespace sfft {
namespace {
using X = Stored<StoreF32>;
const FixedC2C<X, 4096, 256, 1, Sched<-1, 0, 0>, 0, 16, 16, 16> x4096;
const FixedC2C<X, 1024, 64, 4, Sched<-1, 0, 0>, 0, 16, 16, 4> x1024;
const FixedC2C<X, 2048, 128, 2, Sched<-1, 0, 0>, 0, 16, 16, 8> x2048;
const FixedC2C<X, 8192, 512, 1, Sched<-1, 0, 0>, 0, 16, 16, 8, 4> x8192;
const FixedC2C<X, 256, 16, 8, Sched<-1, 0, 0>, 0, 16, 16> x256;
const FixedC2C<X, 512, 32, 4, Sched<-1, 0, 0>, 0, 16, 8, 4> x512;
}  // namespace
}  // namespace sfft
