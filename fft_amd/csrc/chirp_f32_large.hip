// chirp_f32_large.hip -- one-launch chirp-z kernels, FP32: convolution
// lengths 5120...16384, one transform per block, 8 to 16 elements a thread so
// that a CU holds 16 waves or more.  Three stages of radix 32 b 32 (32 elements
// a thread, two waves per SIMD) were slower: M = 5120 105 -> 81 us, 8192 58 ->
// 49, 16384 89 -> 78.  12288 and 15360 lose to 16384, and so does 10240 (n =
// 5003, both directions, 1 / 512 / 4096 transforms: 40.1 / 36.9, 108.6 / 87.6,
// 911 / 671 us), which would go too.
#include "chirp.h"

namespace sfft {
namespace {
const ChirpReg<float, false, 5120, 640, 1, 4, 8, 8, 8, 10> c5120;
const ChirpReg<float, false, 6144, 768, 1, 4, 8, 12, 8, 8> c6144;
const ChirpReg<float, false, 8192, 512, 1, 4, 16, 8, 4, 16> c8192;
const ChirpReg<float, false, 9216, 576, 1, 4, 16, 9, 4, 16> c9216;
const ChirpReg<float, false, 10240, 640, 1, 4, 16, 10, 4, 16> c10240;
const ChirpReg<float, false, 16384, 1024, 1, 4, 16, 16, 4, 16> c16384;
}  // namespace
}  // namespace sfft
