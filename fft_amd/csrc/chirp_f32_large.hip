// chirp_f32_large.hip -- one-launch chirp-z kernels, FP32: convolution
// lengths 5120...16384, 32 b 32 with one radix-32 butterfly a thread (32
// elements in registers: up to 256 registers at two waves per SIMD), or more
// threads where the middle stage would hold more than 32 elements a thread.
#include "chirp.h"

namespace sfft {
namespace {
const ChirpReg<float, 5120, 160, 1, 2, 32, 5, 32> c5120;
const ChirpReg<float, 6144, 192, 1, 2, 32, 6, 32> c6144;
const ChirpReg<float, 7168, 224, 1, 2, 32, 7, 32> c7168;
const ChirpReg<float, 8192, 256, 1, 2, 32, 8, 32> c8192;
const ChirpReg<float, 9216, 344, 1, 2, 32, 9, 32> c9216;
const ChirpReg<float, 10240, 344, 1, 2, 32, 10, 32> c10240;
const ChirpReg<float, 12288, 512, 1, 2, 32, 12, 32> c12288;
const ChirpReg<float, 15360, 512, 1, 2, 32, 15, 32> c15360;
const ChirpReg<float, 16384, 512, 1, 2, 32, 16, 32> c16384;
}  // namespace
}  // namespace sfft
