// chirp_f64.hip -- one-launch chirp-z kernels, FP64: convolution lengths up
// to 8192 (16-byte values: 136 KB of LDS).  As in FP32, with two waves per
// SIMD: 16 elements of 16 bytes in registers.
#include "chirp.h"

namespace sfft {
namespace {
const ChirpReg<double, false, 64, 8, 16, 2, 8, 8> d64;
const ChirpReg<double, false, 128, 16, 8, 2, 8, 2, 8> d128;
const ChirpReg<double, false, 192, 24, 8, 2, 8, 3, 8> d192;
const ChirpReg<double, false, 256, 16, 8, 2, 16, 16> d256;
const ChirpReg<double, false, 320, 40, 4, 2, 8, 5, 8> d320;
const ChirpReg<double, false, 384, 48, 4, 2, 8, 6, 8> d384;
const ChirpReg<double, false, 512, 64, 2, 2, 8, 8, 8> d512;
const ChirpReg<double, false, 640, 80, 2, 2, 8, 10, 8> d640;
const ChirpReg<double, false, 768, 48, 4, 2, 16, 3, 16> d768;
const ChirpReg<double, false, 1024, 64, 2, 2, 16, 4, 16> d1024;
const ChirpReg<double, false, 1280, 80, 2, 2, 16, 5, 16> d1280;
const ChirpReg<double, false, 1536, 96, 2, 2, 16, 6, 16> d1536;
const ChirpReg<double, false, 2048, 128, 1, 2, 16, 8, 16> d2048;
const ChirpReg<double, false, 2560, 256, 1, 2, 16, 10, 16> d2560;
const ChirpReg<double, false, 3072, 256, 1, 2, 16, 12, 16> d3072;
const ChirpReg<double, false, 3840, 256, 1, 2, 16, 15, 16> d3840;
const ChirpReg<double, false, 4096, 256, 1, 2, 16, 16, 16> d4096;
const ChirpReg<double, false, 5120, 320, 1, 2, 16, 4, 5, 16> d5120;
const ChirpReg<double, false, 6144, 384, 1, 2, 16, 4, 6, 16> d6144;
const ChirpReg<double, false, 8192, 512, 1, 2, 16, 8, 4, 16> d8192;
}  // namespace
}  // namespace sfft
