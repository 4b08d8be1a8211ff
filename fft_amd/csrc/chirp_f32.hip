// chirp_f32.hip -- one-launch chirp-z kernels, FP32: convolution lengths up
// to 4096.  ChirpReg<type, M, threads per transform, transforms per block,
// minimum waves per SIMD, radices...>: R b R with M / R threads, one radix-R
// butterfly each; where the middle stage would then hold more than 21
// elements a thread (b of 10 and more) 256 threads take one middle butterfly
// each.  The lengths are a sixth to a quarter apart.
#include "chirp.h"

namespace sfft {
namespace {
const ChirpReg<float, 64, 8, 32, 4, 8, 8> c64;
const ChirpReg<float, 128, 16, 16, 4, 8, 2, 8> c128;
const ChirpReg<float, 192, 24, 8, 4, 8, 3, 8> c192;
const ChirpReg<float, 256, 16, 16, 4, 16, 16> c256;
const ChirpReg<float, 320, 40, 8, 4, 8, 5, 8> c320;
const ChirpReg<float, 384, 48, 4, 4, 8, 6, 8> c384;
const ChirpReg<float, 448, 56, 4, 4, 8, 7, 8> c448;
const ChirpReg<float, 512, 64, 4, 4, 8, 8, 8> c512;
const ChirpReg<float, 640, 80, 4, 4, 8, 10, 8> c640;
const ChirpReg<float, 768, 48, 4, 4, 16, 3, 16> c768;
const ChirpReg<float, 1024, 64, 4, 4, 16, 4, 16> c1024;
const ChirpReg<float, 1280, 80, 4, 3, 16, 5, 16> c1280;
const ChirpReg<float, 1536, 96, 2, 3, 16, 6, 16> c1536;
const ChirpReg<float, 1792, 112, 2, 3, 16, 7, 16> c1792;
const ChirpReg<float, 2048, 128, 2, 4, 16, 8, 16> c2048;
const ChirpReg<float, 2560, 256, 1, 3, 16, 10, 16> c2560;
const ChirpReg<float, 3072, 256, 1, 3, 16, 12, 16> c3072;
const ChirpReg<float, 3840, 256, 1, 3, 16, 15, 16> c3840;
const ChirpReg<float, 4096, 256, 1, 4, 16, 16, 16> c4096;
}  // namespace
}  // namespace sfft
