// chirp_split.hip -- the kernels of chirp-z transforms in three launches:
// columns of N1 = 16 b (ChirpColReg<type, columns per block, radices>: 256-byte
// rows) and rows of N2, a power of two (ChirpReg<type, true, N2, threads per
// row, rows per block, minimum waves per SIMD, radices...>).  The lengths
// M = 16 b N2 are 6 to 15 percent apart.
// Rows of 1024 and 2048, and 4096 in F32, take eight elements a thread and one
// more stage: sixteen need 127 registers and 8.7 KB of LDS a wave (four waves
// a SIMD), eight half of either.  Both directions, sixteen / eight: 100003 x 64
// 288 / 269 us, 400009 x 32 720 / 674, 65537 x 16 81 / 75, FP64 100003 x 32 272
// / 244, 199999 x 8 158 / 148.
#include "chirp.h"

namespace sfft {
namespace {
const ChirpColReg<float, 32, 16, 8> c128;
const ChirpColReg<float, 32, 16, 9> c144;
const ChirpColReg<float, 32, 16, 10> c160;
const ChirpColReg<float, 32, 16, 11> c176;
const ChirpColReg<float, 32, 16, 12> c192;
const ChirpColReg<float, 32, 16, 13> c208;
const ChirpColReg<float, 32, 16, 15> c240;
const ChirpColReg<double, 16, 16, 8> d128;
const ChirpColReg<double, 16, 16, 9> d144;
const ChirpColReg<double, 16, 16, 10> d160;
const ChirpColReg<double, 16, 16, 11> d176;
const ChirpColReg<double, 16, 16, 12> d192;
const ChirpColReg<double, 16, 16, 13> d208;
const ChirpColReg<double, 16, 16, 15> d240;
const ChirpReg<float, true, 128, 16, 16, 4, 8, 2, 8> r128;
const ChirpReg<float, true, 256, 16, 16, 4, 16, 16> r256;
const ChirpReg<float, true, 512, 64, 4, 4, 8, 8, 8> r512;
const ChirpReg<float, true, 1024, 128, 2, 4, 8, 4, 4, 8> r1024;
const ChirpReg<float, true, 2048, 256, 1, 4, 8, 8, 4, 8> r2048;
const ChirpReg<float, true, 4096, 512, 1, 4, 8, 8, 8, 8> r4096;
const ChirpReg<float, true, 8192, 512, 1, 4, 16, 8, 4, 16> r8192;
const ChirpReg<float, true, 16384, 1024, 1, 4, 16, 16, 4, 16> r16384;
const ChirpReg<double, true, 64, 8, 16, 2, 8, 8> s64;
const ChirpReg<double, true, 128, 16, 8, 2, 8, 2, 8> s128;
const ChirpReg<double, true, 256, 16, 8, 2, 16, 16> s256;
const ChirpReg<double, true, 512, 64, 2, 2, 8, 8, 8> s512;
const ChirpReg<double, true, 1024, 128, 1, 4, 8, 4, 4, 8> s1024;
const ChirpReg<double, true, 2048, 256, 1, 4, 8, 8, 4, 8> s2048;
const ChirpReg<double, true, 4096, 256, 1, 2, 16, 16, 16> s4096;
const ChirpReg<double, true, 8192, 512, 1, 2, 16, 8, 4, 16> s8192;
}  // namespace
}  // namespace sfft
