// chirp_f32.hip -- one-launch chirp-z kernels, FP32: convolution lengths up
// to 4096.  ChirpReg<type, rows of a longer one, M, threads per transform,
// transforms per block, minimum waves per SIMD, radices...>: mostly R b R
// with M / R threads, one radix-R butterfly each.  These kernels are bound by vector
// instructions (about 100 per element of M).  The lengths between the powers of
// two are those that beat the next one when all took sixteen elements a thread
// (1280, 1792, 2560 and 3840 did not).  Against the eight of 512 to 4096 now,
// both directions, 1 / 512 / 4096 transforms, this length / the next power of
// two: 448 (n = 223) 11.1 / 10.1, 12.9 / 11.5, 21.1 / 19.3 us, 1536 (n = 761)
// 17.3 / 11.0, 19.5 / 14.4, 71.1 / 60.8 (but 31.4 / 34.0 at 2048), so these two
// would go; 768 and 3072 take a third more than 1024 and 4096 for one transform
// and 6 to 15 % less for 4096.  Two transforms per thread, which halves the table
// loads, measured 0.62-0.98x: half the resident waves.
// 1024, 2048 and 4096 take eight elements a thread and one more stage, which
// halves a wave's registers and LDS (twice the waves).  Both directions, sixteen
// / eight: 509 x 8192 68.2 / 64.8 us, 1009 x 4096 73.4 / 68.2, x 20000 376 / 321,
// 1999 x 2048 74.4 / 70.6, 2029 x 20000 856 / 765, and one transform of 1009 17.1 /
// 11.3, of 1999 18.0 / 14.2.  The shorter radices err less too (round trips of
// the lengths that 4096 serves: 0.774 / 0.739 of the separate launches' error).
#include "chirp.h"

namespace sfft {
namespace {
const ChirpReg<float, false, 64, 8, 32, 4, 8, 8> c64;
const ChirpReg<float, false, 128, 16, 16, 4, 8, 2, 8> c128;
const ChirpReg<float, false, 192, 24, 8, 4, 8, 3, 8> c192;
const ChirpReg<float, false, 256, 16, 16, 4, 16, 16> c256;
const ChirpReg<float, false, 320, 40, 8, 4, 8, 5, 8> c320;
const ChirpReg<float, false, 384, 48, 4, 4, 8, 6, 8> c384;
const ChirpReg<float, false, 448, 56, 4, 4, 8, 7, 8> c448;
const ChirpReg<float, false, 512, 64, 4, 4, 8, 8, 8> c512;
const ChirpReg<float, false, 640, 80, 4, 4, 8, 10, 8> c640;
const ChirpReg<float, false, 768, 48, 4, 4, 16, 3, 16> c768;
const ChirpReg<float, false, 1024, 128, 2, 4, 8, 4, 4, 8> c1024;
const ChirpReg<float, false, 1536, 96, 2, 3, 16, 6, 16> c1536;
const ChirpReg<float, false, 2048, 256, 1, 4, 8, 8, 4, 8> c2048;
const ChirpReg<float, false, 3072, 256, 1, 4, 16, 16, 12> c3072;
const ChirpReg<float, false, 4096, 512, 1, 4, 8, 8, 8, 8> c4096;
}  // namespace
}  // namespace sfft
