// fixed_col_mixed.hip -- compile-time column passes of two-pass plans for the
// mixed-radix column lengths the planner picks (by bytes) for FP32 lengths
// between 16384 and 2^18; radices as the runtime planner's cost model chooses
// them at 16 elements per thread.  Unpadded LDS: over the 185 fast lengths in
// (16384, 2^18] two-pass throughput is 1730 vs 1719 GB/s with the one-in-16 pad
// (up to 8 % faster on single lengths).  Columns per block as in fixed_col.hip:
// paired modes, first pass, second pass, each the fastest of 8, 16, 32 and 64
// measured (81 first pass: 64 columns 112 us, 32 131, 16 149; 375 second pass: 8
// 87, 16 91, 32 121).  The first pass reads its input non-temporally (Sched NT
// 1): two-pass lengths in [16000, 2^18] +6 % (median), R2C +4 %.
#include "fixed.h"

namespace sfft {
namespace {
const FixedCol<float, 480, 32, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15, 2> col480;
const FixedCol<float, 375, 25, 16, 16, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 25, 15> col375;
const FixedCol<float, 486, 54, 16, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 6> col486;
const FixedCol<float, 405, 45, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 5> col405;
const FixedCol<float, 500, 50, 16, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 10, 5> col500;
const FixedCol<float, 400, 25, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 25, 16> col400;
const FixedCol<float, 384, 26, 16, 16, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 8, 3> col384;
const FixedCol<float, 432, 36, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 6, 6> col432;
const FixedCol<float, 450, 30, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15, 2> col450;
const FixedCol<float, 324, 36, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 6, 6> col324;
const FixedCol<float, 320, 22, 16, 16, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 5, 4> col320;
const FixedCol<float, 250, 25, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 25, 10> col250;
const FixedCol<float, 243, 27, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 3> col243;
const FixedCol<float, 360, 24, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 8, 3> col360;
const FixedCol<float, 300, 20, 32, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 5, 4> col300;
const FixedCol<float, 270, 23, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 6, 3> col270;
const FixedCol<float, 288, 24, 32, 32, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12, 2> col288;
const FixedCol<float, 625, 25, 8, 16, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 25, 25> col625;
const FixedRowNarrow<float, 625, 25, 8, 2, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 25, 25> row625;
const FixedCol<float, 225, 15, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15> col225;
const FixedCol<float, 240, 16, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15> col240;
const FixedCol<float, 200, 13, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 25, 8> col200;
const FixedCol<float, 216, 18, 32, 32, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 6, 6, 6> col216;
const FixedCol<float, 192, 16, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 12> col192;
const FixedCol<float, 180, 15, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 12> col180;
const FixedCol<float, 162, 18, 32, 32, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 2> col162;
const FixedCol<float, 160, 16, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 10> col160;
const FixedCol<float, 150, 15, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 10> col150;
const FixedCol<float, 540, 45, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 6, 6> col540;
// 125: five threads per column (one radix-25 butterfly each, then five
// radix-5 ones) and 64 columns a block: two-pass lengths with a 125 pass
// 4-10 % faster than nine threads per column at 32 columns.  The same change
// for other lengths with idle threads in a stage measured slower (150 at five
// threads and 64 columns, 135 at nine, 250 at ten, 324 at 18: medians -2 to
// -9 %).
const FixedCol<float, 125, 5, 64, 64, 64, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 25, 5> col125;
const FixedCol<float, 729, 81, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 9> col729;
const FixedCol<float, 144, 12, 32, 64, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12> col144;
const FixedRowNarrow<float, 144, 12, 32, 1, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12> row144;
const FixedCol<float, 135, 15, 32, 32, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 9> col135;
const FixedCol<float, 81, 9, 32, 64, 32, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9> col81;
}  // namespace
}  // namespace sfft
