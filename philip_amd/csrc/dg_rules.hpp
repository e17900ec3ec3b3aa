// Rules by which the host chooses a kernel or a store policy from sizes and types.  Plain constexpr
// functions without HIP, so that tests read them on the CPU.  Each was measured on an MI355X (256
// compute units, 256 MB last-level cache); both sides of every line are given.
#pragma once

namespace dgx {

// Low-storage RK: whether the next stage's state is stored to stay in the caches for that stage's
// read, or streamed like the other registers (stage_epilogue).  mb: size of the state in 10^6 bytes;
// line: a line kernel, else stage2_kernel.  Step, streamed -> cached:
//   below 12 MB the end of the launch writes the dirty lines back and nothing is won: mixed 3D p=3
//     8.6 MB 78 -> 82 us, p=5 104 -> 110; FP64 p=2 8.6 MB 103 -> 108; conservative mixed p=4 3.6 MB
//     55 -> 61, 2D p=3 3.2 MB 34 -> 40; 2D p=1 and p=2 win earlier: conservative mixed 3.2 MB 48 -> 51,
//     43 -> 45, 7.1 MB 92 -> 80, 82 -> 74
//   box, line kernels: FP64 3D p=3 62 MB 510 -> 483, 119 MB 934 -> 896, 250 MB and above the same
//     within 1 %; mixed 119 MB 753 -> 714; 2D p=1 96 MB 1390 -> 999 and 320 MB 1.37 times
//   stage2_kernel: the state is not the largest part of its traffic.  Conservative, 3D, FP64 p=6 18 MB
//     324 -> 315, 56 MB 857 -> 813, 127 MB 1949 -> 1973; mixed p=3 20 MB 148 -> 155, p=2 84 MB 1.02
//     times, 119 MB 867 -> 883; 2D p=1 and p=2 always (96 MB 996 -> 840, 864 -> 737), p=3 48 MB 257 ->
//     261, p=4 48 MB 316 -> 296, p=5 134 MB 0.96 times
//   curvilinear, 3D from p=3: the metric terms need the cache.  FP64 p=3 62 MB 628 -> 584, 84 MB 0.95
//     times, 119 MB 1192 -> 1201, p=4 122 MB 1772 -> 1781; p=1 59 MB 781 -> 710, 170 MB and above 1.02
constexpr bool store_stays_cached(int dim, int n, bool line, bool curved, double mb)
{
    if (mb < (dim == 2 && n <= 3 ? 6.0 : 12.0)) return false;
    if (curved && dim == 3 && n >= 4) return mb <= 64.0;
    if (!line && dim == 3) return mb >= 40.0 && mb <= 100.0;
    if (!line && n >= 4) return mb <= 100.0;
    return true;
}

} // namespace dgx
