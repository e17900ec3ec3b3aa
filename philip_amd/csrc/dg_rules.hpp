// Rules by which the host chooses a kernel or a store policy from sizes and types.  Plain constexpr
// functions without HIP, so that tests read them on the CPU.  Each was measured on an MI355X (256
// compute units, 256 MB last-level cache); both sides of every line are given.
#pragma once

namespace dgx {

// Volume form of an FP64 line kernel: Chandrashekar / Ranocha split form, the split form with one of
// the other two-point fluxes (a kernel of its own: the generic evaluation sets the register count of
// a kernel that holds both -- p=3: 153 VGPRs, the curved kernel 246), the conservative form.
enum LineForm { FORM_EC = 0, FORM_GEN = 1, FORM_CONS = 2 };

// Elements of a 256-node block, and of a small meshes' block: what fills half a wave per (direction,
// part) of line items.
constexpr int block_elements(int dim, int n)
{
    const int np = dim == 3 ? n * n * n : n * n;
    return np >= 256 ? 1 : 256 / np;
}
constexpr int small_elements(int dim, int n)
{
    return dim == 2 ? (n == 2 ? 16 : n == 3 ? 10 : n == 4 ? 8 : n == 5 ? 6 : n == 6 ? 5 : 4)
                    : (n == 2 ? 8 : n == 3 ? 3 : n == 4 ? 2 : 1);
}

// Whether the line kernel of a form has the small meshes' block (the mixed kernels hold every two-point
// flux in FORM_EC).  FP64 3D p=6 would spill; at 2D p=3 the conservative form and the generic fluxes
// gain nothing (right-hand side, other kernel -> small: 4.5 -> 4.7 us; Ismail-Roe 13.3 -> 14.5).
constexpr bool has_small_block(int dim, int n, bool fp64, int form)
{
    if (!fp64) return form == FORM_EC;
    if (dim == 3 && n == 7) return false;
    return form == FORM_EC || !(dim == 2 && n == 4);
}

// Whether a mesh, or the solves of a batched launch, of `blocks` 256-node blocks takes the small ones
// (`small` of them).  With at most a block per compute unit a launch is bound by the length of one
// block's chain, not by throughput.  Right-hand side, default -> small: FP64 at 0.5 blocks per unit 2D
// p=2 7.5 -> 5.6 us, p=4 8.6 -> 5.9, p=6 10.7 -> 7.3; 3D p=1 9.4 -> 6.1, p=3 9.1 -> 6.6, p=5 12.6 -> 8.2;
// Kennedy-Gruber 3D p=3 9.8 -> 6.9, 2D p=5 14.4 -> 7.5; at one block 2D p=3 7.1 -> 5.9, 3D p=2 10.1 and
// 10.2, p=4 11.7 and 12.3.  Mixed 3D, whose default block has twice the elements at p=3, p=4, p=6: 1.0
// blocks p=3 10.1 -> 6.5, p=4 13.0 -> 8.0, 1.7 blocks p=3 10.3 -> 13.9, 1.3 blocks p=6 17.7 -> 23.2.
// Conservative form (phase kernel -> small) in 3D: as soon as a unit has more than two small blocks it
// loses, p=2 444 blocks 9.0 -> 8.6, 576 blocks 9.0 -> 11.7, p=1 512 blocks 8.8 -> 7.9, 729 blocks 9.0 ->
// 10.5; in 2D it does not, p=1 702 blocks 6.4 -> 5.3, p=2 689 blocks 6.5 -> 5.9.
constexpr bool takes_small_block(int dim, int n, bool fp64, int form, int blocks, int small, int n_cu)
{
    if (!has_small_block(dim, n, fp64, form) || blocks > n_cu) return false;
    return form != FORM_CONS || dim == 2 || small <= 2 * n_cu;
}

// Whether the solves of a batched launch, of `blocks` 256-node blocks in all, take the small meshes' tile
// without timing.  RK4 step, default tile -> small, FP64: 2D p=4 0.5 blocks per unit 58 -> 46 us, 1.0 blocks
// 69 -> 62; 3D p=3 57 -> 46 and 67 -> 62, p=6 84 -> 68 and 104 -> 88.  In 3D at p=2, and FP64 at p=1 and p=4,
// the small blocks of one unit's worth of default ones no longer fit the chip at once: FP64 p=1 67 -> 48 and
// 80 -> 88, p=2 64 -> 51 and 75 -> 83, p=4 69 -> 50 and 79 -> 91, mixed p=2 63 -> 48 and 74 -> 73.
constexpr bool batch_takes_small_tile(int dim, int n, bool fp64, long blocks, int n_cu)
{
    const bool half = dim == 3 && (n == 3 || (fp64 && (n == 2 || n == 5)));
    return blocks <= (half ? n_cu / 2 : n_cu);
}

// FP64 conservative form on the box, the small meshes' block apart: whether `blocks` 256-node blocks go
// to the line kernel, else to stage2_kernel.  The line kernel, in 3D up to p=5, needs half the time at
// many blocks per compute unit and more than the phase kernel at few; in a stage of a step, whose
// registers it loads ahead, it wins from one block on (p=3 12^3, 1.7 blocks: 5 stages 71 -> 62 us, p=5
// 7^3, 1.3 blocks: 69 -> 64).  Right-hand side, stage2_kernel ->
// line kernel, Roe and Lax-Friedrichs: p=3 0.7 blocks per unit 7.1 -> 9.2 and 5.9 -> 8.4 us, 1.7 blocks
// 9.8 -> 10.3 and 7.7 -> 9.4, 3.3 blocks 17.8 -> 14.4 and 13.9 -> 12.4, 24 blocks 89 -> 64 and 72 -> 56; p=5
// 2.0 blocks 10.2 -> 11.0 and 7.9 -> 9.9, 3.9 blocks 19.4 -> 14.8 and 15.6 -> 13.2; p=2 at 1.5 blocks
// already 12.9 -> 10.9 and 9.3 -> 9.5.  With boundary faces the line kernel is the faster one
// throughout (p=3 0.3 blocks 9.6 and 9.6, 1.7 blocks 13.4 -> 10.9) but for p=1 (0.7 blocks 11.5 -> 12.3,
// 1.5 blocks 16.2 -> 14.4).  Elsewhere stage2_kernel is: 2D p=4 300^2 62 against 67 us, 3D p=6 14^3 71
// against 77 us.
constexpr bool has_conservative_line(int dim, int n) { return dim == 3 && n <= 6; }
constexpr bool takes_conservative_line(int dim, int n, bool boundary, bool stage, int blocks, int n_cu)
{
    if (!has_conservative_line(dim, n)) return false;
    if (boundary) return n != 2 || blocks > n_cu;
    return blocks > (n == 3 || stage ? 1 : 2) * n_cu;
}

// Whether a line kernel loads a Butcher stage's registers before the line sums go to LDS rather than in
// the epilogue.  Mixed RK4 step, epilogue -> before: 2D p=3 96 MB 454 -> 377 us, 3D p=3 119 MB 769 -> 626,
// Navier-Stokes p=5 16^3 stage with the lifted gradient 147 -> 129; but 2D p=1 48 MB 212 -> 257, p=2 216 ->
// 235 (96 MB 540 -> 496).
constexpr bool butcher_prefetch(int dim, int n, bool fp64) { return fp64 || dim == 3 || n >= 4; }

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
//     324 -> 315, 24 MB 386 -> 367, 56 MB 857 -> 813, 127 MB 1949 -> 1973; mixed p=3 20 MB 148 -> 155, p=2 84 MB 1.02
//     times, 119 MB 867 -> 883; 2D p=1 and p=2 always (96 MB 996 -> 840, 864 -> 737), p=3 48 MB 257 ->
//     261, p=4 48 MB 316 -> 296, p=5 134 MB 0.96 times
//   curvilinear, 3D from p=3: the metric terms need the cache.  FP64 p=3 62 MB 628 -> 584, 84 MB 0.95
//     times, 119 MB 1192 -> 1201, p=4 122 MB 1772 -> 1781; p=1 59 MB 781 -> 710, 170 MB and above 1.02
constexpr bool store_stays_cached(int dim, int n, bool fp64, bool line, bool curved, double mb)
{
    if (mb < (dim == 2 && n <= 3 ? 6.0 : 12.0)) return false;
    if (curved && dim == 3 && n >= 4) return mb <= 64.0;
    if (!line && dim == 3) return mb >= (fp64 ? 12.0 : 40.0) && mb <= 100.0;
    if (!line && n >= 4) return mb <= 100.0;
    return true;
}

} // namespace dgx
