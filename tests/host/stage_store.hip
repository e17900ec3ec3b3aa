// One low-storage RK stage's epilogue alone, for a look at its stores in the assembly.
#include "../../philip_amd/csrc/dg_kernels.hpp"
using namespace dgx;

extern "C" __global__ void lsrk_epilogue(StageArgs a, Ops1D ops, const double *u, const double *r)
{
    constexpr int NS = 4;
    double ud[NS], acc[NS];
    const int c[3] = {0, 0, 0}, i = threadIdx.x;
    a.mode = MODE_LSRK;
    a.lsrk_first = 0;
    a.s4 = nullptr;
    for (int s = 0; s < NS; ++s) {
        ud[s] = u[i + s];
        acc[s] = r[i + s];
    }
    stage_epilogue<2, 2, double>(a, ops, blockIdx.x, i, c, ud, acc);
}
