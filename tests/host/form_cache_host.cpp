// Host build of what an FP64 line kernel's node cache keeps (philip_amd/csrc/dg_fast.hpp).  Reads
// n two_point and n lines of ua[5] ub[5]; prints per line the two-point flux along e_0 of the nodes,
// of the nodes as the cache gives them back, and of the generic evaluation on the states.
#include <cmath>
#include <cstdio>
#define __device__
#define __forceinline__ inline
#define DGX_HOST_TEST
#include "../../philip_amd/csrc/dg_fast.hpp"
using namespace dgx;

// the fields that are stored, and nothing else
static NodeC<double, 3> cached(const FastConst<double> &fc, NodeC<double, 3> n)
{
    node_to_cache64<3, FORM_GEN>(fc, n);
    NodeC<double, 3> m;
    for (double &x : m.u) x = NAN;
    m.u[0] = n.u[0];
    for (int k = 0; k < 3; ++k) m.vel[k] = n.vel[k];
    m.p = n.p;
    m.b = n.b;
    m.v2 = m.h = m.c = m.sr = NAN;  // not read by a two-point flux
    node_from_cache64<3, FORM_GEN>(m);
    return m;
}

int main()
{
    int n;
    PhysConst pc{};
    if (scanf("%d %d", &n, &pc.two_point) != 2) return 1;
    pc.gam = 1.4;
    pc.gamm1 = pc.gam - 1.0;
    const FastConst<double> fc = fast_const<double>(pc);
    for (int i = 0; i < n; ++i) {
        NodeC<double, 3> a, b;
        for (double &x : a.u)
            if (scanf("%lf", &x) != 1) return 1;
        for (double &x : b.u)
            if (scanf("%lf", &x) != 1) return 1;
        node_fill<double, 3>(a, fc);
        node_fill<double, 3>(b, fc);
        Prim<double, 3> qa, qb;
        qa.rho = a.u[0];
        qb.rho = b.u[0];
        for (int k = 0; k < 3; ++k) {
            qa.vel[k] = a.vel[k];
            qb.vel[k] = b.vel[k];
        }
        qa.p = a.p;
        qb.p = b.p;
        double f[3][5];
        other_flux64<3, 0, false>(a, b, nullptr, pc, f[0]);
        other_flux64<3, 0, false>(cached(fc, a), cached(fc, b), nullptr, pc, f[1]);
        two_point_flux_dir<double, 3>(a.u, qa, b.u, qb, 0, pc, f[2]);
        for (auto &r : f)
            for (double x : r) printf("%.17e ", x);
        printf("\n");
    }
    return 0;
}
