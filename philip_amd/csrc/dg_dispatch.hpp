// Kernel dispatch templates over (dim, nodes per direction, scheme, precision): the stage
// kernels, the auxiliary (lifted-gradient) kernel and the batched line kernel.  Each N is
// instantiated in its own translation unit (dg_inst_n<N>.hip) so the kernels compile in
// parallel; dg_launch.hip calls the instantiations.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "dg_host.hpp"
#include "dg_line.hpp"
#include "dg_rules.hpp"
#include "dg_stage2.hpp"

namespace dgx {

inline int check_launch(dgx_ctx *c, const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        c->err = std::string(what) + ": " + hipGetErrorString(e);
        return DGX_ERR_HIP;
    }
    return DGX_OK;
}

// The small meshes' block of the line kernel, if the mesh is one (takes_small_block); tells whether it
// was launched.
template <int D, int N, typename T, int FORM>
bool line_small_dn(dgx_ctx *c, const StageArgs &a)
{
    constexpr bool FP64 = std::is_same<T, double>::value;
    if constexpr (has_small_block(D, N, FP64, FORM)) {
        using LS = LineGeoSmall<D, N, T>;
        const int blocks = (c->ncells + block_elements(D, N) - 1) / block_elements(D, N);
        const int small = (c->ncells + LS::EPB - 1) / LS::EPB;
        if (c->has_boundary || !takes_small_block(D, N, FP64, FORM, blocks, small, c->n_cu)) return false;
        hipLaunchKernelGGL((line_kernel_small<D, N, T, FORM>), dim3(small),
                           dim3(LS::BLOCK), 0, c->stream, a, c->ops, c->pc);
        return true;
    }
    return false;
}

// Euler on the box in the line kernel, with boundary faces or without.
template <int D, int N, typename T, int FORM>
void line_dn(dgx_ctx *c, const StageArgs &a)
{
    using LG = LineGeoS<D, N, T>;
    if (line_small_dn<D, N, T, FORM>(c, a)) return;
    auto go = [&](auto bc) {
        constexpr bool BND = decltype(bc)::value;
        const dim3 grid((c->ncells + LG::EPB - 1) / LG::EPB), block(LG::BLOCK);
        if constexpr (line_waves<D, N, T>() > 0)
            hipLaunchKernelGGL((line_kernel_wb<D, N, T, line_waves<D, N, T>(), BND, FORM>), grid, block, 0, c->stream,
                               a, c->ops, c->pc);
        else
            hipLaunchKernelGGL((line_kernel<D, N, T, BND, FORM>), grid, block, 0, c->stream, a, c->ops, c->pc);
    };
    if (c->has_boundary) go(std::true_type{});
    else go(std::false_type{});
}

// Stage kernel of a context.  FP64: the line kernel, but for walls with the viscous terms, boundary
// faces on a curvilinear grid, and Kennedy-Gruber or Ismail-Roe fluxes with the viscous terms or on a
// curvilinear grid, which are stage2_kernel's, as the conservative form on the box is in 2D, at p=6 and
// on meshes of few blocks (takes_small_block, takes_conservative_line).  Mixed: the line kernel for the periodic split form and
// for Euler boundary faces on the box, stage2_kernel for the rest.
template <int D, int N, typename T>
void stage2_dn(dgx_ctx *c, StageArgs a, dim3 grid, dim3 block)
{
    constexpr bool FP64 = std::is_same<T, double>::value;
    const bool split = c->P.use_split_form != 0, bnd = c->has_boundary, curv = c->curv;
    const bool nsv = D == 3 && c->P.pde == DGX_NAVIER_STOKES;
    const double mb = 1e-6 * sizeof(double) * c->ncells * Geo<D, N>::NS * Geo<D, N>::NP;
    a.s1_cached = store_stays_cached(D, N, FP64, true, curv, mb);
    if (!nsv && !curv) {
        if constexpr (FP64) {
            if (!split && line_small_dn<D, N, T, FORM_CONS>(c, a)) return;
            if constexpr (has_conservative_line(D, N))
                if (!split && takes_conservative_line(D, N, bnd, a.mode == MODE_LSRK || a.mode == MODE_BUTCHER,
                                                      (int)grid.x, c->n_cu))
                    return line_dn<D, N, T, FORM_CONS>(c, a);
            if (split && c->pc.two_point < 2) return line_dn<D, N, T, FORM_GEN>(c, a);
        }
        if (split) return line_dn<D, N, T, FORM_EC>(c, a);
    }
    if constexpr (FP64) {
        if ((nsv || curv) && !bnd && (!split || c->pc.two_point >= 2)) {
            auto go = [&](auto vc, auto cc, auto fc) {
                constexpr bool V = decltype(vc)::value, CV = decltype(cc)::value;
                constexpr int FORM = decltype(fc)::value ? FORM_CONS : FORM_EC;
                using LV = LineGeoK<D, N, T, V>;
                hipLaunchKernelGGL((line64_kernel<D, N, V, CV, FORM>), dim3((c->ncells + LV::EPB - 1) / LV::EPB),
                                   dim3(LV::BLOCK), 0, c->stream, a, c->ops, c->pc);
            };
            auto form = [&](auto vc, auto cc) {
                if (split) go(vc, cc, std::false_type{});
                else go(vc, cc, std::true_type{});
            };
            if constexpr (D == 3) {
                if (nsv) {
                    if (curv) form(std::true_type{}, std::true_type{});
                    else form(std::true_type{}, std::false_type{});
                    return;
                }
            }
            return form(std::false_type{}, std::true_type{});
        }
    } else if constexpr (D == 3) {
        if (nsv && split && !curv && !bnd) {
            using LV = LineGeoK<D, N, T, true>;
            const dim3 vgrid((c->ncells + LV::EPB - 1) / LV::EPB), vblock(LV::BLOCK);
            if constexpr (N == 6)
                hipLaunchKernelGGL((line_kernel_ns_w4<D, N>), vgrid, vblock, 0, c->stream, a, c->ops, c->pc);
            else
                hipLaunchKernelGGL((line_kernel_ns<D, N>), vgrid, vblock, 0, c->stream, a, c->ops, c->pc);
            return;
        }
    }
    a.s1_cached = store_stays_cached(D, N, FP64, false, curv, mb);
    auto go2 = [&](auto sc, auto vc, auto bc, auto cc) {
        hipLaunchKernelGGL((stage2_kernel<D, N, decltype(sc)::value, decltype(vc)::value, T, decltype(bc)::value,
                                          decltype(cc)::value>),
                           grid, block, 0, c->stream, a, c->ops, c->pc);
    };
    const std::true_type yes{};
    const std::false_type no{};
    if constexpr (D == 3) {
        if (nsv && curv) {
            if (split) go2(yes, yes, yes, yes);
            else go2(no, yes, yes, yes);
            return;
        }
        if (nsv && bnd) {
            if (split) go2(yes, yes, yes, no);
            else go2(no, yes, yes, no);
            return;
        }
        if (nsv) {
            // FP64: Kennedy-Gruber or Ismail-Roe; mixed: the conservative form
            if constexpr (FP64) go2(yes, yes, no, no);
            else go2(no, yes, no, no);
            return;
        }
    }
    if (curv) {
        if (split) go2(yes, no, yes, yes);
        else go2(no, no, yes, yes);
        return;
    }
    if (bnd) go2(no, no, yes, no);  // conservative Euler on the box
    else go2(no, no, no, no);
}

template <int D, int N>
void stage_dn(dgx_ctx *c, const StageArgs &a, dim3 grid, dim3 block)
{
    // FP64: fluxes in double; mixed: fluxes and contractions in float, state and RK registers
    // in double.  The reference's entropy projection u(v(u)) is the identity for collocated GLL
    // nodes and is formed by neither.
    if (c->P.precision == DGX_MIXED) stage2_dn<D, N, float>(c, a, grid, block);
    else stage2_dn<D, N, double>(c, a, grid, block);
}

template <int D, int N>
int launch_stage_dn(dgx_ctx *c, const StageArgs &a)
{
    using S = Geo<D, N>;
    const int blocks = (c->ncells + S::EPB - 1) / S::EPB;
    if (c->timing.enabled && hipEventRecord(c->timing.a, c->stream) != hipSuccess) {
        c->err = "hipEventRecord failed";
        return DGX_ERR_HIP;
    }
    stage_dn<D, N>(c, a, dim3(blocks), dim3(S::BLOCK));
    int rc = check_launch(c, "stage_kernel");
    if (rc) return rc;
    if (c->timing.enabled) {
        float ms = 0.f;
        if (hipEventRecord(c->timing.b, c->stream) != hipSuccess || hipEventSynchronize(c->timing.b) != hipSuccess ||
            hipEventElapsedTime(&ms, c->timing.a, c->timing.b) != hipSuccess) {
            c->err = "stage kernel timing failed";
            return DGX_ERR_HIP;
        }
        c->timing.sum_ms += ms;
        c->timing.n += 1;
    }
    return DGX_OK;
}

template <int D, int N>
int launch_aux_dn(dgx_ctx *c, const double *u)
{
    using S = Shape<D, N>;
    const int blocks = (c->ncells + S::EPB - 1) / S::EPB;
    auto go = [&](auto cc, auto *q0, auto *q1, auto *q2) {
        using Q = std::remove_pointer_t<decltype(q0)>;
        hipLaunchKernelGGL((aux_kernel<D, N, Q, decltype(cc)::value>), dim3(blocks), dim3(S::BLOCK), 0, c->stream, u,
                           q0, q1, q2, c->nbr_dev, c->ncells, 1.0 / c->h, c->ops, c->pc,
                           c->curv ? c->met_dev : nullptr);
    };
    auto grid = [&](auto *q0, auto *q1, auto *q2) {
        if (c->curv) go(std::true_type{}, q0, q1, q2);
        else go(std::false_type{}, q0, q1, q2);
    };
    if (c->P.precision == DGX_MIXED) grid(c->auxf_dev[0], c->auxf_dev[1], c->auxf_dev[2]);
    else grid(c->aux_dev[0], c->aux_dev[1], c->aux_dev[2]);
    return check_launch(c, "aux_kernel");
}

template <int D, int N, typename T, int ES, int W, int XJ, bool GEN>
int line_batch_es(const BatchBlock *blocks, int nblocks, const StageArgs *args, const PhysConst *pcs,
                  const Ops1D &ops, hipStream_t st, int *epb, int *threads)
{
    using LG = LineGeo<D, N, T, ES, false, XJ>;
    if constexpr (LG::SBUF * sizeof(T) > 160 * 1024 - 4096 || LG::BLOCK > 1024) {
        return DGX_ERR_UNSUPPORTED;  // would not fit the 160 KB of LDS or the 1024 threads of a block
    } else {
        if (epb) *epb = LG::EPB;
        if (threads) *threads = LG::BLOCK;
        if (!blocks) return DGX_OK;  // query only
        if constexpr (W > 0)
            hipLaunchKernelGGL((line_kernel_batch_wb<D, N, T, ES, W, XJ, GEN>), dim3(nblocks), dim3(LG::BLOCK), 0, st,
                               blocks, args, pcs, ops);
        else
            hipLaunchKernelGGL((line_kernel_batch<D, N, T, ES, XJ, GEN>), dim3(nblocks), dim3(LG::BLOCK), 0, st, blocks,
                               args, pcs, ops);
        return hipGetLastError() == hipSuccess ? DGX_OK : DGX_ERR_HIP;
    }
}

template <int D, int N, typename T, bool GEN>
int line_batch_t(int tile, const BatchBlock *blocks, int nblocks, const StageArgs *args, const PhysConst *pcs,
                 const Ops1D &ops, hipStream_t st, int *epb, int *threads)
{
    constexpr bool F = std::is_same<T, float>::value;
#define LBT_CASE(V)                                                                                              \
    case V:                                                                                                      \
        return line_batch_es<D, N, T, batch_tile<D, N>(F, V).es, batch_tile<D, N>(F, V).waves, batch_tile<D, N>(F, V).xj, GEN>( \
            blocks, nblocks, args, pcs, ops, st, epb, threads);
    if constexpr (D == 2) {
        switch (tile) {
            LBT_CASE(0) LBT_CASE(1) LBT_CASE(2) LBT_CASE(3) LBT_CASE(4) LBT_CASE(5)
            LBT_CASE(6) LBT_CASE(7) LBT_CASE(8) LBT_CASE(9) LBT_CASE(10) LBT_CASE(11) LBT_CASE(12)
        default: return DGX_ERR_UNSUPPORTED;
        }
    } else {
        switch (tile) {
            LBT_CASE(0) LBT_CASE(1) LBT_CASE(2)
        default: return DGX_ERR_UNSUPPORTED;
        }
    }
#undef LBT_CASE
}

template <int D, int N>
int line_batch_dn(int precision, bool generic, int tile, const BatchBlock *blocks, int nblocks, const StageArgs *args,
                  const PhysConst *pcs, const Ops1D &ops, hipStream_t st, int *epb, int *threads)
{
    if (tile < 0 || tile >= batch_tile_count(D)) return DGX_ERR_UNSUPPORTED;
    if (precision == DGX_MIXED)
        return line_batch_t<D, N, float, false>(tile, blocks, nblocks, args, pcs, ops, st, epb, threads);
    if (generic) return line_batch_t<D, N, double, true>(tile, blocks, nblocks, args, pcs, ops, st, epb, threads);
    return line_batch_t<D, N, double, false>(tile, blocks, nblocks, args, pcs, ops, st, epb, threads);
}

// explicit instantiation (in dg_inst_n<NN>.hip) and its extern declaration (in dg_launch.hip)
#define DGX_KERNELS_N(PREFIX, NN)                                                                          \
    PREFIX template int launch_stage_dn<2, NN>(dgx_ctx *, const StageArgs &);                              \
    PREFIX template int launch_stage_dn<3, NN>(dgx_ctx *, const StageArgs &);                              \
    PREFIX template int launch_aux_dn<3, NN>(dgx_ctx *, const double *);                                   \
    PREFIX template int line_batch_dn<2, NN>(int, bool, int, const BatchBlock *, int, const StageArgs *,          \
                                             const PhysConst *, const Ops1D &, hipStream_t, int *, int *);   \
    PREFIX template int line_batch_dn<3, NN>(int, bool, int, const BatchBlock *, int, const StageArgs *,          \
                                             const PhysConst *, const Ops1D &, hipStream_t, int *, int *);

} // namespace dgx
