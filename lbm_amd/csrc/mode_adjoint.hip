// Adjoint, objective and fp64 dual-number (forward-mode) kernels, D3Q15/19/27.
#include "kernels_adj2.hpp"
#include "kernels_adjoint.hpp"
#include "ops_adjoint.hpp"
#include "ops_impl.hpp"

namespace lbm_amd {

namespace {

template <class L, Mode M>
struct AdjImpl {
    using Calc = typename StorageOf<M>::Calc;

    static hipError_t backward_step(const AdjArgs& a, const StepPlan& p, bool brink, hipStream_t s) {
        if (p.has_bulk) {
            if (brink)
                hipLaunchKernelGGL((k_adj_bulk<L, M, true>), dim3(static_cast<uint32_t>(p.nblocks_bulk)),
                                   dim3(p.BX, p.BY), 0, s, a, p.nbx, p.nby);
            else
                hipLaunchKernelGGL((k_adj_bulk<L, M, false>), dim3(static_cast<uint32_t>(p.nblocks_bulk)),
                                   dim3(p.BX, p.BY), 0, s, a, p.nbx, p.nby);
        }
        if (a.nb > 0) {
            const uint32_t nblk = static_cast<uint32_t>((a.nb + 127) / 128);
            if (brink)
                hipLaunchKernelGGL((k_adj_near<L, M, true>), dim3(nblk), dim3(128), 0, s, a);
            else
                hipLaunchKernelGGL((k_adj_near<L, M, false>), dim3(nblk), dim3(128), 0, s, a);
        }
        return hipGetLastError();
    }

    template <Mode MM>
    static hipError_t objective_impl(const FieldLayout& Ly, const void* src, const uint8_t* kind, int obj,
                                     int plane, const double* target, double* partial, int nblocks,
                                     double* out, hipStream_t s) {
        hipLaunchKernelGGL((k_objective<L, MM>), dim3(nblocks), dim3(256), 0, s, Ly, src, kind, obj, plane,
                           target, partial);
        hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, s, partial, nblocks, out);
        return hipGetLastError();
    }

    static hipError_t to_dual(const FieldLayout& Ly, const void* src, void* dst, hipStream_t s) {
        const uint32_t nblk = static_cast<uint32_t>((Ly.plane + 255) / 256);
        hipLaunchKernelGGL((k_to_dual<L, M>), dim3(nblk), dim3(256), 0, s, Ly, src,
                           static_cast<Dual<double>*>(dst), 0);
        return hipGetLastError();
    }

    template <int V>
    static void launch_hist_step(const StepArgs& a, const StepPlan& p, hipStream_t s) {
        const dim3 grid(static_cast<uint32_t>(p.nblocks_bulk)), block(p.BX, p.BY, 1);
        if (p.brink)
            hipLaunchKernelGGL((k_bulk<L, M, V, false, true, true>), grid, block, 0, s, a, p.nbx, p.nby);
        else
            hipLaunchKernelGGL((k_bulk<L, M, V, false, false, true>), grid, block, 0, s, a, p.nbx, p.nby);
    }
    static hipError_t hist_step(const StepArgs& a, const StepPlan& p, hipStream_t s) {
        if (p.V == 2)
            launch_hist_step<2>(a, p, s);
        else if (p.V == 1)
            launch_hist_step<1>(a, p, s);
        else
            return hipErrorInvalidValue;
        return hipGetLastError();
    }
    static hipError_t hist_backward(const AdjArgs& a, const StepPlan& p, bool brink, hipStream_t s) {
        const dim3 grid(static_cast<uint32_t>(p.nblocks_bulk)), block(p.BX, p.BY);
        if (brink)
            hipLaunchKernelGGL((k_adj_hist<L, M, true>), grid, block, 0, s, a, p.nbx, p.nby);
        else
            hipLaunchKernelGGL((k_adj_hist<L, M, false>), grid, block, 0, s, a, p.nbx, p.nby);
        return hipGetLastError();
    }
    template <bool BRINK, bool CACHED>
    static void launch_hist_step2(const StepArgs& a, const StepPlan& p, hipStream_t s) {
        hipLaunchKernelGGL((k_bulk2<L, M, BRINK, CACHED, true>), dim3(static_cast<uint32_t>(p.tb_nblocks)), dim3(256), 0, s,
                           a, p.tb_ntx, p.tb_nty, p.tb_zc, p.tb_nxcd);
    }
    static hipError_t hist_step2(const StepArgs& a, const StepPlan& p, hipStream_t s) {
        if constexpr (M == Mode::F32) {
            if (p.brink)
                a.cached ? launch_hist_step2<true, true>(a, p, s) : launch_hist_step2<true, false>(a, p, s);
            else
                a.cached ? launch_hist_step2<false, true>(a, p, s) : launch_hist_step2<false, false>(a, p, s);
            return hipGetLastError();
        } else {
            return hipErrorInvalidValue;
        }
    }
    template <bool BRINK, bool CACHED>
    static void launch_adj2(const AdjArgs& a, const StepPlan& p, hipStream_t s) {
        hipLaunchKernelGGL((k_adj2<L, BRINK, CACHED>), dim3(static_cast<uint32_t>(p.tb_nblocks)), dim3(256), 0, s, a,
                           p.tb_ntx, p.tb_nty, p.tb_zc, p.tb_nxcd);
    }
    static hipError_t hist_backward2(const AdjArgs& a, const StepPlan& p, bool brink, hipStream_t s) {
        if constexpr (M == Mode::F32) {
            if (brink)
                a.cached ? launch_adj2<true, true>(a, p, s) : launch_adj2<true, false>(a, p, s);
            else
                a.cached ? launch_adj2<false, true>(a, p, s) : launch_adj2<false, false>(a, p, s);
            return hipGetLastError();
        } else {
            return hipErrorInvalidValue;
        }
    }

    static AdjOps make() {
        AdjOps o{};
        o.backward_step = &backward_step;
        o.objective = &objective_impl<M>;
        o.objective_dual = &objective_impl<Mode::DUAL64>;
        o.to_dual = &to_dual;
        o.dual_step = &OpsImpl<L, Mode::DUAL64>::template step_impl<1>;
        o.hist_step = &hist_step;
        o.hist_step2 = M == Mode::F32 ? &hist_step2 : nullptr;
        o.hist_backward = &hist_backward;
        o.hist_backward2 = M == Mode::F32 ? &hist_backward2 : nullptr;
        o.calc_bytes = sizeof(Calc);
        return o;
    }
};

const AdjOps kF32[3] = {AdjImpl<D3Q15, Mode::F32>::make(), AdjImpl<D3Q19, Mode::F32>::make(),
                        AdjImpl<D3Q27, Mode::F32>::make()};
const AdjOps kF64S[3] = {AdjImpl<D3Q15, Mode::F64S>::make(), AdjImpl<D3Q19, Mode::F64S>::make(),
                         AdjImpl<D3Q27, Mode::F64S>::make()};

}  // namespace

const AdjOps* adj_ops(int q, Mode m) {
    const int i = q == 15 ? 0 : (q == 19 ? 1 : (q == 27 ? 2 : -1));
    if (i < 0) return nullptr;
    if (m == Mode::F32) return &kF32[i];
    if (m == Mode::F64S) return &kF64S[i];
    return nullptr;
}

}  // namespace lbm_amd
