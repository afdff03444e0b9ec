// Adjoint steps of bulk-only (fully periodic) domains from a recorded run.
//
// The forward run records drho and u of every cell and step (StepArgs::hist):
// 16 bytes a cell at fp32 where the populations take 4 Q. The adjoint of a
// step reads nothing else of the forward state, so the backward sweep needs
// no checkpoints and recomputes nothing, and a step moves (8 + 8 Q) instead
// of (12 Q) bytes a cell beside the porosity and its gradient.
//
// k_adj_hist does one step: reverse pull of mu, transposed collision.
// k_adj2 does two steps in one pass, the march of k_bulk2 (kernels_tb.hpp)
// with the directions reversed: step t on a 64 x 8 tile and its one-cell
// ring, mu^t through LDS, step t - 1 on the tile one plane behind, so mu is
// read and written once for both. lambda_q of a cell is mu_q of the cell at
// + c_q; a patch cell therefore sends mu_q to the tile cell x - c_q of plane
// zs - cz: cz = +1 values are read in the same iteration, cz = 0 in the next,
// cz = -1 (held one plane longer) in the one after. fp32 only; the values
// cross LDS in the arithmetic type, so a pass equals two k_adj_hist steps bit
// for bit, gradient sums included (step t's term is added before step
// t - 1's). Both steps' tile cells belong to the same thread, which keeps
// step t's gradient term in a register until the plane is finished.
#pragma once

#include "kernels_adjoint.hpp"
#include "kernels_tb.hpp"

namespace lbm_amd {

// Cells, blocks and grid as k_bulk with V = 1.
template <class L, Mode M, bool BRINK>
__global__ void __launch_bounds__(256) k_adj_hist(AdjArgs a, int nbx, int nby) {
    using IO = Io<M, L>;
    using T = typename IO::T;
    using Calc = typename IO::Calc;
    constexpr int Q = L::Q;
    const FieldLayout& Ly = a.L;
    const int b = blockIdx.x;
    const int bx = b % nbx;
    const int t = b / nbx;
    const int by = t % nby;
    const int z = 1 + t / nby;
    const int x = 1 + bx * blockDim.x + threadIdx.x;
    const int y = 1 + by * blockDim.y + threadIdx.y;
    if (x > Ly.xl || y > Ly.yl) return;
    const int64_t e = cell_elem(Ly, x, y, z);
    const Mom4<Calc> m = static_cast<const Mom4<Calc>*>(a.hist)[cell_index(Ly, x, y, z)];
    Calc lam[Q];
    if (a.terminal) {
        const T* __restrict__ gc = static_cast<const T*>(a.gcur);
        Calc gf[Q];
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            gf[q] = IO::template to_calc<q>(gc[q * Ly.plane + e]);
        });
        objective_grad<L, Calc>(a, x, y, z, gf, lam);
    } else {
        const int xm = wrap1(x - 1, Ly.xl), xp = wrap1(x + 1, Ly.xl);
        const int ym = wrap1(y - 1, Ly.yl), yp = wrap1(y + 1, Ly.yl);
        const int zm = wrap1(z - 1, Ly.zl), zp = wrap1(z + 1, Ly.zl);
        const Calc* __restrict__ mi = static_cast<const Calc*>(a.mu_in);
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            constexpr int cx = L::cx(q), cy = L::cy(q), cz = L::cz(q);
            lam[q] = mi[q * Ly.plane + cell_elem(Ly, cx > 0 ? xp : (cx < 0 ? xm : x),
                                                 cy > 0 ? yp : (cy < 0 ? ym : y), cz > 0 ? zp : (cz < 0 ? zm : z))];
        });
    }
    Calc alpha = Calc(0);
    if constexpr (BRINK) alpha = static_cast<const Calc*>(a.alpha)[e];
    Calc mu[Q];
    const Calc da = adjoint_relax<L, Calc, BRINK>(
        m.v[0], m.v[1], m.v[2], m.v[3], lam, mu, static_cast<Calc>(a.omega), alpha, static_cast<Calc>(a.tau * a.g[0]),
        static_cast<Calc>(a.tau * a.g[1]), static_cast<Calc>(a.tau * a.g[2]));
    Calc* __restrict__ mo = static_cast<Calc*>(a.mu_out);
    with_put<Put::Through>(a.cached, [&](auto pc) {
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            put<decltype(pc)::value>(mo + q * Ly.plane + e, mu[q]);
        });
    });
    if constexpr (BRINK) a.grad_alpha[e] += static_cast<double>(da);
}

// Steps t (a.hist) and t - 1 (a.hist2). Logical blocks as k_bulk2.
template <class L, bool BRINK, bool CACHED>
__global__ void __launch_bounds__(256) k_adj2(AdjArgs a, int ntx, int nty, int zc, int nxcd) {
    using S = TbSlots<L>;
    constexpr int Q = L::Q;
    static_assert(TB_PASS == TB_OUT + 1 && TB_NP - TB_CELLS <= 256, "tile cells on k < TB_OUT, the ring on the last k");
    __shared__ float lds[S::NSLOT][TB_CELLS];

    const FieldLayout& Ly = a.L;
    const int tid = threadIdx.x;
    int b = tb_logical_block(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x), nxcd);
    const int x0 = 1 + (b % ntx) * TB_TX;
    b /= ntx;
    const int y0 = 1 + (b % nty) * TB_TY;
    b /= nty;
    const int z0 = 1 + b * zc;
    const int z1 = min(z0 + zc - 1, Ly.zl);
    const float* __restrict__ mi = static_cast<const float*>(a.mu_in);
    float* __restrict__ mo = static_cast<float*>(a.mu_out);
    const float* __restrict__ alpha = static_cast<const float*>(a.alpha);
    const Mom4<float>* __restrict__ hist = static_cast<const Mom4<float>*>(a.hist);
    const Mom4<float>* __restrict__ hist2 = static_cast<const Mom4<float>*>(a.hist2);
    const float omega = static_cast<float>(a.omega), tgx = static_cast<float>(a.tau * a.g[0]),
                tgy = static_cast<float>(a.tau * a.g[1]), tgz = static_cast<float>(a.tau * a.g[2]);
    // byte offsets within a plane fit 32 bits (the host checks plane bytes)
    const uint32_t py = static_cast<uint32_t>(Ly.px) * 4u, pz = static_cast<uint32_t>(Ly.pxy) * 4u;
    const uint32_t off = static_cast<uint32_t>(Ly.off) * 4u;

    // patch cells as in k_wall2: the tile cells, then the ring
    int pi[TB_PASS], pj[TB_PASS], gx[TB_PASS], gy[TB_PASS];
    bool live[TB_PASS];
#pragma unroll
    for (int k = 0; k < TB_PASS; ++k) {
        bool in = true;
        if (k < TB_OUT) {
            const int c = k * 256 + tid;
            pi[k] = c % TB_TX;
            pj[k] = c / TB_TX;
        } else if (tid < TB_PX) {
            pi[k] = tid - 1;
            pj[k] = -1;
        } else if (tid < 2 * TB_PX) {
            pi[k] = tid - TB_PX - 1;
            pj[k] = TB_TY;
        } else if (tid < 2 * TB_PX + TB_TY) {
            pi[k] = -1;
            pj[k] = tid - 2 * TB_PX;
        } else {
            pi[k] = TB_TX;
            pj[k] = tid - 2 * TB_PX - TB_TY;
            in = tid < TB_NP - TB_CELLS;
        }
        const int ux = x0 + pi[k], uy = y0 + pj[k];
        live[k] = in && ux <= Ly.xl + 1 && uy <= Ly.yl + 1;
        gx[k] = wrap1(ux, Ly.xl);
        gy[k] = wrap1(uy, Ly.yl);
    }
    auto send = [&](auto qc, int k, float v) {
        constexpr int q = decltype(qc)::value;
        const int di = pi[k] - L::cx(q), dj = pj[k] - L::cy(q);
        if (di >= 0 && di < TB_TX && dj >= 0 && dj < TB_TY) lds[S::template slot<q>()][dj * TB_TX + di] = v;
    };

    float hold[TB_PASS][Q];
    float prev[TB_PASS][Q] = {};  // cz = -1 values of the previous plane
    float da[TB_OUT] = {}, dap[TB_OUT] = {};
    for (int zs = z0 - 1; zs <= z1 + 1; ++zs) {
        // (the empty asm keeps the Q plane bases from being hoisted, as in k_bulk2)
        int64_t plane = Ly.plane;
        asm volatile("" : "+s"(plane));
        // step t on plane zs
        const int gz = wrap1(zs, Ly.zl);
        const uint32_t zs3[3] = {off + pz * wrap1(gz - 1, Ly.zl), off + pz * gz, off + pz * wrap1(gz + 1, Ly.zl)};
#pragma unroll
        for (int k = 0; k < TB_PASS; ++k) {
            if (!live[k]) continue;
            const uint32_t xs[3] = {4u * wrap1(gx[k] - 1, Ly.xl), 4u * gx[k], 4u * wrap1(gx[k] + 1, Ly.xl)};
            const uint32_t ys[3] = {py * wrap1(gy[k] - 1, Ly.yl), py * gy[k], py * wrap1(gy[k] + 1, Ly.yl)};
            float lam[Q], mu[Q];
            static_for<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                lam[q] = tb_at(mi + q * plane, zs3[1 + L::cz(q)] + ys[1 + L::cy(q)] + xs[1 + L::cx(q)]);
            });
            const Mom4<float> m = hist[cell_index(Ly, gx[k], gy[k], gz)];  // (ring cells again by other blocks)
            float al = 0.0f;
            if constexpr (BRINK) al = tb_at(alpha, zs3[1] + ys[1] + xs[1]);
            const float d = adjoint_relax<L, float, BRINK>(m.v[0], m.v[1], m.v[2], m.v[3], lam, mu, omega, al, tgx, tgy,
                                                          tgz);
            if (k < TB_OUT) da[k & (TB_OUT - 1)] = d;
            static_for<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if constexpr (L::cz(q) > 0)
                    send(qc, k, mu[q]);
                else
                    hold[k][q] = mu[q];
            });
        }
        __syncthreads();
        // step t - 1 on plane zs - 1
        const int zo = zs - 1;
        if (zo >= z0) {
#pragma unroll
            for (int k = 0; k < TB_OUT; ++k) {
                const int c = k * 256 + tid;
                const int ox = x0 + pi[k], oy = y0 + pj[k];
                if (ox <= Ly.xl && oy <= Ly.yl) {
                    float lam[Q], mu[Q];
                    static_for<0, Q>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        lam[q] = lds[S::template slot<q>()][c];
                    });
                    const uint32_t eb = 4u * (static_cast<uint32_t>(Ly.off) + ox) + pz * zo + py * oy;
                    const Mom4Raw<float> mr =
                        __builtin_nontemporal_load(reinterpret_cast<const Mom4Raw<float>*>(hist2) + cell_index(Ly, ox, oy, zo));
                    const Mom4<float> m = {{mr[0], mr[1], mr[2], mr[3]}};
                    float al = 0.0f;
                    if constexpr (BRINK) al = tb_at(alpha, eb);
                    const float d = adjoint_relax<L, float, BRINK>(m.v[0], m.v[1], m.v[2], m.v[3], lam, mu, omega, al,
                                                                  tgx, tgy, tgz);
                    static_for<0, Q>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        put<CACHED ? Put::Through : Put::Stream>(tb_ptr(mo + q * plane, eb), mu[q]);
                    });
                    if constexpr (BRINK) {
                        double* g = a.grad_alpha + eb / 4u;
                        *g = (*g + static_cast<double>(dap[k])) + static_cast<double>(d);
                    }
                }
            }
        }
        __syncthreads();
        // sends read by step t - 1 of the next iteration: cz = 0 of this
        // plane, cz = -1 of the previous plane
#pragma unroll
        for (int k = 0; k < TB_PASS; ++k) {
            if (k < TB_OUT) dap[k & (TB_OUT - 1)] = da[k & (TB_OUT - 1)];
            if (!live[k]) continue;
            static_for<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if constexpr (L::cz(q) <= 0) send(qc, k, L::cz(q) == 0 ? hold[k][q] : prev[k][q]);
                if constexpr (L::cz(q) < 0) prev[k][q] = hold[k][q];
            });
        }
    }
}

}  // namespace lbm_amd
