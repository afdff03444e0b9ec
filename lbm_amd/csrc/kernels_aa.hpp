// In-place time step (AA pattern): one distribution buffer M instead of two.
//
// The post-collision state is held in one of two representations:
//   E (natural): g_q(x) in M[q][x]
//   O (swapped): g_q(x) in M[qbar][x + c_q]   (already streamed, opposite slot)
// and steps alternate between them:
//   E -> O (k_aa_eo): h_q(x) = M[q][x - c_q]; collide; g'_k -> M[kbar][x + c_k].
//   O -> E (k_aa_oe): h_q(x) = M[qbar][x];     collide; g'_k -> M[k][x].
// A cell reads and writes the same set of locations in either step, and no
// two cells share a location, so the update is in place.
//
// Boundary links. The value a fluid cell x pulls over a link q whose source
// b = x - c_q is not fluid is the boundary rule evaluated on x's own
// post-collision values of the previous step (as in the two-buffer kernels).
// Each step therefore leaves the rule value in the slot the next step reads:
//   after E -> O, in M[k][x] for every k with x + c_k not fluid (the link
//     kbar of x), which O -> E reads as h_kbar(x) = M[k][x];
//   after O -> E, in M[q][b] for every link q of x with a non-fluid source b,
//     which E -> O reads as h_q(x) = M[q][x - c_q].
// E -> O also stores g'_k into the boundary cell's slot M[kbar][x + c_k], so
// the O representation is complete for every fluid cell; the first step after
// set-up reads the boundary cells' stored values, as the two-buffer kernels do.
//
// k_aa_swap turns O into E without a collision, for the readers (moments,
// sums, field export): it swaps each pair M[q][x] <-> M[qbar][x + c_q]. For a
// link to a boundary cell this also leaves the rule value stored in E -> O in
// the boundary cell's slot, where the next E -> O step reads it.
//
// FreeSlip reads other fluid cells' values and has no in-place form here; the
// host rejects it for this layout.
#pragma once

#include "kernels.hpp"

namespace lbm_amd {

// Element of the neighbour x + sgn c_q (wrapped along periodic axes).
template <class L, int q, class I>
__device__ __forceinline__ I aa_nb(const FieldLayout& Ly, bool wraps, I e, int x, int y, int z, int sgn) {
    if (!wraps) return e + static_cast<I>(sgn * (L::cx(q) + L::cy(q) * Ly.px + L::cz(q) * Ly.pxy));
    return static_cast<I>(Ly.off) + static_cast<I>(wrap_if(x + sgn * L::cx(q), Ly.xl, Ly.per[0])) +
           static_cast<I>(Ly.px) * static_cast<I>(wrap_if(y + sgn * L::cy(q), Ly.yl, Ly.per[1])) +
           static_cast<I>(Ly.pxy) * static_cast<I>(wrap_if(z + sgn * L::cz(q), Ly.zl, Ly.per[2]));
}

__device__ __forceinline__ bool aa_wraps(const FieldLayout& Ly, int x, int y, int z) {
    return (Ly.per[0] && (x == 1 || x == Ly.xl)) || (Ly.per[1] && (y == 1 || y == Ly.yl)) ||
           (Ly.per[2] && (z == 1 || z == Ly.zl));
}

// Cell (x, y, z) of this lane in the k_cells tiling; false past the domain.
__device__ __forceinline__ bool aa_tile_cell(const FieldLayout& Ly, int tpp, double rxl, int rev, int& x, int& y, int& z) {
    const int64_t w = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    z = 1 + static_cast<int>(w / tpp);
    if (z > Ly.zl) return false;
    if (rev) z = Ly.zl + 1 - z;
    const int64_t c = (w % tpp) * 64 + (threadIdx.x & 63);
    const int64_t xl = Ly.xl;
    if (c >= xl * Ly.yl) return false;
    int64_t yy = static_cast<int64_t>(static_cast<double>(c) * rxl);
    int64_t xx = c - yy * xl;
    if (xx < 0) {
        --yy;
        xx += xl;
    } else if (xx >= xl) {
        ++yy;
        xx -= xl;
    }
    x = 1 + static_cast<int>(xx);
    y = 1 + static_cast<int>(yy);
    return true;
}

template <class L, Mode M>
__device__ __forceinline__ void aa_collide(const StepArgs& a, int64_t e, typename Io<M, L>::Calc (&f)[L::Q]) {
    using Calc = typename Io<M, L>::Calc;
    if constexpr (M == Mode::EXACT64) {
        collide_exact<L>(f, a.tau, a.omega);
    } else if (a.alpha) {
        const Calc alpha = static_cast<const Calc*>(a.alpha)[e];
        collide_shifted<L, Calc, true, kRcp<M>, Io<M, L>::SX>(f, static_cast<Calc>(a.omega), alpha,
                                                              static_cast<Calc>(a.tau * a.g[0]),
                                                static_cast<Calc>(a.tau * a.g[1]), static_cast<Calc>(a.tau * a.g[2]));
    } else {
        collide_shifted<L, Calc, false, kRcp<M>, Io<M, L>::SX>(f, static_cast<Calc>(a.omega), Calc(0), Calc(0), Calc(0),
                                                               Calc(0));
    }
}

// x's post-collision values (f: the collision's scaled representation) as
// they would be stored (rounded to the storage format), which is what the
// two-buffer kernels' rules read back.
template <class L, Mode M>
__device__ __forceinline__ void aa_own(const typename Io<M, L>::Calc (&f)[L::Q], typename Io<M, L>::Calc (&own)[L::Q]) {
    using IO = Io<M, L>;
    static_for<0, L::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        own[q] = IO::template to_calc<q>(IO::template store<q>(f[q]));
    });
}

// Element of the cell's neighbours and accesses relative to it, in either
// tiling: Nb::at<q, S>() is M[q][x + S c_q], Nb::elem<q, S>() its element.
template <class L, class T, bool B32>
struct AaPlane {
    T* m;
    const FieldLayout& Ly;
    int x, y, z;
    bool wraps;
    typename ElemIdx<B32>::type e;
    __device__ __forceinline__ AaPlane(T* m_, const FieldLayout& L_, int x_, int y_, int z_)
        : m(m_), Ly(L_), x(x_), y(y_), z(z_), wraps(aa_wraps(L_, x_, y_, z_)),
          e(static_cast<typename ElemIdx<B32>::type>(cell_elem(L_, x_, y_, z_))) {}
    template <int q, int S>
    __device__ __forceinline__ auto elem() const {
        return S == 0 ? e : aa_nb<L, q>(Ly, wraps, e, x, y, z, S);
    }
    // M[p][x + S c_q]
    template <int p, int q, int S>
    __device__ __forceinline__ Glob<T>& at() const {
        return plane_ref<B32>(m, p, Ly.plane, elem<q, S>());
    }
};
template <class L, class T>
struct AaRow {
    T* m;
    const FieldLayout& Ly;
    RowNb<T> nb;
    uint32_t e;
    __device__ __forceinline__ AaRow(T* m_, const FieldLayout& L_, int x, int y, int z)
        : m(m_), Ly(L_), nb(L_, x, y, z), e(elem_at<true>(L_, x, y, z)) {}
    template <int q, int S>
    __device__ __forceinline__ uint32_t elem() const {
        return nb.template offset<L, q, S>() / static_cast<uint32_t>(sizeof(T));
    }
    template <int p, int q, int S>
    __device__ __forceinline__ Glob<T>& at() const {
        return nb.template at<L, q, S>(m + (p - q) * Ly.plane, Ly.plane);
    }
};

template <class L, Mode M, class Nb>
__device__ __forceinline__ void aa_eo_cell(const StepArgs& a, const Nb& nb) {
    using IO = Io<M, L>;
    using Calc = typename IO::Calc;
    constexpr int Q = L::Q;
    const uint8_t k = kind_at(a.kind, nb.e);
    if (k >= KIND_COND0) return;
    Calc f[Q];
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        f[q] = IO::template load<q>(nb.template at<q, q, -1>());
    });
    aa_collide<L, M>(a, static_cast<int64_t>(nb.e), f);
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        nb.template at<Q - 1 - q, q, 1>() = IO::template store<q>(f[q]);
    });
    if (k == KIND_NEAR) {
        Calc own[Q];
        aa_own<L, M>(f, own);
        const OwnSums<Calc> os = own_sums<L, Calc>(own);
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            constexpr int j = Q - 1 - q;  // the link of x whose source is x + c_q
            const uint8_t kb = kind_at(a.kind, nb.template elem<q, 1>());
            if (kb >= KIND_COND0 && kb < KIND_INERT)
                nb.template at<q, q, 0>() =
                    IO::template from_calc<j>(rule_value<L, M, j>(cond_at(a.conds, kb - KIND_COND0), os, own[q]));
        });
    }
}

template <class L, Mode M, class Nb>
__device__ __forceinline__ void aa_oe_cell(const StepArgs& a, const Nb& nb) {
    using IO = Io<M, L>;
    using Calc = typename IO::Calc;
    constexpr int Q = L::Q;
    const uint8_t k = kind_at(a.kind, nb.e);
    if (k >= KIND_COND0) return;
    Calc f[Q];
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        f[q] = IO::template load<q>(nb.template at<Q - 1 - q, q, 0>());
    });
    aa_collide<L, M>(a, static_cast<int64_t>(nb.e), f);
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        nb.template at<q, q, 0>() = IO::template store<q>(f[q]);
    });
    if (k == KIND_NEAR) {
        Calc own[Q];
        aa_own<L, M>(f, own);
        const OwnSums<Calc> os = own_sums<L, Calc>(own);
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const uint8_t kb = kind_at(a.kind, nb.template elem<q, -1>());
            if (kb >= KIND_COND0 && kb < KIND_INERT)
                nb.template at<q, q, -1>() =
                    IO::template from_calc<q>(rule_value<L, M, q>(cond_at(a.conds, kb - KIND_COND0), os, own[Q - 1 - q]));
        });
    }
}

// Row tiles (tpr > 0, planes under 4 GiB) or the plane tiling of k_cells. The
// element arithmetic of 2 Q neighbours per lane weighs on 16-bit storage, and
// a wavefront that spans rows touches lines twice. Plane / row tiles, us per
// step of a periodic D3Q19 box: fp32 64^3 8.98 / 6.97, 100^3 31.2 / 25.9, 150^3
// 112 / 93.5, 256^3 495 / 491; fp16 200x150x170 80 / 71.5, 192^3 131 / 109.
// Plain stores: streaming ones measured 18 % slower at 100^3 and equal
// elsewhere, write-through ones 1 to 12 % slower.
template <class L, Mode M, bool B32, bool ROW>
__global__ void __launch_bounds__(256) k_aa_eo(StepArgs a, int tpp, double rxl, int tpr) {
    using T = typename Io<M, L>::T;
    int x, y, z;
    if constexpr (ROW) {
        if (row_tile_cell(a.L, tpr, a.rev, x, y, z)) aa_eo_cell<L, M>(a, AaRow<L, T>(static_cast<T*>(a.dst), a.L, x, y, z));
    } else {
        if (aa_tile_cell(a.L, tpp, rxl, a.rev, x, y, z))
            aa_eo_cell<L, M>(a, AaPlane<L, T, B32>(static_cast<T*>(a.dst), a.L, x, y, z));
    }
}

template <class L, Mode M, bool B32, bool ROW>
__global__ void __launch_bounds__(256) k_aa_oe(StepArgs a, int tpp, double rxl, int tpr) {
    using T = typename Io<M, L>::T;
    int x, y, z;
    if constexpr (ROW) {
        if (row_tile_cell(a.L, tpr, a.rev, x, y, z)) aa_oe_cell<L, M>(a, AaRow<L, T>(static_cast<T*>(a.dst), a.L, x, y, z));
    } else {
        if (aa_tile_cell(a.L, tpp, rxl, a.rev, x, y, z))
            aa_oe_cell<L, M>(a, AaPlane<L, T, B32>(static_cast<T*>(a.dst), a.L, x, y, z));
    }
}

// O -> E without a collision: swap M[q][x] <-> M[qbar][x + c_q]. A fluid cell
// takes the pairs of its first Q/2 directions, and those of the others whose
// partner cell is not fluid (that partner takes no pairs).
template <class L, Mode M, bool B32>
__global__ void __launch_bounds__(256) k_aa_swap(StepArgs a, int tpp, double rxl) {
    using T = typename Io<M, L>::T;
    constexpr int Q = L::Q;
    const FieldLayout& Ly = a.L;
    int x, y, z;
    if (!aa_tile_cell(Ly, tpp, rxl, a.rev, x, y, z)) return;
    using I = typename ElemIdx<B32>::type;
    const I e = static_cast<I>(cell_elem(Ly, x, y, z));
    if (kind_at(a.kind, e) >= KIND_COND0) return;
    T* __restrict__ m = static_cast<T*>(a.dst);
    const bool wraps = aa_wraps(Ly, x, y, z);
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (q != L::rest) {
            const I pe = aa_nb<L, q>(Ly, wraps, e, x, y, z, 1);
            if (q < Q / 2 || kind_at(a.kind, pe) >= KIND_COND0) {
                Glob<T>* p0 = &plane_ref<B32>(m, q, Ly.plane, e);
                Glob<T>* p1 = &plane_ref<B32>(m, Q - 1 - q, Ly.plane, pe);
                const T v0 = *p0;
                *p0 = *p1;
                *p1 = v0;
            }
        }
    });
}

}  // namespace lbm_amd
