// Batched adjoint kernels (D3Q19; F32 and F64S storage).
#include "batch_adjoint.hpp"
#include "kernels_adjoint.hpp"

namespace lbm_amd {

namespace {

// Cell (x, y, z) of lane `lane` in cell tile `local` of a domain; false past
// the plane's last cell. The row is a double estimate of c / xl (off by at
// most one) corrected in integers.
__device__ __forceinline__ bool tile_cell(const BatchAdjView& v, int local, int lane, int& x, int& y, int& z) {
    z = 1 + local / v.tpp;
    const int c = (local % v.tpp) * 64 + lane;
    const int xl = v.L.xl;
    if (c >= xl * v.L.yl) return false;
    int yy = static_cast<int>(static_cast<double>(c) * v.rxl);
    int xx = c - yy * xl;
    if (xx < 0) {
        --yy;
        xx += xl;
    } else if (xx >= xl) {
        ++yy;
        xx -= xl;
    }
    x = 1 + xx;
    y = 1 + yy;
    return true;
}

// Slot i of a domain's chunk. The address is the same for the whole
// wavefront; readfirstlane keeps it (and every address derived from it) in
// scalar registers instead of a 64-bit product per lane.
template <class T>
__device__ __forceinline__ T* slot(const BatchAdjView& v, int i) {
    const uint64_t p = reinterpret_cast<uint64_t>(static_cast<T*>(v.chunk) + i * v.slot_elems);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(p & 0xffffffffu)));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(p >> 32)));
    return reinterpret_cast<T*>((static_cast<uint64_t>(hi) << 32) | lo);
}

// One forward step of every domain from slot src_slot to slot dst_slot.
template <class L, Mode M, bool B32>
__global__ void __launch_bounds__(256) k_badj_recompute(BatchAdjArgs b) {
    using T = typename StorageOf<M>::T;
    const int lane = threadIdx.x & 63;
    const TileWalk w = tile_walk(b.ntiles, b.nxcd);
    for (int t = w.t; t < w.end; t += w.stride) {
        const TileRef tr = b.tiles[t];
        const BatchAdjView& v = b.views[tr.dom];
        int x, y, z;
        if (!tile_cell(v, tr.local, lane, x, y, z)) continue;
        StepArgs a{};
        a.L = v.L;
        a.src = slot<T>(v, b.src_slot);
        a.dst = slot<T>(v, b.dst_slot);
        a.kind = v.kind;
        a.lmask = v.lmask;
        a.lcond = v.lcond;
        a.rword = v.rword;
        a.span32 = v.span32;
        a.cached = b.cached;
        a.conds = v.conds;
        a.materialised = b.materialised;
        a.tau = v.tau;
        a.omega = v.omega;
        any_cell<L, M, false, B32>(a, x, y, z);  // the adjoint takes no FreeSlip condition
    }
}

// One adjoint step of every domain: g^{t-1} in gprev_slot, mu^{t+1} in
// mu_in_slot, mu^t into mu_out_slot; kinetic-energy objective.
template <class L, Mode M, bool B32>
__global__ void __launch_bounds__(256) k_badj_backward(BatchAdjArgs b) {
    using T = typename StorageOf<M>::T;
    static_assert(sizeof(T) == sizeof(typename StorageOf<M>::Calc), "mu slots hold the arithmetic type");
    const int lane = threadIdx.x & 63;
    const TileWalk w = tile_walk(b.ntiles, b.nxcd);
    for (int t = w.t; t < w.end; t += w.stride) {
        const TileRef tr = b.tiles[t];
        const BatchAdjView& v = b.views[tr.dom];
        int x, y, z;
        if (!tile_cell(v, tr.local, lane, x, y, z)) continue;
        const auto e = elem_at<B32>(v.L, x, y, z);
        const uint8_t k = kind_at(v.kind, e);
        if (k >= KIND_COND0) continue;
        AdjArgs a{};
        a.L = v.L;
        a.gprev = slot<T>(v, b.gprev_slot);
        a.gcur = v.gfinal;
        a.mu_in = slot<T>(v, b.mu_in_slot);
        a.mu_out = slot<T>(v, b.mu_out_slot);
        a.kind = v.kind;
        a.conds = v.conds;
        a.materialised = b.materialised;
        a.terminal = b.terminal;
        a.tau = v.tau;
        a.omega = v.omega;
        a.objective = OBJ_KINETIC;
        const bool near = k == KIND_NEAR;
        adj_any_cell<L, M, false, B32>(a, x, y, z, e, near, v.gw + (near ? 3 * static_cast<int64_t>(v.near_idx[e]) : 0));
    }
}

// Step hist_step's record of a domain (wavefront-uniform, as slot).
template <class Calc>
__device__ __forceinline__ Calc* record(const BatchAdjView& v, int64_t step) {
    const uint64_t p = reinterpret_cast<uint64_t>(static_cast<Calc*>(v.hist) + (step - 1) * v.hist_stride);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(p & 0xffffffffu)));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(p >> 32)));
    return reinterpret_cast<Calc*>((static_cast<uint64_t>(hi) << 32) | lo);
}
__device__ __forceinline__ int64_t record_near(const BatchAdjView& v) {
    return 4 * static_cast<int64_t>(v.L.xl) * v.L.yl * v.L.zl;
}

// One forward step of every domain, recording.
template <class L, Mode M, bool B32, bool CACHED>
__global__ void __launch_bounds__(256) k_badj_hist_forward(BatchAdjArgs b) {
    using Calc = typename StorageOf<M>::Calc;
    const int lane = threadIdx.x & 63;
    const TileWalk w = tile_walk(b.ntiles, b.nxcd);
    for (int t = w.t; t < w.end; t += w.stride) {
        const TileRef tr = b.tiles[b.rev ? b.ntiles - 1 - t : t];
        const BatchAdjView& v = b.views[tr.dom];
        int x, y, z;
        if (!tile_cell(v, tr.local, lane, x, y, z)) continue;
        StepArgs a{};
        a.L = v.L;
        a.src = v.buf[b.parity];
        a.dst = v.buf[b.parity ^ 1];
        a.kind = v.kind;
        a.lmask = v.lmask;
        a.lcond = v.lcond;
        a.rword = v.rword;
        a.span32 = v.span32;
        a.cached = b.cached;
        a.conds = v.conds;
        a.materialised = b.materialised;
        a.tau = v.tau;
        a.omega = v.omega;
        Calc* r = record<Calc>(v, b.hist_step);
        a.hist = r;
        a.rho_own = r + record_near(v);
        a.near_idx = v.near_idx;
        if (!any_cell<L, M, false, B32, CACHED, true>(a, x, y, z)) b.status[tr.dom] = 1;
    }
}

// One adjoint step of every domain from the record of step hist_step: mu in
// mu_in_slot to mu_out_slot; kinetic-energy objective.
template <class L, Mode M, bool B32>
__global__ void __launch_bounds__(256) k_badj_hist_backward(BatchAdjArgs b) {
    using T = typename StorageOf<M>::T;
    using Calc = typename StorageOf<M>::Calc;
    const int lane = threadIdx.x & 63;
    const TileWalk w = tile_walk(b.ntiles, b.nxcd);
    for (int t = w.t; t < w.end; t += w.stride) {
        const TileRef tr = b.tiles[b.rev ? b.ntiles - 1 - t : t];
        const BatchAdjView& v = b.views[tr.dom];
        int x, y, z;
        if (!tile_cell(v, tr.local, lane, x, y, z)) continue;
        const auto e = elem_at<B32>(v.L, x, y, z);
        const uint8_t k = kind_at(v.kind, e);
        if (k >= KIND_COND0) continue;
        AdjArgs a{};
        a.L = v.L;
        a.gcur = v.gfinal;
        a.mu_in = slot<T>(v, b.mu_in_slot);
        a.mu_out = slot<T>(v, b.mu_out_slot);
        a.kind = v.kind;
        a.conds = v.conds;
        a.materialised = b.materialised;
        a.terminal = b.terminal;
        a.tau = v.tau;
        a.omega = v.omega;
        a.objective = OBJ_KINETIC;
        const Calc* r = record<Calc>(v, b.hist_step);
        a.hist = r;
        a.cached = b.cached;
        adj_hist_cell<L, M, B32>(a, v.lmask, v.rword, x, y, z, e, k == KIND_NEAR, r + record_near(v), v.near_idx, v.gw);
    }
}

// near_idx[element of NEAR cell i] = i
__global__ void __launch_bounds__(256) k_badj_near_index(FieldLayout Ly, const CellCoord* blist, int64_t nb, int* near_idx) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= nb) return;
    const CellCoord c = blist[i];
    near_idx[cell_elem(Ly, c.x, c.y, c.z)] = static_cast<int>(i);
}

// Per-domain sums of the gradient accumulators: block d sums domain d's NEAR
// cells with a fixed assignment and a fixed tree, so the result does not
// depend on scheduling.
__global__ void __launch_bounds__(256) k_badj_reduce(const BatchAdjView* views, double* out) {
    const BatchAdjView& v = views[blockIdx.x];
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    for (int64_t i = threadIdx.x; i < v.nb; i += blockDim.x) {
        const double* g = v.gw + 3 * i;
        s0 += g[0];
        s1 += g[1];
        s2 += g[2];
    }
    __shared__ double sh[3][256];
    sh[0][threadIdx.x] = s0;
    sh[1][threadIdx.x] = s1;
    sh[2][threadIdx.x] = s2;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (static_cast<int>(threadIdx.x) < w)
            for (int k = 0; k < 3; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 3) out[3 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0];
}

template <class L, Mode M>
struct BatchAdjImpl {
    static hipError_t recompute(const BatchAdjArgs& a, int grid, hipStream_t s) {
        if (a.idx32)
            hipLaunchKernelGGL((k_badj_recompute<L, M, true>), dim3(grid), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((k_badj_recompute<L, M, false>), dim3(grid), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    static hipError_t backward(const BatchAdjArgs& a, int grid, hipStream_t s) {
        if (a.idx32)
            hipLaunchKernelGGL((k_badj_backward<L, M, true>), dim3(grid), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((k_badj_backward<L, M, false>), dim3(grid), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    static hipError_t hist_forward(const BatchAdjArgs& a, int grid, hipStream_t s) {
        if (a.idx32 && a.cached)
            hipLaunchKernelGGL((k_badj_hist_forward<L, M, true, true>), dim3(grid), dim3(256), 0, s, a);
        else if (a.idx32)
            hipLaunchKernelGGL((k_badj_hist_forward<L, M, true, false>), dim3(grid), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((k_badj_hist_forward<L, M, false, false>), dim3(grid), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    static hipError_t hist_backward(const BatchAdjArgs& a, int grid, hipStream_t s) {
        if (a.idx32)
            hipLaunchKernelGGL((k_badj_hist_backward<L, M, true>), dim3(grid), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((k_badj_hist_backward<L, M, false>), dim3(grid), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    static hipError_t near_index(const FieldLayout& Ly, const CellCoord* blist, int64_t nb, int* near_idx, hipStream_t s) {
        if (nb > 0)
            hipLaunchKernelGGL(k_badj_near_index, dim3(static_cast<uint32_t>((nb + 255) / 256)), dim3(256), 0, s, Ly,
                               blist, nb, near_idx);
        return hipGetLastError();
    }
    static hipError_t reduce(const BatchAdjView* views, int ndom, double* out, hipStream_t s) {
        hipLaunchKernelGGL(k_badj_reduce, dim3(ndom), dim3(256), 0, s, views, out);
        return hipGetLastError();
    }
    static BatchAdjOps make() {
        BatchAdjOps o{};
        o.recompute = &recompute;
        o.backward = &backward;
        o.hist_forward = &hist_forward;
        o.hist_backward = &hist_backward;
        o.near_index = &near_index;
        o.reduce = &reduce;
        return o;
    }
};

const BatchAdjOps kF32 = BatchAdjImpl<D3Q19, Mode::F32>::make();
const BatchAdjOps kF64S = BatchAdjImpl<D3Q19, Mode::F64S>::make();

}  // namespace

const BatchAdjOps* batch_adj_ops(int q, Mode m) {
    if (q != 19) return nullptr;
    if (m == Mode::F32) return &kF32;
    if (m == Mode::F64S) return &kF64S;
    return nullptr;
}

}  // namespace lbm_amd
