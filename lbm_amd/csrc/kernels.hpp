// Fused pull-stream + collide kernels and the per-field kernels of one mode.
//
// One time step of the reference (src/main.cpp:50-52: stream, swap, collide)
// is one pass here: every interior fluid cell x pulls f_q from x - c_q in the
// source buffer (post-collision values of the previous step), collides in
// registers and writes its Q values to the destination buffer.
//
// The reference's second collide pass (boundary rules on non-fluid cells,
// include/domain.hpp:157-165) writes into a non-fluid cell b exactly those
// directions q for which b + c_q is an interior fluid cell, and the only
// reader of that value is the pull of that fluid cell in the next step. So a
// fluid cell x that pulls direction q from a non-fluid b = x - c_q evaluates
// b's rule for (b, q) itself, from its own post-collision values (all rules
// read only the neighbour b + c_q = x, except FreeSlip, which reads fluid
// cells next to b). Right after initialisation or after the host wrote the
// field, non-fluid cells hold values that the next pull reads as stored
// (the first step of the reference pulls the initial weights from every
// boundary cell); the `materialised` flag selects that.
//
// Two kernels per step:
//   k_bulk - every interior cell of kind BULK (all Q sources fluid), V cells
//            per thread along x, one plane-contiguous load per direction.
//   k_near - the listed cells of kind NEAR (fluid with a non-fluid source),
//            one thread per cell, evaluates boundary rules.
#pragma once

#include <type_traits>

#include "collide.hpp"
#include "domain_view.hpp"
#include "lbm_hip/lattice.hpp"
#include "storage.hpp"

namespace lbm_amd {

template <class T, int V>
struct alignas(sizeof(T) * V) VecT {
    T v[V];
};

// Pulled values, converted by here. bf16's conversion is one shift, which the
// compiler otherwise moves to the uses behind the branches that follow, and
// then holds raw and converted values at once: k_cell_rows D3Q19 spilled 32 of
// its 80 registers, D3Q27 took 136 (3 waves per SIMD), k_bulk D3Q27 172 (2).
// With this and through_storage's they take 80 (no spills), 110 and 133. us a
// step, without / with: D3Q19 64^3 sphere channel 19.3 / 13.8, 160x150x140
// 122 / 92, walls across z 28x60x50 11.4 / 9.4, D3Q27 periodic 192x160x128
// singly 126 / 101 (but D3Q27 channels of 32^3 12.4 / 13.5).
// (An empty asm at each load made the loads wait for one another: the walled
// two-step pass took 1.4 times as long.)
template <Mode M, int Q, class Calc>
__device__ __forceinline__ void converted(Calc (&f)[Q]) {
    if constexpr (M == Mode::BF16) {
#pragma unroll
        for (int q = 0; q < Q; ++q) __asm__("" : "+v"(f[q]));
    }
}

// drho and u of one cell and step (StepArgs::hist).
template <class Calc>
struct alignas(16) Mom4 {
    Calc v[4];
};
template <class Calc>
using Mom4Raw = Calc __attribute__((ext_vector_type(4)));  // the same as one memory access

// How a step's output is stored.
//   Stream: non-temporal. On a field beyond the caches every value is read
//     long after it would have been evicted, so keeping it only displaces
//     source lines (256^3 fp32 box 0.456 against 0.470 ms a single step).
//   Where both buffers fit the 256 MiB memory-side cache (StepArgs::cached)
//   streamed values would leave it and the next step fetch them from HBM:
//   Keep: plain (cell tiles, whose wavefronts write parts of lines);
//   Through: agent scope, written on at once, so that the launch does not end
//     with the L2s' dirty lines (row kernels and passes, whose wavefronts
//     write whole lines).
// Measured, us a step, Stream / Keep / Through, buffers together: passes over
// periodic D3Q19 boxes fp32 80^3 (98 MB) 19.3 / 16.2 / 15.4, 104^3 (218 MB)
// 32.0 / 23.5 / 22.4, 112^3 (252 MB) 37.9 / 29.4 / 29.7, 120^3 (289 MB) 42.1 /
// 38.4 / 38.4, fp16 150^3 (337 MB) 51.8 / 52.6 / 52.0; cell tiles on cavities
// fp32 48^3 (19 MB) 12.1 / 12.7 / 12.8, 64^3 (63 MB) 16.5 / 15.5 / 15.1, 104^3
// 53.5 / 40.6 / 40.9, fp16 96^3 (71 MB) 30.5 / 24.7 / 26.6, fp64 64^3 (105 MB)
// 24.7 / 20.9 / 20.5; 30 batched cavities (340 MB) 90 / 105 / 111.
enum class Put { Stream, Keep, Through };

template <int BYTES>
struct RawOf;
template <>
struct RawOf<1> { using type = uint8_t; };
template <>
struct RawOf<2> { using type = uint16_t; };
template <>
struct RawOf<4> { using type = uint32_t; };
template <>
struct RawOf<8> { using type = uint32_t __attribute__((ext_vector_type(2))); };
template <>
struct RawOf<16> { using type = uint32_t __attribute__((ext_vector_type(4))); };
template <>
struct RawOf<32> { using type = uint32_t __attribute__((ext_vector_type(8))); };

template <Put P, class T, class Ptr>
__device__ __forceinline__ void put(Ptr p, const T& v) {
    using R = typename RawOf<sizeof(T)>::type;
    if constexpr (P == Put::Stream) {
        R r;
        __builtin_memcpy(&r, &v, sizeof(R));
        if constexpr (std::is_same<Ptr, T*>::value)
            __builtin_nontemporal_store(r, reinterpret_cast<R*>(p));
        else
            __builtin_nontemporal_store(r, reinterpret_cast<__attribute__((address_space(1))) R*>(p));
    } else if constexpr (P == Put::Through && sizeof(T) <= 8) {
        using U = std::conditional_t<sizeof(T) == 8, uint64_t, std::conditional_t<sizeof(T) == 4, uint32_t, uint16_t>>;
        U u;
        __builtin_memcpy(&u, &v, sizeof(U));
        __hip_atomic_store((__attribute__((address_space(1))) U*)p, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *p = v;
    }
}

// body(policy) with the policy for a field that does or does not fit the
// caches. The empty asm keeps the compiler from merging the two branches'
// stores into one without the non-temporal hint.
template <Put Cached, class Body>
__device__ __forceinline__ void with_put(int cached, Body body) {
    if (cached) {
        asm volatile("");
        body(std::integral_constant<Put, Cached>{});
        asm volatile("");
    } else {
        body(std::integral_constant<Put, Put::Stream>{});
    }
}

// Element indices within a plane: 32-bit where a plane holds less than
// 4 GiB (B32), so that an access is a uniform direction-plane base plus one
// 32-bit byte offset per lane; 64-bit otherwise.
template <bool B32>
struct ElemIdx {
    using type = int64_t;
};
template <>
struct ElemIdx<true> {
    using type = uint32_t;
};

// Objects in the global address space. Every field, kind array and
// condition table lives in device (global) memory, but where a kernel reads
// their pointers from a table in memory (the batched kernels) the compiler
// cannot prove it and addresses them with flat instructions, which take no
// scalar base and wait on the LDS counter too. Accesses through Glob<T>
// references are global loads and stores in every kernel.
template <class T>
using Glob = __attribute__((address_space(1))) T;

template <class T>
__device__ __forceinline__ Glob<T>* glob(T* p) {
    return (Glob<T>*)p;
}

// Dual-number fields (the fp64 tangent run) keep generic references: a
// class with user-declared constructors is not copied out of an
// address-space-qualified object.
template <class T>
struct IsDual : std::false_type {};
template <class U>
struct IsDual<Dual<U>> : std::true_type {};
template <class T>
using PlaneElem = std::conditional_t<IsDual<std::remove_const_t<T>>::value, T, Glob<T>>;

// Element e of direction plane q of field m (global memory).
template <bool B32, class T, class I>
__device__ __forceinline__ PlaneElem<T>& plane_ref(T* m, int q, int64_t plane, I e) {
    using Byte = std::conditional_t<std::is_const_v<T>, const char, char>;
    using E = PlaneElem<T>;
    using EB = std::conditional_t<IsDual<std::remove_const_t<T>>::value, Byte, Glob<Byte>>;
    E* base = (E*)(m + q * plane);
    if constexpr (B32)
        return *reinterpret_cast<E*>(reinterpret_cast<EB*>(base) +
                                     static_cast<uint32_t>(e) * static_cast<uint32_t>(sizeof(T)));
    else
        return base[e];
}

// Cell kind at element e, and condition i of a domain's table.
template <class I>
__device__ __forceinline__ uint8_t kind_at(const uint8_t* kind, I e) {
    return glob(kind)[e];
}
using GCond = Glob<const Cond>;
__device__ __forceinline__ const GCond& cond_at(const Cond* conds, int i) { return glob(conds)[i]; }

// cell_elem in the index type of plane_ref. With B32 every element index of
// the field is below 2^32 and all terms are non-negative, so 32-bit
// arithmetic gives it exactly.
template <bool B32>
__device__ __forceinline__ typename ElemIdx<B32>::type elem_at(const FieldLayout& L, int x, int y, int z) {
    if constexpr (B32)
        return static_cast<uint32_t>(L.off) + static_cast<uint32_t>(x) +
               static_cast<uint32_t>(L.px) * static_cast<uint32_t>(y) +
               static_cast<uint32_t>(L.pxy) * static_cast<uint32_t>(z);
    else
        return cell_elem(L, x, y, z);
}

__device__ __forceinline__ int wrap1(int v, int l) { return v == 0 ? l : (v == l + 1 ? 1 : v); }

__device__ __forceinline__ int wrap_if(int v, int l, int per) {
    return per ? wrap1(v, l) : v;
}

// ---------------------------------------------------------------------------
// Bulk kernel. Block (BX, BY) threads covers BX*V cells of BY rows at one z.
// Grid is flattened: blockIdx.x = bx + nbx * (by + nby * (z - 1)).
//
// Source rows are wrapped unconditionally: along a periodic axis that is the
// periodic image, and along a walled axis any cell next to the wall pulls
// from a ghost cell, is NEAR and is masked out before its values are used.
// V cells (x0 .. x0+V-1, y, z) of one thread. Returns false when a cell it
// updated read a NaN or infinite value (finite_calc of the collision's base).
// POLICY false: output streamed whatever a.cached says (the batch's row tiles:
// both policies in one kernel took 325 for 268 us a step, 30 cavities).
template <class L, Mode M, int V, bool FLAGS, bool BRINK, bool HIST = false, bool POLICY = true>
__device__ __forceinline__ bool bulk_cells(const StepArgs& a, int x0, int y, int z,
                                           bool* near_lanes = nullptr) {
    using IO = Io<M, L>;
    using T = typename IO::T;
    using Calc = typename IO::Calc;
    constexpr int Q = L::Q;
    const FieldLayout& Ly = a.L;
    if (x0 > Ly.xl || y > Ly.yl) return true;

    const int64_t e0 = cell_elem(Ly, x0, y, z);
    bool act[V];
    bool any = false;
    if constexpr (FLAGS) {
        const VecT<uint8_t, V> kv = *reinterpret_cast<const VecT<uint8_t, V>*>(a.kind + e0);
#pragma unroll
        for (int i = 0; i < V; ++i) {
            act[i] = (kv.v[i] == KIND_BULK) && (x0 + i <= Ly.xl);
            any |= act[i];
            if (near_lanes) near_lanes[i] = (kv.v[i] == KIND_NEAR) && (x0 + i <= Ly.xl);
        }
    } else {
#pragma unroll
        for (int i = 0; i < V; ++i) {
            act[i] = (x0 + i <= Ly.xl);
            any |= act[i];
        }
    }
    const int ym = wrap1(y - 1, Ly.yl), yp = wrap1(y + 1, Ly.yl);
    const int zm = wrap1(z - 1, Ly.zl), zp = wrap1(z + 1, Ly.zl);
    const int xm = wrap1(x0 - 1, Ly.xl);  // source of lane 0 for cx = +1
    const int xpv = wrap1(x0 + V, Ly.xl); // source of lane V-1 for cx = -1
    const bool partial = (x0 + V - 1 > Ly.xl);

    const T* __restrict__ src = static_cast<const T*>(a.src);
    T* __restrict__ dst = static_cast<T*>(a.dst);

    Calc f[V][Q];
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        constexpr int cx = L::cx(q), cy = L::cy(q), cz = L::cz(q);
        const int sy = cy > 0 ? ym : (cy < 0 ? yp : y);
        const int sz = cz > 0 ? zm : (cz < 0 ? zp : z);
        const T* __restrict__ row = src + q * Ly.plane + Ly.off + Ly.px * sy + Ly.pxy * sz;
        T v[V];
        if constexpr (V == 1) {
            v[0] = row[cx == 0 ? x0 : (cx > 0 ? xm : xpv)];
        } else {
            const VecT<T, V> A = *reinterpret_cast<const VecT<T, V>*>(row + x0);
            if constexpr (cx == 0) {
#pragma unroll
                for (int i = 0; i < V; ++i) v[i] = A.v[i];
            } else if constexpr (cx > 0) {
                v[0] = row[xm];
#pragma unroll
                for (int i = 1; i < V; ++i) v[i] = A.v[i - 1];
            } else {
#pragma unroll
                for (int i = 0; i < V - 1; ++i) v[i] = A.v[i + 1];
                v[V - 1] = row[xpv];
                // last, partially filled vector of a periodic row: lane of x = xl
                // takes x = 1 (on a walled row that lane is NEAR and masked)
                if (partial) {
#pragma unroll
                    for (int i = 0; i < V - 1; ++i)
                        if (x0 + i == Ly.xl) v[i] = row[1];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < V; ++i) f[i][q] = IO::template load<q>(v[i]);
    });

    // the loads above are issued before this test (every row they touch lies
    // inside the ghosted box), so the kind lookup costs no extra round trip
    if (!any) return true;
#pragma unroll
    for (int i = 0; i < V; ++i) converted<M>(f[i]);

    Calc alpha[V];
    if constexpr (BRINK) {
        const Calc* al = static_cast<const Calc*>(a.alpha);
#pragma unroll
        for (int i = 0; i < V; ++i) alpha[i] = act[i] ? al[e0 + i] : Calc(0);
    }

    bool finite = true;
#pragma unroll
    for (int i = 0; i < V; ++i) {
        if constexpr (M == Mode::EXACT64) {
            collide_exact<L>(f[i], a.tau, a.omega);
        } else {
            Mom4<Calc> mom;
            const Calc base = collide_shifted<L, Calc, BRINK, kRcp<M>, IO::SX>(f[i], static_cast<Calc>(a.omega),
                                            BRINK ? alpha[i] : Calc(0),
                                            static_cast<Calc>(a.tau * a.g[0]),
                                            static_cast<Calc>(a.tau * a.g[1]),
                                            static_cast<Calc>(a.tau * a.g[2]), HIST ? mom.v : nullptr);
            if constexpr (HIST) {
                if (act[i]) static_cast<Mom4<Calc>*>(a.hist)[cell_index(Ly, x0 + i, y, z)] = mom;
            }
            finite &= !act[i] || finite_calc(base);
        }
    }

    bool all = true;
#pragma unroll
    for (int i = 0; i < V; ++i) all &= act[i];
    with_put<Put::Through>(POLICY ? a.cached : 0, [&](auto pc) {
        constexpr Put P = decltype(pc)::value;
        static_for<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            T* __restrict__ out = dst + q * Ly.plane + e0;
            if (all) {
                VecT<T, V> o;
#pragma unroll
                for (int i = 0; i < V; ++i) o.v[i] = IO::template store<q>(f[i][q]);
                put<P>(reinterpret_cast<VecT<T, V>*>(out), o);
            } else {
#pragma unroll
                for (int i = 0; i < V; ++i)
                    if (act[i]) put<P>(out + i, IO::template store<q>(f[i][q]));
            }
        });
    });
    return finite;
}

template <class L, Mode M, int V, bool FLAGS, bool BRINK, bool HIST = false>
__global__ void __launch_bounds__(256) k_bulk(StepArgs a, int nbx, int nby) {
    const int b = blockIdx.x;
    const int bx = b % nbx;
    const int t = b / nbx;
    const int by = t % nby;
    const int z = 1 + t / nby;
    const int xv = bx * blockDim.x + threadIdx.x;
    const int y = 1 + by * blockDim.y + threadIdx.y;
    bulk_cells<L, M, V, FLAGS, BRINK, HIST>(a, 1 + xv * V, y, z);
}

// ---------------------------------------------------------------------------
// Boundary rules, evaluated by the fluid cell x for a non-fluid source b.
// own[] holds x's post-collision values (the values the reference's rule
// reads from its fluid neighbour), in the Calc representation of the mode.

// The rules read x's own values only through their plain sum, their three
// momentum sums and the single value own[qbar]. OwnSums holds the sums, each
// accumulated from 0 over ascending q: the order of the reference's density()
// and velocity() (include/collision.hpp:7-31), which EXACT64 keeps bit for
// bit (adding -v equals subtracting v; directions with c_d = 0 add nothing).
template <class Calc>
struct OwnSums {
    Calc s, m0, m1, m2;
};

template <class L, class Calc>
struct OwnAcc {
    OwnSums<Calc> r{Calc(0), Calc(0), Calc(0), Calc(0)};
    template <int q>
    __device__ __forceinline__ void add(Calc v) {
        r.s += v;
        if constexpr (L::cx(q) > 0) r.m0 += v;
        if constexpr (L::cx(q) < 0) r.m0 -= v;
        if constexpr (L::cy(q) > 0) r.m1 += v;
        if constexpr (L::cy(q) < 0) r.m1 -= v;
        if constexpr (L::cz(q) > 0) r.m2 += v;
        if constexpr (L::cz(q) < 0) r.m2 -= v;
    }
};

template <class L, class Calc>
__device__ __forceinline__ OwnSums<Calc> own_sums(const Calc (&own)[L::Q]) {
    OwnAcc<L, Calc> acc;
    static_for<0, L::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        acc.template add<q>(own[q]);
    });
    return acc.r;
}

// Own values read from the source field at element e (one pass, nothing kept).
template <class L, Mode M, bool B32 = false>
__device__ __forceinline__ OwnSums<typename Io<M, L>::Calc> own_sums_at(
    const typename Io<M, L>::T* __restrict__ src, int64_t plane, typename ElemIdx<B32>::type e) {
    using IO = Io<M, L>;
    OwnAcc<L, typename IO::Calc> acc;
    static_for<0, L::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        acc.template add<q>(IO::template to_calc<q>(plane_ref<B32>(src, q, plane, e)));
    });
    return acc.r;
}

// c ? a : b by bit masks. A plain select between two array elements can be
// turned into a select between their addresses, which moves both arrays
// out of registers into scratch memory.
template <class T>
__device__ __forceinline__ T pick_bits(bool c, T a, T b) {
    using U = typename std::conditional<sizeof(T) == 8, uint64_t, uint32_t>::type;
    static_assert(sizeof(T) == sizeof(U), "float or double");
    const U m = U(0) - static_cast<U>(c);
    return __builtin_bit_cast(T, (__builtin_bit_cast(U, a) & m) | (__builtin_bit_cast(U, b) & ~m));
}

// The MovingWall and Outflow/Pressure values of the fp32/fp64 storage modes,
// shared by rule_value and rule_value_flat so that both round alike.
// MovingWall (include/boundary.hpp:55-65) with c_q . u_wall tabulated per
// condition.
template <class L, class Calc, int q>
__device__ __forceinline__ Calc moving_wall_rule(const OwnSums<Calc>& os, Calc finv, const GCond& cd) {
    const Calc rho = Calc(1) + os.s;
    Calc cu;
    if constexpr (std::is_same<Calc, float>::value)
        cu = cd.cu32[q];
    else
        cu = static_cast<Calc>(cd.cu64[q]);
    return finv + static_cast<Calc>(6.0 * weight<L>(q)) * rho * cu;
}

// Outflow / Pressure (include/boundary.hpp:140-147, 206-211):
// (feq_q - w) + (feq_qbar - w) - finv at the condition's density and x's
// velocity; the odd part of the two equilibria cancels.
template <class L, class Calc, int q>
__device__ __forceinline__ Calc outflow_rule(const OwnSums<Calc>& os, Calc finv, const GCond& cd) {
    const Calc rr = static_cast<Calc>(cd.rho);
    const Calc ir = Calc(1) / rr;
    const Calc ux = os.m0 * ir, uy = os.m1 * ir, uz = os.m2 * ir;
    const Calc cu = Calc(L::cx(q)) * ux + Calc(L::cy(q)) * uy + Calc(L::cz(q)) * uz;
    const Calc uu = ux * ux + uy * uy + uz * uz;
    const Calc even = (rr - Calc(1)) + rr * (Calc(4.5) * cu * cu - Calc(1.5) * uu);
    return static_cast<Calc>(2.0 * weight<L>(q)) * even - finv;
}

// Value of a NoSlip, MovingWall, Inflow, Outflow or Pressure rule for
// direction q, from x's own sums and own[qbar] (finv).
template <class L, Mode M, int q, int RULES = RULES_ALL>
__device__ __forceinline__ typename Io<M, L>::Calc rule_value(const GCond& cd,
                                                             const OwnSums<typename Io<M, L>::Calc>& os,
                                                             typename Io<M, L>::Calc finv) {
    using Calc = typename Io<M, L>::Calc;
    constexpr int Q = L::Q;
    const int kind = cd.kind;
    if constexpr ((RULES & RULE_MOVINGWALL) != 0) {
        if (kind == BC_MOVINGWALL) {  // boundary.hpp:55-65
            if constexpr (M == Mode::EXACT64) {
                double c_dot_u = 0;
                c_dot_u += static_cast<double>(L::cx(q)) * cd.vel[0];
                c_dot_u += static_cast<double>(L::cy(q)) * cd.vel[1];
                c_dot_u += static_cast<double>(L::cz(q)) * cd.vel[2];
                constexpr double cs = kCS;
                return finv + 2.0 * weight<L>(q) * os.s * c_dot_u / (cs * cs);
            } else {
                return moving_wall_rule<L, Calc, q>(os, finv, cd);
            }
        }
    }
    if constexpr ((RULES & RULE_INFLOW) != 0) {
        if (kind == BC_INFLOW)  // boundary.hpp:176-178, feq precomputed on the host
            return (M == Mode::EXACT64) ? static_cast<Calc>(cd.feq[q]) : static_cast<Calc>(cd.geq[q]);
    }
    if constexpr ((RULES & RULE_OUTFLOW) != 0) {
        if (kind == BC_OUTFLOW || kind == BC_PRESSURE) {  // boundary.hpp:140-147, 206-211
            if constexpr (M == Mode::EXACT64) {
                const double u[3] = {os.m0 / cd.rho, os.m1 / cd.rho, os.m2 / cd.rho};
                const double fq = feq_exact<L, q>(cd.rho, u);
                const double fb = feq_exact<L, Q - 1 - q>(cd.rho, u);
                return fq + fb - finv;
            } else {
                return outflow_rule<L, Calc, q>(os, finv, cd);
            }
        }
    }
    return finv;  // BC_NOSLIP, boundary.hpp:26-28
}

// rule_value without branches (fp32/fp64 storage modes): every family built
// in is evaluated and the condition's kind selects one. cd must be a valid
// condition even where the result is not used, so a caller can issue the
// loads of all its links at once instead of one link after another.
template <class L, Mode M, int q, int RULES = RULES_ALL>
__device__ __forceinline__ typename Io<M, L>::Calc rule_value_flat(const GCond& cd,
                                                                  const OwnSums<typename Io<M, L>::Calc>& os,
                                                                  typename Io<M, L>::Calc finv) {
    static_assert(M != Mode::EXACT64, "the reference-order mode keeps rule_value");
    using Calc = typename Io<M, L>::Calc;
    const int kind = cd.kind;
    Calc v = finv;  // BC_NOSLIP
    if constexpr ((RULES & RULE_MOVINGWALL) != 0) {
        const Calc w = moving_wall_rule<L, Calc, q>(os, finv, cd);
        v = kind == BC_MOVINGWALL ? w : v;
    }
    if constexpr ((RULES & RULE_INFLOW) != 0) {
        const Calc g = static_cast<Calc>(cd.geq[q]);
        v = kind == BC_INFLOW ? g : v;
    }
    if constexpr ((RULES & RULE_OUTFLOW) != 0) {
        const Calc o = outflow_rule<L, Calc, q>(os, finv, cd);
        v = (kind == BC_OUTFLOW || kind == BC_PRESSURE) ? o : v;
    }
    return v;
}

// FreeSlip candidates (include/boundary.hpp:93-110), in order: which of the
// boundary cell's coordinates (x, y, z) are replaced by the fluid cell's, i.e.
// which velocity components the candidate's population reflects.
constexpr int kFsSwap[6][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {0, 1, 1}, {1, 0, 1}, {1, 1, 0}};

// Direction index of velocity (cx, cy, cz) (include/model.h velocity_index),
// evaluated at compile time.
template <class L>
constexpr int dir_of(int cx, int cy, int cz) {
    for (int q = 0; q < L::Q; ++q)
        if (L::cx(q) == cx && L::cy(q) == cy && L::cz(q) == cz) return q;
    return -1;
}


// Value that fluid cell x = (x,y,z) pulls in direction q from the non-fluid
// cell b = (sx,sy,sz) (element se) with condition cd: the value the reference's
// rule writes into b[q] in collide pass 2 (include/boundary.hpp). os holds
// the sums of x's own post-collision values and own(k) returns own value k.
// Sets stale when the rule writes nothing (FreeSlip with no fluid candidate);
// the value returned is then b's stored value, which is what the reference
// reads too. FS = false builds the rule without the FreeSlip case, for
// domains that have no FreeSlip condition. B32 indexes with 32-bit offsets
// (planes under 4 GiB).
template <class L, Mode M, int q, bool FS = true, bool B32 = false, class OwnFn>
__device__ __forceinline__ typename Io<M, L>::Calc pull_boundary(
    const StepArgs& a, const GCond& cd, const OwnSums<typename Io<M, L>::Calc>& os, OwnFn own, int x,
    int y, int z, int sx, int sy, int sz, typename ElemIdx<B32>::type se, bool& stale) {
    using IO = Io<M, L>;
    using T = typename IO::T;
    constexpr int Q = L::Q;
    constexpr int cx = L::cx(q), cy = L::cy(q), cz = L::cz(q);
    const FieldLayout& Ly = a.L;
    const T* __restrict__ src = static_cast<const T*>(a.src);
    stale = false;
    if constexpr (FS) {
        if (cd.kind == BC_FREESLIP) {  // boundary.hpp:91-110 with b = (sx,sy,sz), b + c_q = x
            // Candidates in the reference's order; candidate j replaces the
            // coordinates flagged in kFsSwap[j] by x's and reflects those
            // velocity components. The reflected directions are compile-time.
            typename IO::Calc v{};
            bool found = false;
            static_for<0, 6>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                constexpr int rq = dir_of<L>(kFsSwap[j][0] ? -cx : cx, kFsSwap[j][1] ? -cy : cy,
                                             kFsSwap[j][2] ? -cz : cz);
                static_assert(rq >= 0, "reflected velocity outside the lattice");
                if (!found) {
                    const auto ce = elem_at<B32>(Ly, kFsSwap[j][0] ? x : sx, kFsSwap[j][1] ? y : sy,
                                                 kFsSwap[j][2] ? z : sz);
                    if (kind_at(a.kind, ce) < KIND_COND0) {
                        v = IO::template to_calc<rq>(plane_ref<B32>(src, rq, Ly.plane, ce));
                        found = true;
                    }
                }
            });
            if (found) return v;
            stale = true;
            return IO::template to_calc<q>(plane_ref<B32>(src, q, Ly.plane, se));
        }
    }
    if (cd.kind < BC_NOSLIP || cd.kind > BC_PRESSURE) {
        stale = true;
        return IO::template to_calc<q>(plane_ref<B32>(src, q, Ly.plane, se));
    }
    return rule_value<L, M, q>(cd, os, own(std::integral_constant<int, Q - 1 - q>{}));
}

// The same with x's own values already in registers.
template <class L, Mode M, int q, bool FS = true>
__device__ __forceinline__ typename Io<M, L>::Calc pull_nonfluid(
    const StepArgs& a, const GCond& cd, const typename Io<M, L>::Calc (&own)[L::Q], int x, int y,
    int z, int sx, int sy, int sz, int64_t se, bool& stale) {
    using Calc = typename Io<M, L>::Calc;
    const OwnSums<Calc> os = own_sums<L, Calc>(own);
    return pull_boundary<L, M, q, FS>(a, cd, os, [&](auto kc) { return own[decltype(kc)::value]; }, x, y, z,
                                  sx, sy, sz, se, stale);
}

// ---------------------------------------------------------------------------
// One NEAR cell (fluid with a non-fluid source). Returns false when the cell
// read a NaN or infinite value.
template <class L, Mode M>
__device__ __forceinline__ bool near_cell(const StepArgs& a, int x, int y, int z) {
    using IO = Io<M, L>;
    using T = typename IO::T;
    using Calc = typename IO::Calc;
    constexpr int Q = L::Q;
    const FieldLayout& Ly = a.L;
    const int64_t e = cell_elem(Ly, x, y, z);
    const T* __restrict__ src = static_cast<const T*>(a.src);
    T* __restrict__ dst = static_cast<T*>(a.dst);

    // x's own post-collision values (the rules' inputs): sums now, single
    // values reloaded when a rule needs one
    const OwnSums<Calc> os = own_sums_at<L, M>(src, Ly.plane, e);
    auto own = [&](auto kc) {
        constexpr int k = decltype(kc)::value;
        return IO::template to_calc<k>(src[k * Ly.plane + e]);
    };

    Calc f[Q];
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        constexpr int cx = L::cx(q), cy = L::cy(q), cz = L::cz(q);
        const int sx = wrap_if(x - cx, Ly.xl, Ly.per[0]);
        const int sy = wrap_if(y - cy, Ly.yl, Ly.per[1]);
        const int sz = wrap_if(z - cz, Ly.zl, Ly.per[2]);
        const int64_t se = cell_elem(Ly, sx, sy, sz);
        const uint8_t k = kind_at(a.kind, se);
        if (k < KIND_COND0 || a.materialised) {
            f[q] = IO::template load<q>(src[q * Ly.plane + se]);
        } else {
            bool stale;
            f[q] = IO::template through_storage<q>(pull_boundary<L, M, q>(a, cond_at(a.conds, k - KIND_COND0), os, own,
                                                                          x, y, z, sx, sy, sz, se, stale));
        }
    });

    bool finite = true;
    if constexpr (M == Mode::EXACT64) {
        collide_exact<L>(f, a.tau, a.omega);
    } else {
        Calc alpha = Calc(0);
        if (a.alpha) alpha = static_cast<const Calc*>(a.alpha)[e];
        if (a.alpha) {
            finite = finite_calc(collide_shifted<L, Calc, true, kRcp<M>, IO::SX>(f, static_cast<Calc>(a.omega), alpha,
                                           static_cast<Calc>(a.tau * a.g[0]),
                                           static_cast<Calc>(a.tau * a.g[1]),
                                           static_cast<Calc>(a.tau * a.g[2])));
        } else {
            finite = finite_calc(collide_shifted<L, Calc, false, kRcp<M>, IO::SX>(f, static_cast<Calc>(a.omega), Calc(0),
                                                                          Calc(0), Calc(0), Calc(0)));
        }
    }
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        dst[q * Ly.plane + e] = IO::template store<q>(f[q]);
    });
    return finite;
}

// Element o of base (B32: at byte offset o) in global memory.
template <bool B32, class T>
__device__ __forceinline__ PlaneElem<const T>& elem_ref(const T* base, typename ElemIdx<B32>::type o) {
    using E = PlaneElem<const T>;
    using EB = std::conditional_t<IsDual<T>::value, const char, Glob<const char>>;
    if constexpr (B32)
        return *reinterpret_cast<E*>(reinterpret_cast<EB*>((E*)base) + o);
    else
        return ((E*)base)[o];
}

// Byte offsets of a cell's neighbours in a plane under 4 GiB, for a wavefront
// whose lanes share y and z (row tiles): per lane along x, in scalar registers
// along y and z, wrapped along periodic axes. Index 0, 1, 2: -1, 0, +1. An
// access is then a scalar base, direction plane and row included, plus one of
// three lane offsets: no address arithmetic per lane and no divergence at
// periodic faces.
template <class T>
struct RowNb {
    uint32_t x[3];
    int64_t y[3], z[3];
    __device__ __forceinline__ RowNb(const FieldLayout& L, int cx, int cy, int cz) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            x[i] = static_cast<uint32_t>(sizeof(T)) * static_cast<uint32_t>(wrap_if(cx + i - 1, L.xl, L.per[0]));
            y[i] = static_cast<int64_t>(sizeof(T)) * L.px * wrap_if(cy + i - 1, L.yl, L.per[1]);
            z[i] = static_cast<int64_t>(sizeof(T)) * (L.off + L.pxy * wrap_if(cz + i - 1, L.zl, L.per[2]));
        }
    }
    // value of plane q at x + S c_q
    template <class L, int q, int S>
    __device__ __forceinline__ Glob<T>& at(T* base, int64_t plane) const {
        auto* p = reinterpret_cast<Glob<char>*>((Glob<T>*)(base + q * plane)) + (y[1 + S * L::cy(q)] + z[1 + S * L::cz(q)]);
        return *reinterpret_cast<Glob<T>*>(p + x[1 + S * L::cx(q)]);
    }
    template <class L, int q, int S>
    __device__ __forceinline__ Glob<const T>& at(const T* base, int64_t plane) const {
        return at<L, q, S>(const_cast<T*>(base), plane);
    }
    // the same as an offset from the plane's start
    template <class L, int q, int S>
    __device__ __forceinline__ uint32_t offset() const {
        return x[1 + S * L::cx(q)] + static_cast<uint32_t>(y[1 + S * L::cy(q)] + z[1 + S * L::cz(q)]);
    }
};

// Row tiles: wavefront w of z plane 1 + blockIdx.y takes cells 64 (w mod tpr)
// + 1 .. of row 1 + w / tpr. False past the row or the plane.
__device__ __forceinline__ bool row_tile_cell(const FieldLayout& L, int tpr, int rev, int& x, int& y, int& z) {
    const int w = static_cast<int>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    y = 1 + w / tpr;
    z = rev ? L.zl - static_cast<int>(blockIdx.y) : 1 + static_cast<int>(blockIdx.y);
    x = 1 + (w % tpr) * 64 + static_cast<int>(threadIdx.x & 63);
    return y <= L.yl && x <= L.xl;
}

// f[q] <- the value at source(q) of plane q (byte offset for B32, else element).
template <class L, Mode M, bool B32, class Source>
__device__ __forceinline__ void pull_plain(const typename Io<M, L>::T* __restrict__ src, int64_t plane, Source source,
                                           typename Io<M, L>::Calc (&f)[L::Q]) {
    static_for<0, L::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        f[q] = Io<M, L>::template load<q>(elem_ref<B32>(src + q * plane, source(qc)));
    });
}

// ---------------------------------------------------------------------------
// The Q values a fluid cell takes in: the pulls from x - c_q, and for each
// link q in `links` (NoSlip sources) its own value of the opposite direction,
// which is what that rule returns. Where a lane of the wavefront has links,
// each load's address is selected per lane, so bounce-back costs no loads of
// its own. (Loading all Q own values beside the pulls, as any rule may need
// them, the 64-cell tiles of small or narrow domains, where nearly every
// wavefront holds a wall lane, issued 47 loads a tile for 20 wanted. Single
// steps: 96^3 fp64 cavity 71.3 -> 57.8 us, 256^3 fp16 cavity 276 -> 254 us,
// 192 x 96 x 96 D3Q27 fp64 sphere channel 239 -> 206 us.) source(q) is the
// byte offset (B32) or element of x - c_q in its plane, e the element of x.
// Selected addresses are 32-bit byte offsets from the buffer where it is
// under 4 GiB (span32), else (FAR) 64-bit.
template <class L, Mode M, bool B32, bool FAR = true, class Source, class Plain>
__device__ __forceinline__ void pull_all(const typename Io<M, L>::T* __restrict__ src, int64_t plane,
                                         typename ElemIdx<B32>::type e, uint32_t links, int span32, Source source,
                                         typename Io<M, L>::Calc (&f)[L::Q], Plain plain) {
    using IO = Io<M, L>;
    using T = typename IO::T;
    constexpr int Q = L::Q;
    if (!__any(static_cast<int>(links))) {
        plain();
        return;
    }
    if constexpr (B32) {
        if (!FAR || span32) {
            const uint32_t plane_bytes = static_cast<uint32_t>(plane) * static_cast<uint32_t>(sizeof(T));
            static_for<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                // (the empty asm has the multiples recomputed where they are
                // used: hoisted, they overflow the scalar registers)
                uint32_t pb = plane_bytes;
                asm volatile("" : "+s"(pb));
                const uint32_t from = source(qc) + q * pb;
                const uint32_t own = e * static_cast<uint32_t>(sizeof(T)) + (Q - 1 - q) * pb;
                const uint32_t m = 0u - ((links >> q) & 1u);
                f[q] = IO::template load<q>(elem_ref<true>(src, (own & m) | (from & ~m)));
            });
            return;
        }
    }
    if constexpr (FAR || !B32) static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const T* from = (const T*)&elem_ref<B32>(src + q * plane, source(qc));
        const T* own = src + ((Q - 1 - q) * plane + static_cast<int64_t>(e));
        using E = PlaneElem<const T>;
        f[q] = IO::template load<q>(*(E*)(((links >> q) & 1u) ? own : from));
    });
}

template <class L, Mode M, bool B32, bool FAR = true, class Source>
__device__ __forceinline__ void pull_all(const typename Io<M, L>::T* __restrict__ src, int64_t plane,
                                         typename ElemIdx<B32>::type e, uint32_t links, int span32, Source source,
                                         typename Io<M, L>::Calc (&f)[L::Q]) {
    pull_all<L, M, B32, FAR>(src, plane, e, links, span32, source, f,
                             [&] { pull_plain<L, M, B32>(src, plane, source, f); });
}

// ---------------------------------------------------------------------------
// The pulls of a NEAR cell x with LINK_RULES (element e, ghosted-box coordinates x, y, z)
// from non-fluid sources, f[q] for every link q of its mask, replaced by
// their boundary values, from x's stored values in a.src (the reference's
// boundary pass folded into the pull).
// ALL: any NEAR cell, those with NoSlip links only among them; the condition
// that all links share comes first.
template <class L, Mode M, bool FS, bool B32, bool ALL = false>
__device__ __forceinline__ void near_rules(const StepArgs& a, typename ElemIdx<B32>::type e, int x, int y, int z,
                                           typename Io<M, L>::Calc (&f)[L::Q]) {
    using IO = Io<M, L>;
    using T = typename IO::T;
    using Calc = typename IO::Calc;
    using I = typename ElemIdx<B32>::type;
    constexpr int Q = L::Q;
    const FieldLayout& Ly = a.L;
    const T* __restrict__ src = static_cast<const T*>(a.src);
    const OwnSums<Calc> os = own_sums_at<L, M, B32>(src, Ly.plane, e);
    auto own = [&](auto kc) {
        constexpr int kk = decltype(kc)::value;
        return IO::template to_calc<kk>(plane_ref<B32>(src, kk, Ly.plane, e));
    };
    const uint32_t lm = glob(a.lmask)[e] & LINK_BITS;
    // Every link that is not NoSlip under one condition (not FreeSlip,
    // whose rule reads other cells), as on edges between a lid and walls:
    // one branch on its kind, then that family's loads go out together,
    // where the path below waits for two lookups a link, one link after
    // the other. The values are rule_value's (same functions). (A caller
    // without the rule words takes the path below.) With the shared path
    // only where all links agree, and not in fp64: 16^3 fp32 cavity, 10
    // steps with moments 140 -> 90 us, 64^3 fp64 cavity, 100 steps 2.21 ->
    // 1.83 ms, 250 x 54 x 54 fp16 pipe 2.51 -> 2.14 ms, 30 mixed cavities
    // 89.9 -> 83.6 us a step, D3Q27 sphere channel 192 x 96 x 96, 100
    // steps 10.8 -> 10.4 ms.
    uint32_t rm = lm;
    int rc = LCOND_MIXED;
    if constexpr (ALL) rc = glob(a.lcond)[e];
    if (rc == LCOND_MIXED && a.rword) {
        const uint32_t rw = glob(a.rword)[e];
        if ((rw >> RULE_SHIFT) != RULE_SLOW) {
            rm = rw;
            rc = static_cast<int>(rw >> RULE_SHIFT);
        } else if constexpr (!ALL) {  // (more than RULE_SLOW conditions)
            rc = glob(a.lcond)[e];
        }
    }
    if (rc != LCOND_MIXED) {
        const GCond& cd = cond_at(a.conds, rc);
        const int ck = cd.kind;
        // (the reference-order outflow rule, two equilibria a link, is
        // built once, below)
        if ((!FS || ck != BC_FREESLIP) && (M != Mode::EXACT64 || (ALL && ck == BC_NOSLIP) || ck == BC_MOVINGWALL || ck == BC_INFLOW)) {
            auto finv = [&](auto qc) { return own(std::integral_constant<int, Q - 1 - decltype(qc)::value>{}); };
            auto put = [&](auto qc, Calc own_inv, Calc v) {
                constexpr int q = decltype(qc)::value;
                const Calc b = pick_bits(((rm >> q) & 1u) != 0, v, own_inv);  // (NoSlip: the own value)
                f[q] = pick_bits(((lm >> q) & 1u) != 0, IO::template through_storage<q>(b), f[q]);
            };
            if (ck == BC_MOVINGWALL) {
                static_for<0, Q>([&](auto qc) {
                    const Calc w = finv(qc);
                    put(qc, w, rule_value<L, M, decltype(qc)::value, RULE_MOVINGWALL>(cd, os, w));
                });
            } else if (ck == BC_INFLOW) {
                static_for<0, Q>([&](auto qc) {
                    const Calc w = finv(qc);
                    put(qc, w, rule_value<L, M, decltype(qc)::value, RULE_INFLOW>(cd, os, w));
                });
            } else if (ALL && ck == BC_NOSLIP) {
                static_for<0, Q>([&](auto qc) {
                    const Calc w = finv(qc);
                    put(qc, w, w);
                });
            } else if constexpr (M != Mode::EXACT64) {  // Outflow, Pressure
                static_for<0, Q>([&](auto qc) {
                    const Calc w = finv(qc);
                    put(qc, w, outflow_rule<L, Calc, decltype(qc)::value>(os, w, cd));
                });
            }
            return;
        }
    }
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        constexpr int cx = L::cx(q), cy = L::cy(q), cz = L::cz(q);
        if (lm & (1u << q)) {
            const int sx = wrap_if(x - cx, Ly.xl, Ly.per[0]);
            const int sy = wrap_if(y - cy, Ly.yl, Ly.per[1]);
            const int sz = wrap_if(z - cz, Ly.zl, Ly.per[2]);
            const I se = elem_at<B32>(Ly, sx, sy, sz);
            const uint8_t sk = kind_at(a.kind, se);
            bool stale;
            f[q] = IO::template through_storage<q>(pull_boundary<L, M, q, FS, B32>(
                a, cond_at(a.conds, sk - KIND_COND0), os, own, x, y, z, sx, sy, sz, se, stale));
        }
    });
}

// One interior cell of any kind, for kernels that hand every cell of a region
// to a thread (the cell tiles). Non-fluid cells return at once. The link word
// says which directions bounce back (pull_all); a cell with a link of another
// rule pulls every direction plainly (sources wrapped along periodic axes;
// along a walled axis the source may be a ghost or solid cell) and then
// replaces the values pulled from non-fluid sources by their boundary values
// (as near_cell). All lanes collide and store together. The bits
// equal those of bulk_cells / near_cell for the same cell. B32 takes the
// cell's own and plain-pull addresses as 32-bit byte offsets (planes under
// 4 GiB). Returns false when a fluid cell read a NaN or infinite value.
// HIST records drho and u of the incoming populations, and 1 + the sum of
// the own values of a cell with moving-wall links (StepArgs::hist, rho_own).
// AHEAD sends the pulls ahead of the cell's kind, and every NEAR cell takes
// the values of all its links from near_rules: a shorter chain of accesses for
// lanes without links, a longer one and Q more loads for those with. make_plan
// and pulls_ahead (domain_impl.hpp) say where it is taken.
template <class L, Mode M, bool FS = true, bool B32 = false, bool CACHED = false, bool HIST = false, bool ROW = false,
          bool AHEAD = false>
__device__ __forceinline__ bool any_cell(const StepArgs& a, int x, int y, int z) {
    using IO = Io<M, L>;
    using T = typename IO::T;
    using Calc = typename IO::Calc;
    using I = typename ElemIdx<B32>::type;
    constexpr int Q = L::Q;
    const FieldLayout& Ly = a.L;
    const I e = elem_at<B32>(Ly, x, y, z);
    const uint32_t w = AHEAD ? kind_at(a.kind, e) : glob(a.lmask)[e];  // cell kind (AHEAD) or link word
    const T* __restrict__ src = static_cast<const T*>(a.src);
    T* __restrict__ dst = static_cast<T*>(a.dst);
    if (!AHEAD && (w & LINK_NOT_FLUID)) return true;

    // A cell with a link of another rule than NoSlip pulls plainly and
    // patches all its links below; one in its first step pulls stored values.
    // (Pulls sent ahead of the link word with only the bounced values loaded
    // afterwards took 2 to 14 % longer on cavities from 64^3 up, and 2.43
    // against 1.98 ms in the AHEAD form on 512 batched ones.)
    constexpr I US = B32 ? static_cast<I>(sizeof(T)) : I(1);  // unit of the sources
    Calc f[Q];
    // Away from the faces of periodic axes every source is a fixed element
    // offset c_x + c_y px + c_z pxy away; on those faces the source wraps.
    const bool wraps = (Ly.per[0] && (x == 1 || x == Ly.xl)) || (Ly.per[1] && (y == 1 || y == Ly.yl)) ||
                       (Ly.per[2] && (z == 1 || z == Ly.zl));
    auto near_src = [&](auto qc) -> I {
        constexpr int q = decltype(qc)::value;
        constexpr int cx = L::cx(q), cy = L::cy(q), cz = L::cz(q);
        const int64_t d = cx + (cy > 0 ? Ly.px : (cy < 0 ? -Ly.px : 0)) + (cz > 0 ? Ly.pxy : (cz < 0 ? -Ly.pxy : 0));
        return (e - static_cast<I>(d)) * US;
    };
    auto wrap_src = [&](auto qc) -> I {
        constexpr int q = decltype(qc)::value;
        return elem_at<B32>(Ly, wrap_if(x - L::cx(q), Ly.xl, Ly.per[0]), wrap_if(y - L::cy(q), Ly.yl, Ly.per[1]),
                            wrap_if(z - L::cz(q), Ly.zl, Ly.per[2])) * US;
    };
    const bool rules = (AHEAD ? w == KIND_NEAR : (w & LINK_RULES) != 0) && !a.materialised;
    const uint32_t links = (AHEAD || rules || a.materialised) ? 0u : w;
    if constexpr (AHEAD) {
        static_assert(!HIST, "plain steps");
        if constexpr (ROW) {
            const RowNb<T> nb(Ly, x, y, z);
            static_for<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                f[q] = IO::template load<q>(nb.template at<L, q, -1>(src, Ly.plane));
            });
        } else if (!wraps) {
            pull_plain<L, M, B32>(src, Ly.plane, near_src, f);
        } else {
            pull_plain<L, M, B32>(src, Ly.plane, wrap_src, f);
        }
        if (w >= KIND_COND0) return true;
    } else if constexpr (ROW) {
        static_assert(B32, "row tiles take 32-bit offsets");
        const RowNb<T> nb(Ly, x, y, z);
        pull_all<L, M, true>(src, Ly.plane, e, links, a.span32,
                             [&](auto qc) { return nb.template offset<L, decltype(qc)::value, -1>(); }, f, [&] {
            static_for<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                f[q] = IO::template load<q>(nb.template at<L, q, -1>(src, Ly.plane));
            });
        });
    } else if (!wraps) {
        pull_all<L, M, B32>(src, Ly.plane, e, links, a.span32, near_src, f);
    } else {
        pull_all<L, M, B32>(src, Ly.plane, e, links, a.span32, wrap_src, f);
    }
    converted<M>(f);
    if (rules) {
        near_rules<L, M, FS, B32, AHEAD>(a, e, x, y, z, f);
        if constexpr (HIST) {  // (read by the moving walls' gradient only)
            const int lc = glob(a.lcond)[e];
            if (lc == LCOND_MIXED || cond_at(a.conds, lc).kind == BC_MOVINGWALL) {
                Calc r = Calc(1);
                static_for<0, Q>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    r += IO::template to_calc<q>(plane_ref<B32>(src, q, Ly.plane, e));
                });
                glob(static_cast<Calc*>(a.rho_own))[glob(a.near_idx)[e]] = r;
            }
        }
    }

    bool finite = true;
    if constexpr (M == Mode::EXACT64) {
        collide_exact<L>(f, a.tau, a.omega);
    } else if (a.alpha) {
        const Calc alpha = static_cast<const Calc*>(a.alpha)[e];
        finite = finite_calc(collide_shifted<L, Calc, true, kRcp<M>, IO::SX>(f, static_cast<Calc>(a.omega), alpha,
                                                static_cast<Calc>(a.tau * a.g[0]),
                                                static_cast<Calc>(a.tau * a.g[1]),
                                                static_cast<Calc>(a.tau * a.g[2])));
    } else {
        Mom4<Calc> mom;
        finite = finite_calc(collide_shifted<L, Calc, false, kRcp<M>, IO::SX>(
            f, static_cast<Calc>(a.omega), Calc(0), Calc(0), Calc(0), Calc(0), HIST ? mom.v : nullptr));
        if constexpr (HIST) {
            const Mom4Raw<Calc> m = {mom.v[0], mom.v[1], mom.v[2], mom.v[3]};
            __builtin_nontemporal_store(m, &glob(static_cast<Mom4Raw<Calc>*>(a.hist))[cell_index(Ly, x, y, z)]);
        }
    }
    static_for<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        put<CACHED ? Put::Keep : Put::Stream, T>(&plane_ref<B32>(dst, q, Ly.plane, e), IO::template store<q>(f[q]));
    });
    return finite;
}

// Blocks of 256 per CU the cell-tile kernel is compiled for: 6 (80 VGPRs)
// with 32- and 16-bit storage up to D3Q19, 4 in fp64 reference order; no bound
// with F64S, whose values take twice the registers, or with D3Q27, where 80
// VGPRs spill. FreeSlip's rule takes more: D3Q19 spilled 39 (fp32), 20 (fp16),
// 12 (bf16) and 76 (fp64) registers under those bounds, which cost more than
// the waves gave: there 5 blocks, and no bound in fp64. us a step, those
// bounds / these, half-slip cavities: 28x30x30 fp32 16.4 / 14.5, fp16 16.4 /
// 14.7, bf16 16.1 / 14.6, fp64 18.7 / 15.8; 160x128x128 103 / 92, 73.8 / 70.5,
// 75.2 / 71.1, 194 / 179.
template <class L, Mode M, bool FS>
constexpr int cells_min_blocks() {
    if (M == Mode::EXACT64) return L::Q > 19 || (FS && L::Q > 15) ? 1 : 4;
    if (M == Mode::F64S || L::Q > 19) return 1;
    return FS && L::Q > 15 ? 5 : 6;
}

// Cell-tile kernels. k_cell_rows (planes under 4 GiB, no FreeSlip): row tiles,
// for padded rows: whole lines per access, y and z in scalar registers, no
// division per lane. Plane / row tiles, us a
// single step of a cavity x * 90 * 80: fp32 x 65 25.1 / 22.0, 100 31.3 / 27.4,
// 250 75.2 / 58.2; fp16 100 22.1 / 22.1, 250 36.9 / 31.7; fp64 40 24.0 / 23.5,
// 131 74.4 / 62.6, 250 136 / 113 (30, half a tile: 20.8 / 22.0).
// k_cells: wavefront w of the grid takes the 64 cells 64 (w mod tpp) .. + 63
// (x fastest) of the z plane 1 + w / tpp, for packed rows and the rest.
// AHEAD: as any_cell (StepPlan::ahead).
// CACHED: the output policy, built in (a branch on it spilled registers).
template <class L, Mode M, bool CACHED, bool AHEAD = false>
__global__ void __launch_bounds__(256, (cells_min_blocks<L, M, false>())) k_cell_rows(StepArgs a, int tpr) {
    int x, y, z;
    if (row_tile_cell(a.L, tpr, a.rev, x, y, z)) any_cell<L, M, false, true, CACHED, false, true, AHEAD>(a, x, y, z);
}

template <class L, Mode M, bool FS = true, bool B32 = false, bool CACHED = false, bool AHEAD = false>
__global__ void __launch_bounds__(256, (cells_min_blocks<L, M, FS>())) k_cells(StepArgs a, int tpp, double rxl) {
    const int64_t w = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    int z = 1 + static_cast<int>(w / tpp);
    if (z > a.L.zl) return;
    if (a.rev) z = a.L.zl + 1 - z;
    const int64_t c = (w % tpp) * 64 + (threadIdx.x & 63);
    const int64_t xl = a.L.xl;
    if (c >= xl * a.L.yl) return;
    // row = c / xl: a double estimate is off by at most one, then corrected
    int64_t y = static_cast<int64_t>(static_cast<double>(c) * rxl);
    int64_t x = c - y * xl;
    if (x < 0) {
        --y;
        x += xl;
    } else if (x >= xl) {
        ++y;
        x -= xl;
    }
    any_cell<L, M, FS, B32, CACHED, false, false, AHEAD>(a, 1 + static_cast<int>(x), 1 + static_cast<int>(y), z);
}

// Near-boundary kernel: one thread per listed NEAR cell.
template <class L, Mode M>
__global__ void __launch_bounds__(128) k_near(StepArgs a) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= a.nb) return;
    const CellCoord c = a.blist[i];
    near_cell<L, M>(a, c.x, c.y, c.z);
}

}  // namespace lbm_amd
