// C ABI of a domain's density and velocity fields (include/lbm_hip.h):
// lbm_moments and lbm_init_equilibrium, whose arrays of 32 bytes a cell pass
// between the host and the device in staged chunks.
#include <hip/hip_runtime.h>

#include <cstring>
#include <string>

#include "domain_impl.hpp"
#include "lbm_hip.h"
#include "staging.hpp"

using namespace lbm_amd;

namespace lbm_amd {
void staging_domain_created() { StagingPool::get().domain_created(); }
void staging_domain_destroyed() { StagingPool::get().domain_destroyed(); }
}  // namespace lbm_amd

extern "C" {

int lbm_init_equilibrium(lbm_domain* d, const double* rho, const double* u) {
    if (int rc = check_handle(d)) return rc;
    if (!d->finalized) return fail(LBM_ERR_STATE, "call lbm_finalize first (fluid cells are needed)");
    if (!rho || !u) return fail(LBM_ERR_ARG, "null input");
    const int64_t n = static_cast<int64_t>(d->L.xl) * d->L.yl * d->L.zl;
    // A restart: the next step pulls stored values from non-fluid cells, so
    // these go back to what a new domain holds. By now they may hold rule
    // values of an earlier state (in the in-place layout always; else where a
    // two-step pass or a reader of whole cells wrote them) or of lbm_set_pdf.
    if (d->nb || d->aa) {
        if (int rc = fill_initial(d, d->buf[d->cur])) return rc;
        d->aa_phase = 0;
    }
    const hipError_t e = staged_write(
        d->desc.device, d->stream, n, 4 * sizeof(double),
        [&](char* v, int64_t i0, int64_t m) {
            const size_t part = static_cast<size_t>(m) * sizeof(double);
            std::memcpy(v, rho + i0, part);
            std::memcpy(v + part, u + 3 * i0, 3 * part);
        },
        [&](void* slot, int64_t i0, int64_t m, hipStream_t s) {
            const double* v = static_cast<const double*>(slot);
            return d->ops->init_eq(d->L, d->buf[d->cur], d->d_kind, v, v + m, i0, m, s);
        });
    if (e != hipSuccess) return fail(LBM_ERR_HIP, std::string("init_equilibrium: ") + hipGetErrorString(e));
    d->materialised = true;
    return LBM_OK;
}

int lbm_moments(lbm_domain* d, double* rho, double* u) {
    if (int rc = check_handle(d)) return rc;
    if (int rc = aa_settle(d)) return rc;
    const int64_t n = static_cast<int64_t>(d->L.xl) * d->L.yl * d->L.zl;
    // only solid cells inside the box would show the boundary links' values
    if (d->n_fluid != static_cast<uint64_t>(n))
        if (int rc = materialise_boundaries(d)) return rc;
    const hipError_t e = staged_read(
        d->desc.device, d->stream, n, 4 * sizeof(double),
        [&](void* slot, int64_t i0, int64_t m, hipStream_t s) {
            double* v = static_cast<double*>(slot);
            return d->ops->moments(d->L, d->buf[d->cur], rho ? v : nullptr, u ? v + m : nullptr, i0, m, s);
        },
        [&](const char* v, int64_t i0, int64_t m) {
            const size_t part = static_cast<size_t>(m) * sizeof(double);
            if (rho) std::memcpy(rho + i0, v, part);
            if (u) std::memcpy(u + 3 * i0, v + part, 3 * part);
        });
    if (e != hipSuccess) return fail(LBM_ERR_HIP, std::string("moments: ") + hipGetErrorString(e));
    return LBM_OK;
}

}  // extern "C"
