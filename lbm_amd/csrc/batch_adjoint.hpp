// Batched adjoint over the domains of a batch (D3Q19, F32 / F64S).
//
// Every domain owns one device chunk of field-sized slots: checkpoints of the
// forward run, the recomputed states of the current segment and two adjoint
// (mu) buffers. The kernels walk the batch's 64-cell tiles; a launch names
// its slots by index, the same for every domain, so one launch advances all
// domains by one recompute or one adjoint step. The per-cell arithmetic is
// the single-domain code (any_cell forward, adj_cell backward).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "batch.hpp"
#include "domain_view.hpp"
#include "storage.hpp"

namespace lbm_amd {

struct BatchAdjView {
    FieldLayout L;
    void* chunk;          // slots of slot_elems storage elements each
    int64_t slot_elems;   // Q * plane
    const void* gfinal;   // the forward run's final field (the domain's buffer)
    const uint8_t* kind;
    const uint32_t* lmask;
    const uint8_t* lcond;
    const uint32_t* rword;
    int span32;           // StepArgs::span32
    const Cond* conds;
    double tau, omega;
    const int* near_idx;  // per element: index of a NEAR cell in the domain's list
    int64_t nb;           // NEAR cells
    double* gw;           // 3 doubles per NEAR cell: dJ/du_wall accumulated per cell
    // Recorded runs: the domain's two buffers, and per step hist_stride Calc
    // values: drho and u of every interior cell, then 1 + the own sum of every
    // NEAR cell.
    void* buf[2];
    void* hist;
    int64_t hist_stride;
    int tpp;              // 64-cell tiles per z plane
    double rxl;           // 1 / xl
};

struct BatchAdjArgs {
    const BatchAdjView* views;
    const TileRef* tiles;  // cell tiles: local = i + tpp * (z - 1)
    int64_t ntiles;
    int src_slot, dst_slot;                  // recompute step
    int gprev_slot, mu_in_slot, mu_out_slot; // adjoint step
    int64_t hist_step;                       // recorded step (1 .. T) of hist_forward and hist_backward
    int parity;                              // hist_forward: buf[parity] -> buf[parity ^ 1]
    int* status;                             // hist_forward: non-finite flags as BatchArgs::status
    int terminal;
    int materialised;
    int rev;     // hist_*: walk the tiles from the last to the first (StepArgs::rev)
    int cached;  // StepArgs::cached, for what one launch reads and writes of all domains
    int idx32;  // every domain's plane is under 4 GiB (32-bit byte offsets)
    int nxcd;   // L2 domains the launch's blocks are dealt to (tile_walk)
};

struct BatchAdjOps {
    hipError_t (*recompute)(const BatchAdjArgs& a, int grid, hipStream_t s);
    hipError_t (*backward)(const BatchAdjArgs& a, int grid, hipStream_t s);
    // one forward step of every domain that records, one adjoint step from the record
    hipError_t (*hist_forward)(const BatchAdjArgs& a, int grid, hipStream_t s);
    hipError_t (*hist_backward)(const BatchAdjArgs& a, int grid, hipStream_t s);
    // near_idx[element of list entry i] = i
    hipError_t (*near_index)(const FieldLayout& Ly, const CellCoord* blist, int64_t nb, int* near_idx, hipStream_t s);
    // out[3 d + k] = sum over the NEAR cells of domain d of gw (fixed order)
    hipError_t (*reduce)(const BatchAdjView* views, int ndom, double* out, hipStream_t s);
};

const BatchAdjOps* batch_adj_ops(int q, Mode m);

}  // namespace lbm_amd
