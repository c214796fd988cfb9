// Host transfers of per-cell and per-node arrays: kernels convert between the
// device's float4 records in tile order and the caller's doubles in its own
// order, straight into (out of) pinned staging, and a few host threads move the
// staged chunk while the next one is under way.
#pragma once

#include <hip/hip_runtime.h>

struct lbfs_ctx;

namespace lbfs {

// the caller's doubles of n records of four: four arrays, or one array of
// records (aos)
struct CellArrays {
    double *soa[4];
    double *aos;
};

// pinned staging of one context, allocated at first use (at most 16 MiB)
struct Staging {
    double *buf[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
    size_t bytes = 0;
    void release();
};

// records of every cell, in caller order, with add0 added to the first
// component; both wait for the context's stream
int read_cells(lbfs_ctx *ctx, const float4 *src, double add0, const CellArrays &out);
// dst = the caller's records (aos), rounded to float, in tile order
int write_cells(lbfs_ctx *ctx, const double *src, float4 *dst);
// positions (absolute), velocities and forces of the membrane nodes, 3 per
// node; any may be null
int read_nodes(lbfs_ctx *ctx, double *X, double *U, double *F);

}  // namespace lbfs
