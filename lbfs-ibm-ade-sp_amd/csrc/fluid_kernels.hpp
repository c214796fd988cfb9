// Device-side argument block and launchers of the fluid kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "lbfs_abi.h"
#include "tile_rec.hpp"

namespace lbfs {

struct FluidArgs {
    int n_cells, n_bc, n_tiles, max_tile_faces;
    int max_tile_cells;            // largest tile
    int max_grad_slots, max_slots; // largest tile plus its halo, plus its second halo (LDS of the fused step)
    int block_threads;             // workgroup size of the flux/update kernel (256 or 512)
    int lattice, flags;
    float rho0, inv_gamma, two_gamma, visc3_over_gamma, dt;
    float body_force[3];
    // per cell (internal tile order)
    const int *stencil;            // [6 n] SoA
    const float *gw;               // [18 n] SoA
    const float *inv_vol;          // [n]
    const float *visc_factor;      // [n] or null
    const float *cell_force;       // [3 n] or null (IBM force density)
    float4 *face_moments;          // [tile faces] or null: S0, S1 of each face (kept for the adjoint)
    float4 *grad_out;              // [3 n] or null: the fused pass also writes the gradients of its
                                   // tile's cells (kept for the adjoint, the layout of the gradient pass)
    // tiles: records, halo cell ids, boundary face ids, and the slot patterns
    // shared by tiles alike (DeviceLayout)
    const TileRec *tiles;
    const int *tile_cell_start;
    const int *halo_ids, *tile_bc;
    const uint32_t *face_gslot;    // owner slot | neighbour slot << 16
    const uint16_t *cell_slots, *cell_nbrs;
    const float *tile_w;           // 18 rows per tile: its gradient slots' weights W_k (the halo's are
                                   // copies, so each row is read as one run: gathered from gw, a halo
                                   // in x takes a cache line per cell and row)
    // tile faces: normal * area, dt (negative: general face) | owner offset, neighbour offset x |
    // neighbour offset yz
    const float4 *fA, *fB;
    const float2 *fC;
    // boundary conditions
    const int2 *bc_type;           // (rho type, vel type)
    const float4 *bc_val;          // (rho - rho0, u, v, w)
    // time stepping: 0 constant dt; LBFS_TS_LOCAL: dt_i = dt / (c.x + c.y / rho_i);
    // LBFS_TS_MIN: the minimum of those, reduced into *dt_min before the update
    int ts_mode;
    const float2 *cfl_coef;        // [n] or null
    unsigned int *dt_min;          // float bits of the global step (LBFS_TS_MIN)
};

// a.tile_w (set-up) from a.gw
hipError_t launch_tile_weights(const FluidArgs &a, float *tile_w, hipStream_t s);
hipError_t launch_gradients(const FluidArgs &a, const float4 *st, float4 *grad, hipStream_t s);
hipError_t launch_flux_update(const FluidArgs &a, const float4 *st, const float4 *grad, float4 *st_out,
                              float4 *res_out, int do_update, hipStream_t s);
// the whole fluid step in one pass per tile (gradients in LDS); equals
// launch_gradients + launch_flux_update bit for bit, gradients included when
// a.grad_out is set
hipError_t launch_fluid_fused(const FluidArgs &a, const float4 *st, float4 *st_out, float4 *res_out, int do_update,
                              hipStream_t s);
size_t fluid_fused_lds(const FluidArgs &a);
hipError_t launch_face_flux_all(const FluidArgs &a, const float4 *st, const float4 *grad, float4 *out, hipStream_t s);
// global minimum of the local steps into *a.dt_min (LBFS_TS_MIN)
hipError_t launch_dt_min(const FluidArgs &a, const float4 *st, hipStream_t s);
hipError_t launch_diag_partials(int n, float rho0, const float4 *st, const float4 *res, const float *force,
                                const float *inv_vol, double *part, hipStream_t s);

}  // namespace lbfs
