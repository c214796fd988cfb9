// The opaque context behind the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <functional>
#include <string>
#include <vector>

#include "coupling.hpp"
#include "fixed_point.hpp"
#include "fluid_kernels.hpp"
#include "lbfs_abi.h"
#include "mesh_host.hpp"
#include "transfer.hpp"

namespace lbfs {
struct AdjointState;  // adjoint.cpp
void adjoint_release(lbfs_ctx *ctx);
}  // namespace lbfs

// Coupled meshes up to this many cells run a step's kernels in order on one
// stream: the waits across streams cost a step 17 us in a graph, more than the
// overlap gains there.  One stream against two, a cell of 642 nodes: 9600 cells
// 38.6 and 47.4 us a step, 41k 38.9 and 44.7, 77k 40.1 and 43.7, 147k 47.5 and
// 46.4, 251k 55.5 and 50.2; of 2562 nodes 73 and 83, 58 and 65, 53 and 58, 59 and
// 60, 71 and 66; suspensions of 0.2 nodes a cell 32k 78.6 and 85.5, 58k 99.6 and
// 101.7, 123k 107.3 and 108.2, of 0.025 34.7 and 40.8, 39.3 and 42.8, 51.6 and 54.3.
constexpr int ONE_STREAM_CELLS = 128 * 1024;

struct lbfs_ctx {
    std::string err;
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t side = nullptr;       // second stream: the coupling chain beside the fluid passes (or the reverse)
    hipStream_t side2 = nullptr;      // third stream: membrane forces (step schedule 2)
    hipEvent_t ev_fork = nullptr, ev_join = nullptr, ev_fork2 = nullptr, ev_join2 = nullptr;
    lbfs_params params{};
    std::vector<lbfs::HostBlock> blocks;   // logical boxes of the mesh (empty: none)

    lbfs::Geometry geo;
    lbfs::DeviceLayout lay;
    lbfs::FluidArgs args{};
    std::vector<int> bc_vel_type;   // caller velocity BC type per boundary face

    float4 *st[2] = {nullptr, nullptr};
    int cur = 0;
    float4 *grad = nullptr, *res = nullptr, *face_scratch = nullptr;
    double *diag_part = nullptr;
    int *dev_err = nullptr;         // device error word: ERR_FIX_* bits (fixed_point.hpp), sticky until
                                    // the next lbfs_add_membranes
    float *static_force = nullptr;  // [3 n] body force + closure term
    float *cell_force = nullptr;    // [3 n] static force + spread IBM force
    int *cell_inv = nullptr;        // [n] internal id of each caller cell
    lbfs::Staging staging;          // pinned buffers of the host transfers
    std::vector<void *> allocs;
    float *tile_w = nullptr;        // weight rows of the fused pass (FluidArgs::tile_w)
    // Device memory; where it is short, the fused pass's weight rows (126 B a cell
    // with 8x8x8 tiles) are given back and the steps run the two passes, which need
    // none of them and give the same bits.
    hipError_t device_alloc(void **p, size_t bytes);
    void release_tile_weights();

    // membranes and IBM coupling (lbfs_add_membranes)
    bool have_membranes = false;
    lbfs::MemArgs mem{};
    lbfs::IbmArgs ibm{};
    std::vector<int> mem_node_start;
    double *mem_energy = nullptr;   // [7 n_mem] output of lbfs_get_membrane_energies
    double *energy_scratch = nullptr; // this device's static staging of lbfs_get_membrane_energies_noalloc
    int ibm_binned_option = -1;     // LBFS_OPT_IBM_BINNED: -1 by node density, else IBM_SPREAD_*
    // host copies behind lbfs_set_membrane_moduli: per-membrane parameters,
    // per-edge spring constant per unit shear modulus (FP64), edge ranges
    std::vector<lbfs::MemParamDev> mem_params;
    std::vector<float4> mem_edge_const;
    std::vector<double> mem_ks_unit;
    std::vector<int> mem_edge_start;
    std::vector<double> mem_shear;
    std::vector<void *> coupling_allocs;
    float *visc_factor = nullptr;   // [n] internal viscosity field, null while every ratio is 1
    lbfs::ViscGrid visc_grid{};     // its search structure (allocated with it)
    int visc_search = 1;            // LBFS_OPT_VISC_SEARCH
    float delta_h = 0.1f;           // smoothing width of the field (unstructured_mesh.cpp:263-264)
    long long t_step = 0;           // steps since the membranes were attached

    // checkpoints and buffers of the discrete adjoint (lbfs_adjoint_*)
    lbfs::AdjointState *adj = nullptr;

    // hipGraphs of graph_steps(k) consecutive steps (even numbers) starting from
    // cur == 0.  A graph launch costs the host 16 us and the device a gap of 3-5
    // us however many steps it holds: per step of 64x64 cells 8.0 us in graphs of
    // two, 5.7 of 8, 5.2 of 32, and 5.9 launched one by one; of 128x64x64 40.6,
    // 39.1 and 38.9, with its cell (six launches on two streams) 62.6, 61.8 and
    // 61.8.  Capturing the long graph costs as much as it saves over some 200 to
    // 600 steps, so a solver takes it from its LONG_GRAPH_AFTER-th step on.
    static constexpr long long LONG_GRAPH_AFTER = 256;
    long long steps_enqueued = 0;   // steps of enqueue_steps so far
    int graph_steps(int k) const { return k == 1 ? 2 : (have_membranes ? 8 : 32); }
    int schedule_option = 0;        // LBFS_OPT_STEP_SCHEDULE
    bool fused_ok = false;          // the tiles fit the fused fluid pass's LDS, and its weight rows memory
    bool fused = false;             // LBFS_OPT_FUSED_FLUID: whole steps run the fused fluid pass
    bool use_graph = true;
    hipGraphExec_t graph_exec[2] = {nullptr, nullptr};
    void drop_graph();
    // arguments of the apply pass that ends a coupled step
    lbfs::ApplyArgs apply_args(float4 *st_new, float *cell_force_out, int all) const
    {
        lbfs::ApplyArgs p{};
        p.tile_cell_start = args.tile_cell_start;
        p.n_tiles = lay.n_tiles;
        p.dt = args.dt;
        p.rho0 = args.rho0;
        p.st = st_new;
        p.cell_force_out = cell_force_out;
        p.all = all;
        p.mem_acc = mem.mem_acc;
        p.glob = mem.glob;
        p.n_mem = mem.n_mem;
        return p;
    }

    // lbfs_step_residual: the face pass of an eager step also writes the flux
    // residual (never set while a graph is captured)
    bool res_track = false;
    float4 *res_out() const { return res_track ? res : nullptr; }

    int fail(int code, const char *fmt, ...);
    // waits for the stream and turns a set device error word into LBFS_E_NONFINITE
    int check_device_error();
    int enqueue_step();
    int enqueue_steps(int nsteps);
    void release_extensions();

    // The step as an ordered list of kernel stages (each enqueues one launch
    // on `stream`), with the modelled device bytes of that launch.
    struct Stage {
        const char *name;
        std::function<int()> run;
        double model_bytes;
    };
    // fused: the fluid passes as the one fused launch "fluid"; otherwise
    // "gradients" and "flux_update".  one_force_pass: the membrane forces as the
    // one launch "mem_forces" where the step takes it; otherwise "mem_volume",
    // "mem_edges" and "mem_nodes".  (The stage API splits both; whole steps and
    // their timing take the step's own launches.)
    std::vector<Stage> step_stages(bool with_visc = false, bool fused = false, bool one_force_pass = false);
    // the internal viscosity field is rebuilt at t = 1 (mod 10000) (Solver_gpu.cu:884-889)
    bool visc_due(long long t) const { return visc_factor && (t % 10000) == 1; }
    int run_stages(bool with_visc);
};
