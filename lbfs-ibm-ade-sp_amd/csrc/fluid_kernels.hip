// LBFS fluid kernels for gfx950 (FP32 working precision, density stored as
// rho - rho0).
//
//   k_gradients      per-cell least-squares gradients of (rho, u, v, w)
//                    (LBFS.cu:2177-2240, ghost rows of LBFS.cu:1933-2048 folded in)
//   k_flux_update    one workgroup per tile of cells: every face touching the
//                    tile is reconstructed once into LDS (LBFS.cu:2574-2810),
//                    then each cell gathers its six face fluxes in a fixed
//                    order and advances (LBFS.cu:2242-2281, 2089-2172).  No
//                    atomics: results are bitwise repeatable.
//
// Face reconstruction works on deviations from the rest state: with
// g_k = feq_k - w_k rho0, the interface density deviation and momentum are
// sum g_k and sum e_k g_k, and the flux of the interface equilibrium is taken
// from its closed-form moments (rho cs^2 I + rho u u / gamma), which the
// discrete sums of the reference reproduce exactly on these lattices.
#include <hip/hip_runtime.h>

#include <utility>

#include "fluid_device.hpp"
#include "fluid_kernels.hpp"
#include "lattice.hpp"

namespace lbfs {

#pragma clang fp contract(off)  // (fluid_device.hpp)

// ---------------------------------------------------------------------------
// gradients
// ---------------------------------------------------------------------------
// least-squares gradient of cell i (12 components: rho, u, v, w along x, y, z):
// the loads of its stencil (every index, then every neighbour state, a ghost
// entry loading the cell's own, and every weight, so they are in flight
// together rather than one index and one state at a time), then the sums
struct CellStencil {
    float4 si, sk[6];
    int jk[6];
    float wk[18];
};
__device__ __forceinline__ void load_stencil_ids(const FluidArgs &a, int i, CellStencil &c)
{
#pragma unroll
    for (int k = 0; k < 6; k++) c.jk[k] = a.stencil[(size_t)k * a.n_cells + i];
}
// (after the ids) cell i's weights are entry e of rows of length n
__device__ __forceinline__ void load_stencil(const float4 *__restrict__ st, int i, const float *__restrict__ w, int n,
                                             unsigned e, CellStencil &c)
{
    c.si = st[i];
#pragma unroll
    for (int k = 0; k < 6; k++) c.sk[k] = st[c.jk[k] >= 0 ? c.jk[k] : i];
#pragma unroll
    for (int k = 0; k < 18; k++) c.wk[k] = w[(size_t)k * n + e];
}
__device__ __forceinline__ void stencil_gradient(const FluidArgs &a, const CellStencil &c, float R[12])
{
    const float4 si = c.si;
#pragma unroll
    for (int t = 0; t < 12; t++) R[t] = 0.0f;
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int j = c.jk[k];
        float dr, du, dv, dw;
        if (j >= 0) {
            const float4 sj = c.sk[k];
            dr = sj.x - si.x; du = sj.y - si.y; dv = sj.z - si.z; dw = sj.w - si.w;
        } else {
            // ghost: Dirichlet mirror 2 bc - owner (velocity codes 1 and 3),
            // Neumann and empty copy (Solution.cpp:759-833, LBFS.cu:1843-1928)
            const int bc = -1 - j;
            const int2 ty = a.bc_type[bc];
            const float4 bv = a.bc_val[bc];
            const bool mv = ty.y == 1 || ty.y == 3;
            dr = ty.x == 1 ? 2.0f * (bv.x - si.x) : 0.0f;
            du = mv ? 2.0f * (bv.y - si.y) : 0.0f;
            dv = mv ? 2.0f * (bv.z - si.z) : 0.0f;
            dw = mv ? 2.0f * (bv.w - si.w) : 0.0f;
        }
        const float wx = c.wk[3 * k], wy = c.wk[3 * k + 1], wz = c.wk[3 * k + 2];
        const float d[4] = {dr, du, dv, dw};
#pragma unroll
        for (int v = 0; v < 4; v++) {
            R[3 * v] = fmaf(wx, d[v], R[3 * v]);
            R[3 * v + 1] = fmaf(wy, d[v], R[3 * v + 1]);
            R[3 * v + 2] = fmaf(wz, d[v], R[3 * v + 2]);
        }
    }
}
__device__ __forceinline__ void cell_gradient(const FluidArgs &a, const float4 *__restrict__ st, int i, float R[12])
{
    CellStencil c;
    load_stencil_ids(a, i, c);
    load_stencil(st, i, a.gw, a.n_cells, i, c);
    stencil_gradient(a, c, R);
}

__global__ __launch_bounds__(256) void k_gradients(FluidArgs a, const float4 *__restrict__ st,
                                                   float4 *__restrict__ grad)
{
    const int nblk = gridDim.x;
    const int b = xcd_remap(blockIdx.x, nblk);
    const int i = b * 256 + threadIdx.x;
    if (i >= a.n_cells) return;
    float R[12];
    cell_gradient(a, st, i, R);
    grad[3 * (size_t)i + 0] = make_float4(R[0], R[1], R[2], R[3]);
    grad[3 * (size_t)i + 1] = make_float4(R[4], R[5], R[6], R[7]);
    grad[3 * (size_t)i + 2] = make_float4(R[8], R[9], R[10], R[11]);
}

// Sources of the cell gradients a face reads: the gradient array of the
// two-pass step, or the fused step's tile (the gradients of the tile's cells
// and of the cells across its border in LDS, at the face's slots)
struct GlobalGrad {
    const float4 *__restrict__ grad;
    int o, n;  // owner and neighbour ids
    __device__ __forceinline__ void load_owner(float g[12]) const { load_grad(grad, o, g); }
    __device__ __forceinline__ void load_nbr(float g[12]) const { load_grad(grad, n, g); }
};
struct TileGrad {
    const float4 *lg;  // LDS: 3 float4 per gradient slot
    uint32_t slots;    // the face's owner slot | neighbour slot << 16
    __device__ __forceinline__ void load_owner(float g[12]) const { load_grad(lg, slots & 0xffffu, g); }
    __device__ __forceinline__ void load_nbr(float g[12]) const { load_grad(lg, slots >> 16, g); }
};

// ---------------------------------------------------------------------------
// face reconstruction and flux
// ---------------------------------------------------------------------------
// states and gradients extrapolated to an interior face from both sides, and
// their mean
__device__ __forceinline__ void interior_sides(const FaceRec &fr, const float4 &so, const float4 &sn,
                                               const float go[12], const float gn[12], float po[4], float pn[4],
                                               float p0[4])
{
    const float sov[4] = {so.x, so.y, so.z, so.w}, snv[4] = {sn.x, sn.y, sn.z, sn.w};
#pragma unroll
    for (int v = 0; v < 4; v++) {
        po[v] = sov[v] - dot3(fr.d1.x, fr.d1.y, fr.d1.z, go[3 * v], go[3 * v + 1], go[3 * v + 2]);
        pn[v] = snv[v] - dot3(fr.d2.x, fr.d2.y, fr.d2.z, gn[3 * v], gn[3 * v + 1], gn[3 * v + 2]);
        p0[v] = 0.5f * (po[v] + pn[v]);
    }
}

// equilibrium deviation of the rest point, which takes the mean state
template <class L>
__device__ __forceinline__ float rest_point(const float p0[4], float rho0, float ig)
{
    const float uu = dot3(p0[1], p0[2], p0[3], p0[1], p0[2], p0[3]);
    return L::w(0) * fmaf(rho0 + p0[0], -1.5f * ig * uu, p0[0]);
}

// The flux of tile-face tf from its record, the states of its owner (cell o)
// and neighbour (nb: cell id, or n_cells + boundary face, whose sn is unused)
// and their gradients
template <class L, bool BAND, class G>
__device__ __forceinline__ float4 face_flux(const FluidArgs &a, const G &gsrc, int tf, const FaceRaw &raw,
                                            const float4 &so, const float4 &sn, int o, int nb)
{
    static_assert(opposite_pairs<L>(), "lattice directions must come in opposite pairs after the rest point");
    const FaceRec fr = unpack_face(raw);
    const float3 fb = fr.d1;
    const float nx = fr.nx, ny = fr.ny, nz = fr.nz, A = fr.A, dt = fr.dt;
    const float rho0 = a.rho0, ig = a.inv_gamma;
    float go[12], gn[12];
    gsrc.load_owner(go);
    float po[4], pn[4], p0[4];
    FaceSums f;
    f.S1x = f.S1y = f.S1z = f.Tx = f.Ty = f.Tz = 0.0f;
    if (!fr.general) {
        gsrc.load_nbr(gn);
        interior_sides(fr, so, sn, go, gn, po, pn, p0);
        f.S0 = rest_point<L>(p0, rho0, ig);
        const float ig15 = 1.5f * ig;
        all_pairs_fast<L>(std::make_integer_sequence<int, (L::Q - 1) / 2>{}, f, po, pn, go, gn, nx, ny, nz, dt,
                          rho0 * ig15, ig15, a.two_gamma);
    } else {
        const bool ghost = nb >= a.n_cells;
        if (!ghost) {
            gsrc.load_nbr(gn);
            interior_sides(fr, so, sn, go, gn, po, pn, p0);
        } else {
            const float sov[4] = {so.x, so.y, so.z, so.w};
            // ghost gradient (gradients.cpp:393-505 / LBFS.cu:1933-2048) and face
            // value from the boundary condition (Solver.cpp:855-900)
            const int bc = nb - a.n_cells;
            const int2 ty = a.bc_type[bc];
            if (ty.y == LBFS_BC_EMPTY) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);  // Solver.cpp:308-310
            const float4 bv = a.bc_val[bc];
            const float bvv[4] = {bv.x, bv.y, bv.z, bv.w};
            const float d1n = sqrtf(dot3(fb.x, fb.y, fb.z, fb.x, fb.y, fb.z));
            const float inv_dmag = 2.0f / d1n;  // ghost centroid sits halfway to the face
            float dir[3];
            if (a.flags & LBFS_FLAG_GHOST_DIR_GPU) { dir[0] = -fb.x / d1n; dir[1] = -fb.y / d1n; dir[2] = -fb.z / d1n; }
            else { dir[0] = nx; dir[1] = ny; dir[2] = nz; }
            const float nv[3] = {nx, ny, nz};
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int type = v == 0 ? ty.x : ty.y;
                if (type == 1 || type == 3) {
                    const float dphi = 2.0f * (bvv[v] - sov[v]) * inv_dmag;
#pragma unroll
                    for (int c = 0; c < 3; c++) gn[3 * v + c] = dphi * dir[c];
                    // code 3 (parabolic/shear targets) extrapolates the face value
                    // with the ghost gradient (LBFS.cu:358-378)
                    p0[v] = type == 1 ? bvv[v]
                                      : sov[v] - dot3(fb.x, fb.y, fb.z, gn[3 * v], gn[3 * v + 1], gn[3 * v + 2]);
                } else {
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        const float fac = (a.flags & LBFS_FLAG_NEUMANN_SIGNED) ? 1.0f - nv[c] : 1.0f - fabsf(nv[c]);
                        gn[3 * v + c] = go[3 * v + c] * fac;
                    }
                    p0[v] = sov[v] - dot3(fb.x, fb.y, fb.z, gn[3 * v], gn[3 * v + 1], gn[3 * v + 2]);
                }
                po[v] = p0[v];
                pn[v] = p0[v];
            }
            // the GPU reconstruction hands the ghost gradient to the owner-side
            // points too (grad_*_1 = grad_*_2, LBFS.cu:391-394)
            if (a.flags & LBFS_FLAG_GHOST_FACE_GRAD) {
#pragma unroll
                for (int t = 0; t < 12; t++) go[t] = gn[t];
            }
        }
#pragma unroll
        for (int t = 0; t < 12; t++) { go[t] *= dt; gn[t] *= dt; }
        f.S0 = rest_point<L>(p0, rho0, ig);
        all_pairs<L, BAND>(std::make_integer_sequence<int, (L::Q - 1) / 2>{}, f, po, pn, p0, go, gn, nx, ny, nz,
                           0.001f * dt, ghost, rho0, ig);
    }
    const float S0 = f.S0, S1x = f.S1x, S1y = f.S1y, S1z = f.S1z, Tx = f.Tx, Ty = f.Ty, Tz = f.Tz;
    if (a.face_moments) a.face_moments[tf] = make_float4(S0, S1x, S1y, S1z);
    const float rho_f = rho0 + S0;
    const float mn = dot3(S1x, S1y, S1z, nx, ny, nz);
    const float vf = a.visc_factor ? a.visc_factor[o] : 1.0f;
    const float tau = a.visc3_over_gamma * vf * __builtin_amdgcn_rcpf(dt);
    const float c1 = 1.0f - tau;
    const float third = S0 * (1.0f / 3.0f);
    const float q = mn * __builtin_amdgcn_rcpf(rho_f) * ig;
    float4 r;
    r.x = mn * A;
    r.y = A * fmaf(c1, fmaf(S1x, q, third * nx), tau * Tx);
    r.z = A * fmaf(c1, fmaf(S1y, q, third * ny), tau * Ty);
    // a planar lattice carries no z momentum flux (its sum e_z e_z w is zero)
    r.w = L::dims == 3 ? A * fmaf(c1, fmaf(S1z, q, third * nz), tau * Tz) : 0.0f;
    return r;
}

// the cell update of a tile from its face fluxes in LDS: each cell gathers
// its six signed face slots in a fixed order (LBFS.cu:2242-2281), adds the
// force density and advances (LBFS.cu:2089-2172)
template <int NT>
__device__ __forceinline__ void tile_update(const FluidArgs &a, const float4 *lds_flux, const TileRec &T,
                                            const float4 *__restrict__ st, float4 *__restrict__ st_out,
                                            float4 *__restrict__ res_out, int do_update)
{
    for (int q = threadIdx.x; q < T.nc; q += NT) {
        const int i = T.c0 + q;
        const uint32_t *sl = reinterpret_cast<const uint32_t *>(a.cell_slots) + 3 * (size_t)(T.pc + q);
        const uint32_t s01 = sl[0], s23 = sl[1], s45 = sl[2];
        // the cell's state and force loaded with its slots, not after the sums
        const float4 s0 = do_update ? st[i] : float4{};
        float cfv[3] = {0.0f, 0.0f, 0.0f};
        if (do_update && a.cell_force) {
            const float *cf = a.cell_force + 3 * (size_t)i;
            cfv[0] = cf[0]; cfv[1] = cf[1]; cfv[2] = cf[2];
        }
        const uint32_t s[6] = {s01 & 0xffffu, s01 >> 16, s23 & 0xffffu, s23 >> 16, s45 & 0xffffu, s45 >> 16};
        float r0 = 0.0f, r1 = 0.0f, r2 = 0.0f, r3 = 0.0f;
#pragma unroll
        for (int k = 0; k < 6; k++) {
            const float4 fl = lds_flux[s[k] & 0x7fffu];
            const float sg = (s[k] & 0x8000u) ? -1.0f : 1.0f;
            r0 = fmaf(sg, fl.x, r0); r1 = fmaf(sg, fl.y, r1); r2 = fmaf(sg, fl.z, r2); r3 = fmaf(sg, fl.w, r3);
        }
        const float iv = a.inv_vol[i];
        if (res_out) res_out[i] = make_float4(r0 * iv, r1 * iv, r2 * iv, r3 * iv);
        if (!do_update) continue;
        float fx = a.body_force[0], fy = a.body_force[1], fz = a.body_force[2];
        if (a.cell_force) {
            fx += cfv[0]; fy += cfv[1]; fz += cfv[2];
        }
        r0 *= iv; r1 = fmaf(r1, iv, fx); r2 = fmaf(r2, iv, fy); r3 = fmaf(r3, iv, fz);
        float dt = a.dt;
        if (a.ts_mode == LBFS_TS_LOCAL) {
            const float2 c = a.cfl_coef[i];
            dt = a.dt / (c.x + c.y / (a.rho0 + s0.x));
        } else if (a.ts_mode == LBFS_TS_MIN) {
            dt = __uint_as_float(*a.dt_min);
        }
        const float drho = fmaf(dt, r0, s0.x);
        const float rho = a.rho0 + drho;
        const float inv_rho = 1.0f / rho;
        float4 sn;
        sn.x = drho;
        sn.y = fmaf(dt * fmaf(-s0.y, r0, r1), inv_rho, s0.y);
        sn.z = fmaf(dt * fmaf(-s0.z, r0, r2), inv_rho, s0.z);
        sn.w = fmaf(dt * fmaf(-s0.w, r0, r3), inv_rho, s0.w);
        st_out[i] = sn;
    }
}

// face q of tile T from the gradient array
template <class L, bool BAND>
__device__ __forceinline__ float4 tile_face_flux(const FluidArgs &a, const float4 *__restrict__ st,
                                                 const float4 *__restrict__ grad, const TileRec &T, int q)
{
    const uint32_t gs = a.face_gslot[T.pf + q];
    const int o = slot_cell(a, T, gs & 0xffffu), nb = face_neighbour(a, T, gs, q);
    const int n = q < T.nif ? nb : o;  // (a boundary face loads its owner's, unused)
    return face_flux<L, BAND>(a, GlobalGrad{grad, o, n}, T.f0 + q, load_face_raw(a, T.f0 + q), st[o], st[n], o, nb);
}

// two-pass step, second pass: the tile's faces from the gradient array
template <class L, bool BAND, int NT>
__global__ __launch_bounds__(NT) void k_flux_update(FluidArgs a, const float4 *__restrict__ st,
                                                     const float4 *__restrict__ grad, float4 *__restrict__ st_out,
                                                     float4 *__restrict__ res_out, int do_update)
{
    extern __shared__ float4 lds_flux[];
    const TileRec T = a.tiles[xcd_remap(blockIdx.x, gridDim.x)];
    for (int q = threadIdx.x; q < T.nf; q += NT)
        lds_flux[q] = tile_face_flux<L, BAND>(a, st, grad, T, q);
    __syncthreads();
    tile_update<NT>(a, lds_flux, T, st, st_out, res_out, do_update);
}

// Fused step, one workgroup per tile: the gradients of the tile's cells and
// of the cells across its border that its faces reach into LDS (the same
// arithmetic as the gradient pass), the tile's faces from them, then the cell
// update.  Results equal the two-pass step bit for bit; the gradient array is
// not read, and written (the tile's own cells) only when a.grad_out is set.
//
// Bound by memory: at 256x128x128 the same loads without the face arithmetic
// take 0.97 of its time, 335 us for the 330 B a cell it moves (4.1 TB/s; a
// device copy on the same card 5.1).  What it reads is laid out for it: cells
// by slots of shared patterns rather than ids (faces 40 B, no stencil), the
// weights of a tile and its halo as whole rows, each thread's next face on its
// way while the present one is reconstructed.  D3Q19, 8x8x8 tiles, with face
// ids, stencil ids and gathered weights before: 128x64x64 42.9 -> 38.3 us,
// 256x128x128 428 -> 335 us.
template <class L, bool BAND, int NT>
__global__ __launch_bounds__(NT) void k_fluid_fused(FluidArgs a, const float4 *__restrict__ st,
                                                     float4 *__restrict__ st_out, float4 *__restrict__ res_out,
                                                     int do_update)
{
    extern __shared__ float4 lds[];
    float4 *lg = lds;                                        // 3 per gradient slot
    float4 *lds_flux = lg + 3 * (size_t)a.max_grad_slots;    // 1 per face
    int *ids = reinterpret_cast<int *>(lds_flux + a.max_tile_faces);  // cell id of each slot
    const TileRec T = a.tiles[xcd_remap(blockIdx.x, gridDim.x)];
    const int ns = T.nc + T.nh;
    for (int q = threadIdx.x; q < ns + T.n2; q += NT) ids[q] = q < T.nc ? T.c0 + q : a.halo_ids[T.h0 + q - T.nc];
    // the first face's record and slots are on their way while the gradients
    // are computed (here and below a thread past the end loads the last one's)
    int q = threadIdx.x;
    const int ql = T.nf - 1;
    FaceRaw raw = load_face_raw(a, T.f0 + min(q, ql));
    uint32_t gs = a.face_gslot[T.pf + min(q, ql)], gs1 = a.face_gslot[T.pf + min(q + NT, ql)];
    __syncthreads();
    for (int p = threadIdx.x; p < ns; p += NT) {
        const int i = ids[p];
        const uint32_t *nl = reinterpret_cast<const uint32_t *>(a.cell_nbrs) + 3 * (size_t)(T.pn + p);
        const uint32_t n01 = nl[0], n23 = nl[1], n45 = nl[2];
        const uint32_t nb[6] = {n01 & 0xffffu, n01 >> 16, n23 & 0xffffu, n23 >> 16, n45 & 0xffffu, n45 >> 16};
        CellStencil c;
#pragma unroll
        for (int k = 0; k < 6; k++)
            c.jk[k] = nb[k] & 0x8000u ? -1 - a.tile_bc[T.b0 + (nb[k] & 0x7fffu)] : ids[nb[k]];
        float R[12];
        load_stencil(st, i, a.tile_w + 18 * (size_t)T.s0, ns, p, c);
        stencil_gradient(a, c, R);
        float4 *o = lg + 3 * p;
        o[0] = make_float4(R[0], R[1], R[2], R[3]);
        o[1] = make_float4(R[4], R[5], R[6], R[7]);
        o[2] = make_float4(R[8], R[9], R[10], R[11]);
        if (a.grad_out && p < T.nc) {
            float4 *g = a.grad_out + 3 * (size_t)i;
            g[0] = o[0];
            g[1] = o[1];
            g[2] = o[2];
        }
    }
    // a boundary face's neighbour slot is 0xffff: it loads the last gradient slot's
    // state, unused
    const int last = ns - 1;
    float4 so = st[ids[gs & 0xffffu]], sn = st[ids[min((int)(gs >> 16), last)]];
    __syncthreads();
    while (q < T.nf) {
        // the next face's record and states, and the slots of the one after,
        // load while this one is reconstructed
        const FaceRaw raw1 = load_face_raw(a, T.f0 + min(q + NT, ql));
        const float4 so1 = st[ids[gs1 & 0xffffu]], sn1 = st[ids[min((int)(gs1 >> 16), last)]];
        const uint32_t gs2 = a.face_gslot[T.pf + min(q + 2 * NT, ql)];
        const int o = ids[gs & 0xffffu];
        const int nb = q < T.nif ? 0 : a.n_cells + a.tile_bc[T.b0 + q - T.nif];
        lds_flux[q] = face_flux<L, BAND>(a, TileGrad{lg, gs}, T.f0 + q, raw, so, sn, o, nb);
        raw = raw1;
        so = so1;
        sn = sn1;
        gs = gs1;
        gs1 = gs2;
        q += NT;
    }
    __syncthreads();
    tile_update<NT>(a, lds_flux, T, st, st_out, res_out, do_update);
}

// every tile-face's flux (one workgroup per tile)
template <class L, bool BAND>
__global__ __launch_bounds__(256) void k_face_flux_all(FluidArgs a, const float4 *__restrict__ st,
                                                       const float4 *__restrict__ grad, float4 *__restrict__ out)
{
    const TileRec T = a.tiles[blockIdx.x];
    for (int q = threadIdx.x; q < T.nf; q += 256) out[T.f0 + q] = tile_face_flux<L, BAND>(a, st, grad, T, q);
}

// ---------------------------------------------------------------------------
// global minimum of the local time steps (min<128> + min_block,
// Solver_gpu.cu:773-776): positive floats order like their bit patterns, so an
// unsigned atomic minimum is exact and independent of the visiting order
// ---------------------------------------------------------------------------
__global__ void k_dt_reset(unsigned int *dt_min) { *dt_min = 0x7f800000u; }

__global__ __launch_bounds__(256) void k_dt_min(FluidArgs a, const float4 *__restrict__ st)
{
    __shared__ float sh[256];
    const int i = blockIdx.x * 256 + threadIdx.x;
    float v = INFINITY;
    if (i < a.n_cells) {
        const float2 c = a.cfl_coef[i];
        v = a.dt / (c.x + c.y / (a.rho0 + st[i].x));
    }
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int stp = 128; stp > 0; stp >>= 1) {
        if ((int)threadIdx.x < stp) sh[threadIdx.x] = fminf(sh[threadIdx.x], sh[threadIdx.x + stp]);
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicMin(a.dt_min, __float_as_uint(sh[0]));
}

// ---------------------------------------------------------------------------
// FP64 diagnostics: per-block partial sums (fixed order), summed on the host
// ---------------------------------------------------------------------------
// (force: the momentum force density added to the residual, 3 per cell, as
// the reference adds force_x/y/z before squaring, Solver_gpu.cu:1008-1046)
__global__ __launch_bounds__(256) void k_diag_partials(int n, float rho0, const float4 *__restrict__ st,
                                                       const float4 *__restrict__ res, const float *__restrict__ force,
                                                       const float *__restrict__ inv_vol, double *__restrict__ part)
{
    __shared__ double sh[6][256];
    const int i = blockIdx.x * 256 + threadIdx.x;
    double v[6] = {0, 0, 0, 0, 0, 0};
    if (i < n) {
        const float4 s = st[i];
        const float4 r = res[i];
        double r1 = r.y, r2 = r.z, r3 = r.w;
        if (force) {
            r1 += (double)force[3 * (size_t)i];
            r2 += (double)force[3 * (size_t)i + 1];
            r3 += (double)force[3 * (size_t)i + 2];
        }
        v[0] = (double)r.x * r.x;
        v[1] = r1 * r1;
        v[2] = r2 * r2;
        v[3] = r3 * r3;
        v[4] = ((double)rho0 + (double)s.x) / (double)inv_vol[i];
        const double sp = sqrt((double)s.y * s.y + (double)s.z * s.z + (double)s.w * s.w);
        v[5] = (isfinite(s.x) && isfinite(s.y) && isfinite(s.z) && isfinite(s.w)) ? sp : INFINITY;
    }
    for (int t = 0; t < 6; t++) sh[t][threadIdx.x] = v[t];
    __syncthreads();
    for (int stp = 128; stp > 0; stp >>= 1) {
        if ((int)threadIdx.x < stp) {
            for (int t = 0; t < 5; t++) sh[t][threadIdx.x] += sh[t][threadIdx.x + stp];
            sh[5][threadIdx.x] = fmax(sh[5][threadIdx.x], sh[5][threadIdx.x + stp]);
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[6 * (size_t)blockIdx.x + threadIdx.x] = sh[threadIdx.x][0];
}

// the weight rows of each tile's gradient slots from the cells' (set-up)
__global__ __launch_bounds__(256) void k_tile_weights(FluidArgs a, float *__restrict__ tw)
{
    const TileRec T = a.tiles[blockIdx.x];
    const int ns = T.nc + T.nh;
    float *w = tw + 18 * (size_t)T.s0;
    for (int p = threadIdx.x; p < ns; p += 256) {
        const int i = slot_cell(a, T, p);
        for (int r = 0; r < 18; r++) w[(size_t)r * ns + p] = a.gw[(size_t)r * a.n_cells + i];
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_tile_weights(const FluidArgs &a, float *tile_w, hipStream_t s)
{
    hipLaunchKernelGGL(k_tile_weights, dim3(a.n_tiles), dim3(256), 0, s, a, tile_w);
    return hipGetLastError();
}

hipError_t launch_gradients(const FluidArgs &a, const float4 *st, float4 *grad, hipStream_t s)
{
    const int blocks = (a.n_cells + 255) / 256;
    hipLaunchKernelGGL(k_gradients, dim3(blocks), dim3(256), 0, s, a, st, grad);
    return hipGetLastError();
}

// instantiate a kernel template for the context's lattice and tie-band mode
template <template <class, bool> class K, class... Args>
static hipError_t dispatch(const FluidArgs &a, dim3 grid, size_t lds, hipStream_t s, Args... args)
{
    const bool band = (a.flags & LBFS_FLAG_UPWIND_BAND) != 0;
    switch (a.lattice * 2 + (band ? 1 : 0)) {
    case 0: K<D3Q15, false>::launch(grid, lds, s, a, args...); break;
    case 1: K<D3Q15, true>::launch(grid, lds, s, a, args...); break;
    case 2: K<D3Q19, false>::launch(grid, lds, s, a, args...); break;
    case 3: K<D3Q19, true>::launch(grid, lds, s, a, args...); break;
    case 4: K<D2Q9, false>::launch(grid, lds, s, a, args...); break;
    case 5: K<D2Q9, true>::launch(grid, lds, s, a, args...); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <class L, bool BAND>
struct FluxUpdate {
    static void launch(dim3 g, size_t lds, hipStream_t s, const FluidArgs &a, const float4 *st, const float4 *grad,
                       float4 *st_out, float4 *res_out, int do_update)
    {
        if (a.block_threads == 576)
            hipLaunchKernelGGL((k_flux_update<L, BAND, 576>), g, dim3(576), lds, s, a, st, grad, st_out, res_out, do_update);
        else if (a.block_threads == 512)
            hipLaunchKernelGGL((k_flux_update<L, BAND, 512>), g, dim3(512), lds, s, a, st, grad, st_out, res_out, do_update);
        else
            hipLaunchKernelGGL((k_flux_update<L, BAND, 256>), g, dim3(256), lds, s, a, st, grad, st_out, res_out, do_update);
    }
};

template <class L, bool BAND>
struct FaceFluxAll {
    static void launch(dim3 g, size_t lds, hipStream_t s, const FluidArgs &a, const float4 *st, const float4 *grad,
                       float4 *out)
    {
        hipLaunchKernelGGL((k_face_flux_all<L, BAND>), g, dim3(256), lds, s, a, st, grad, out);
    }
};

hipError_t launch_flux_update(const FluidArgs &a, const float4 *st, const float4 *grad, float4 *st_out,
                              float4 *res_out, int do_update, hipStream_t s)
{
    const size_t lds = sizeof(float4) * (size_t)a.max_tile_faces;
    return dispatch<FluxUpdate>(a, dim3(a.n_tiles), lds, s, st, grad, st_out, res_out, do_update);
}

template <class L, bool BAND>
struct FluidFused {
    static void launch(dim3 g, size_t lds, hipStream_t s, const FluidArgs &a, const float4 *st, float4 *st_out,
                       float4 *res_out, int do_update)
    {
        if (a.block_threads == 576)
            hipLaunchKernelGGL((k_fluid_fused<L, BAND, 576>), g, dim3(576), lds, s, a, st, st_out, res_out, do_update);
        else if (a.block_threads == 512)
            hipLaunchKernelGGL((k_fluid_fused<L, BAND, 512>), g, dim3(512), lds, s, a, st, st_out, res_out, do_update);
        else
            hipLaunchKernelGGL((k_fluid_fused<L, BAND, 256>), g, dim3(256), lds, s, a, st, st_out, res_out, do_update);
    }
};

size_t fluid_fused_lds(const FluidArgs &a)
{
    return sizeof(float4) * (3 * (size_t)a.max_grad_slots + (size_t)a.max_tile_faces) + sizeof(int) * a.max_slots;
}

hipError_t launch_fluid_fused(const FluidArgs &a, const float4 *st, float4 *st_out, float4 *res_out, int do_update,
                              hipStream_t s)
{
    return dispatch<FluidFused>(a, dim3(a.n_tiles), fluid_fused_lds(a), s, st, st_out, res_out, do_update);
}

hipError_t launch_face_flux_all(const FluidArgs &a, const float4 *st, const float4 *grad, float4 *out, hipStream_t s)
{
    return dispatch<FaceFluxAll>(a, dim3(a.n_tiles), 0, s, st, grad, out);
}

hipError_t launch_dt_min(const FluidArgs &a, const float4 *st, hipStream_t s)
{
    hipLaunchKernelGGL(k_dt_reset, dim3(1), dim3(1), 0, s, a.dt_min);
    hipLaunchKernelGGL(k_dt_min, dim3((a.n_cells + 255) / 256), dim3(256), 0, s, a, st);
    return hipGetLastError();
}

hipError_t launch_diag_partials(int n, float rho0, const float4 *st, const float4 *res, const float *force,
                                const float *inv_vol, double *part,
                                hipStream_t s)
{
    const int blocks = (n + 255) / 256;
    hipLaunchKernelGGL(k_diag_partials, dim3(blocks), dim3(256), 0, s, n, rho0, st, res, force, inv_vol, part);
    return hipGetLastError();
}

}  // namespace lbfs
