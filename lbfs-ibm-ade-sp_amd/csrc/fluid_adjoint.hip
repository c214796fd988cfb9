// Adjoint (reverse-mode derivative) of the fluid step, hand-written for gfx950.
//
//   k_adj_update  per cell: adjoint of the forward-Euler update
//                 (LBFS.cu:2089-2172) with respect to the state, the cell
//                 residual and the cell force
//   k_adj_flux    one workgroup per tile of cells, as the forward flux pass:
//                 the transpose of each face's reconstruction + equilibrium +
//                 flux (LBFS.cu:2574-2810) is evaluated in chunks of faces
//                 staged in LDS, then every cell gathers its own side of its
//                 six faces (state and gradient adjoints) in a fixed order
//   k_adj_grad    per cell: transpose of the least-squares gradients
//                 (LBFS.cu:2177-2240): its own stencil rows plus, per
//                 neighbour, the neighbour's row that points back to it
//                 (weights gathered once on the host), plus the
//                 interpolation adjoint held in fixed point
//
// Strict upwinding (ties to the owner) is piecewise smooth; its derivative is
// taken on the side the forward step took.  No floating-point atomics:
// results are bitwise repeatable.
#include <hip/hip_runtime.h>

#include "adjoint.hpp"
#include "fluid_device.hpp"

namespace lbfs {

// ---------------------------------------------------------------------------
// update
// ---------------------------------------------------------------------------
// forward: drho' = drho + dt r0, rho' = rho0 + drho',
//          u'_t  = u_t + dt (r_t + f_t - u_t r0) / rho'
// Cell i of the update's adjoint from the step's state adjoint L, its start
// state s0, residual r and cell force cf; p: the cell's body-force terms.
__device__ __forceinline__ void adj_update_cell(const FluidArgs &a, const AdjFluidArgs &j, const float *cf_all, int i,
                                                float4 L, float4 s0, float4 r, double p[3])
{
    float fx = a.body_force[0], fy = a.body_force[1], fz = a.body_force[2];
    if (cf_all) {
        const float *cf = cf_all + 3 * (size_t)i;
        fx += cf[0]; fy += cf[1]; fz += cf[2];
    }
    const float r0 = r.x, r1 = r.y + fx, r2 = r.z + fy, r3 = r.w + fz;
    const float dt = a.dt;
    const float rho = a.rho0 + (s0.x + dt * r0);
    const float inv = 1.0f / rho;
    const float a1 = dt * (r1 - s0.y * r0), a2 = dt * (r2 - s0.z * r0), a3 = dt * (r3 - s0.w * r0);
    const float lrho = -inv * inv * (L.y * a1 + L.z * a2 + L.w * a3);
    const float ld = L.x + lrho;
    const float lr0 = dt * ld - dt * inv * (L.y * s0.y + L.z * s0.z + L.w * s0.w);
    const float c = dt * inv;
    const float lr1 = L.y * c, lr2 = L.z * c, lr3 = L.w * c;
    const float keep = 1.0f - dt * r0 * inv;
    const float iv = a.inv_vol[i];
    j.mu[i] = make_float4(lr0 * iv, lr1 * iv, lr2 * iv, lr3 * iv);
    j.lcf[i] = make_float4(lr1, lr2, lr3, 0.0f);
    j.ls[i] = make_float4(ld, L.y * keep, L.z * keep, L.w * keep);
    p[0] = lr1; p[1] = lr2; p[2] = lr3;
}

// the workgroup's body-force terms (256 threads, one cell each) added to its
// own partials: the running sums need no atomics
__device__ __forceinline__ void adj_force_partials(const AdjFluidArgs &j, const double p[3])
{
    __shared__ double sh[3][256];
    for (int t = 0; t < 3; t++) sh[t][threadIdx.x] = p[t];
    __syncthreads();
    for (int stp = 128; stp > 0; stp >>= 1) {
        if ((int)threadIdx.x < stp)
            for (int t = 0; t < 3; t++) sh[t][threadIdx.x] += sh[t][threadIdx.x + stp];
        __syncthreads();
    }
    if (threadIdx.x < 3) j.fpart[3 * (size_t)blockIdx.x + threadIdx.x] += sh[threadIdx.x][0];
}

__global__ __launch_bounds__(256) void k_adj_update(FluidArgs a, AdjFluidArgs j, const float4 *__restrict__ st,
                                                    const float4 *__restrict__ res)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    double p[3] = {0.0, 0.0, 0.0};
    if (i < a.n_cells) adj_update_cell(a, j, a.cell_force, i, j.lam_in[i], st[i], res[i], p);
    adj_force_partials(j, p);
}

// fixed-order sum of the partials into the body-force gradient
__global__ __launch_bounds__(256) void k_adj_force_sum(AdjFluidArgs j)
{
    __shared__ double sh[3][256];
    double p[3] = {0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < j.n_fpart; b += 256)
        for (int t = 0; t < 3; t++) p[t] += j.fpart[3 * (size_t)b + t];
    for (int t = 0; t < 3; t++) sh[t][threadIdx.x] = p[t];
    __syncthreads();
    for (int stp = 128; stp > 0; stp >>= 1) {
        if ((int)threadIdx.x < stp)
            for (int t = 0; t < 3; t++) sh[t][threadIdx.x] += sh[t][threadIdx.x + stp];
        __syncthreads();
    }
    if (threadIdx.x < 3) j.gforce[threadIdx.x] = sh[threadIdx.x][0];
}

// ---------------------------------------------------------------------------
// face flux
// ---------------------------------------------------------------------------
// adjoint of g = w (q0 + (rho0 + q0) P), P = eu (3 + 4.5 ig eu) - 1.5 ig |q_u|^2
__device__ __forceinline__ void eq_point_vjp(const float q[4], float eu, float lg, float w, float rho0, float ig,
                                             float lq[4], float &leu)
{
    const float uu = q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
    const float P = eu * (3.0f + 4.5f * ig * eu) - 1.5f * ig * uu;
    const float R = lg * w * (rho0 + q[0]);
    lq[0] = lg * w * (1.0f + P);
    leu = R * (3.0f + 9.0f * ig * eu);
    const float c = -3.0f * ig * R;
    lq[1] = c * q[1];
    lq[2] = c * q[2];
    lq[3] = c * q[3];
}

// adjoint moments of the face: S0 += gs, S1 += e gd, T += e (e.n) gs
struct FaceAdj {
    float lS0, lS1x, lS1y, lS1z, lTx, lTy, lTz;
};

// One pair of opposite directions in reverse: the forward reconstruction of
// the two lattice points (owner side along s e, neighbour side along -s e,
// s = sign(e.n); a tie feeds both from the owner) and the transpose of it.
template <class L, int K>
__device__ __forceinline__ void pair_vjp(const FaceAdj &fa, const float po[4], const float pn[4], const float Go[12],
                                         const float Gn[12], float nx, float ny, float nz, float rho0, float ig,
                                         float lpo[4], float lpn[4], float lGo[12], float lGn[12])
{
    constexpr int ex = L::ex[K], ey = L::ey[K], ez = L::ez[K];
    constexpr float w = L::w(K);
    const float en = edot<ex, ey, ez>(nx, ny, nz);
    const bool tie = en == 0.0f;
    const float sg = en > 0.0f ? 1.0f : -1.0f;
    float ego[4], egn[4], qo[4], qn[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        ego[v] = edot<ex, ey, ez>(Go[3 * v], Go[3 * v + 1], Go[3 * v + 2]);
        egn[v] = edot<ex, ey, ez>(Gn[3 * v], Gn[3 * v + 1], Gn[3 * v + 2]);
        qo[v] = po[v] - sg * ego[v];
        qn[v] = tie ? po[v] - ego[v] : pn[v] + sg * egn[v];
    }
    const float eu_o = sg * edot<ex, ey, ez>(qo[1], qo[2], qo[3]);
    const float eu_n = -sg * edot<ex, ey, ez>(qn[1], qn[2], qn[3]);
    const float lgs = fa.lS0 + en * edot<ex, ey, ez>(fa.lTx, fa.lTy, fa.lTz);
    const float lgd = edot<ex, ey, ez>(fa.lS1x, fa.lS1y, fa.lS1z);
    const float lgo = lgs + sg * lgd, lgn = lgs - sg * lgd;
    float lqo[4], lqn[4], leo, len;
    eq_point_vjp(qo, eu_o, lgo, w, rho0, ig, lqo, leo);
    eq_point_vjp(qn, eu_n, lgn, w, rho0, ig, lqn, len);
    leo *= sg;
    len *= -sg;
    eacc<ex>(lqo[1], leo); eacc<ey>(lqo[2], leo); eacc<ez>(lqo[3], leo);
    eacc<ex>(lqn[1], len); eacc<ey>(lqn[2], len); eacc<ez>(lqn[3], len);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        // qo = po - s ego; qn = pn + s egn, or po - ego on a tie
        float lego = -sg * lqo[v], legn = 0.0f;
        lpo[v] += lqo[v];
        if (tie) {
            lpo[v] += lqn[v];
            lego -= lqn[v];
        } else {
            lpn[v] += lqn[v];
            legn = sg * lqn[v];
        }
        eacc<ex>(lGo[3 * v], lego); eacc<ey>(lGo[3 * v + 1], lego); eacc<ez>(lGo[3 * v + 2], lego);
        eacc<ex>(lGn[3 * v], legn); eacc<ey>(lGn[3 * v + 1], legn); eacc<ez>(lGn[3 * v + 2], legn);
    }
}

template <class L, int... P>
__device__ __forceinline__ void all_pair_vjps(std::integer_sequence<int, P...>, const FaceAdj &fa, const float po[4],
                                              const float pn[4], const float Go[12], const float Gn[12], float nx,
                                              float ny, float nz, float rho0, float ig, float lpo[4], float lpn[4],
                                              float lGo[12], float lGn[12])
{
    (pair_vjp<L, 2 * P + 1>(fa, po, pn, Go, Gn, nx, ny, nz, rho0, ig, lpo, lpn, lGo, lGn), ...);
}

// What one tile-face's adjoint reads: its record, its moments S0 and S1 as the
// forward pass computed them, and the state, gradient and residual adjoint of
// both sides (a boundary face's neighbour is unused)
struct FaceLoads {
    FaceRaw raw;
    float4 mom, so, sn, mo, mn, go[3], gn[3];
};
__device__ __forceinline__ FaceLoads load_face(const FluidArgs &a, const float4 *__restrict__ st,
                                               const float4 *__restrict__ grad, const float4 *__restrict__ mu, int tf,
                                               int o, int n)
{
    FaceLoads l;
    l.raw = load_face_raw(a, tf);
    l.mom = a.face_moments[tf];
    l.so = st[o]; l.sn = st[n];
    l.mo = mu[o]; l.mn = mu[n];
#pragma unroll
    for (int k = 0; k < 3; k++) { l.go[k] = grad[3 * (size_t)o + k]; l.gn[k] = grad[3 * (size_t)n + k]; }
    return l;
}
__device__ __forceinline__ void grad_array(const float4 v[3], float g[12])
{
#pragma unroll
    for (int k = 0; k < 3; k++) { g[4 * k] = v[k].x; g[4 * k + 1] = v[k].y; g[4 * k + 2] = v[k].z; g[4 * k + 3] = v[k].w; }
}

// reverse of the flux from the moments to the moments' adjoints; lam: the flux
// adjoint (neighbour's residual adjoint less the owner's)
template <class L>
__device__ __forceinline__ FaceAdj flux_vjp(const FluidArgs &a, const FaceRec &fr, float4 fm, float4 lam, int o)
{
    const float nx = fr.nx, ny = fr.ny, nz = fr.nz, A = fr.A, ig = a.inv_gamma;
    const float rho_f = a.rho0 + fm.x;
    const float mnrm = fm.y * nx + fm.z * ny + fm.w * nz;
    const float vf = a.visc_factor ? a.visc_factor[o] : 1.0f;
    const float tau = a.visc3_over_gamma * vf / fr.dt;
    const float c1 = 1.0f - tau;
    const float irf = 1.0f / rho_f;
    const float q = mnrm * irf * ig;
    const float Lx = lam.y, Ly = lam.z, Lz = L::dims == 3 ? lam.w : 0.0f;
    const float lq = A * c1 * (Lx * fm.y + Ly * fm.z + Lz * fm.w);
    const float lmn = lam.x * A + lq * ig * irf;
    const float lrf = -lq * mnrm * ig * irf * irf;
    FaceAdj fj;
    fj.lS0 = A * c1 * (Lx * nx + Ly * ny + Lz * nz) * (1.0f / 3.0f) + lrf;
    fj.lS1x = Lx * A * c1 * q + lmn * nx;
    fj.lS1y = Ly * A * c1 * q + lmn * ny;
    fj.lS1z = Lz * A * c1 * q + lmn * nz;
    fj.lTx = Lx * A * tau;
    fj.lTy = Ly * A * tau;
    fj.lTz = Lz * A * tau;
    return fj;
}

// adjoint of the rest point (the mean state of both sides)
template <class L>
__device__ __forceinline__ void rest_vjp(const FluidArgs &a, const FaceAdj &fj, const float p0[4], float lp0[4])
{
    const float ig = a.inv_gamma, w0 = L::w(0);
    const float P0 = -1.5f * (p0[1] * p0[1] + p0[2] * p0[2] + p0[3] * p0[3]) * ig;
    lp0[0] = fj.lS0 * w0 * (1.0f + P0);
    const float c = fj.lS0 * w0 * (a.rho0 + p0[0]) * (-3.0f * ig);
    lp0[1] = c * p0[1];
    lp0[2] = c * p0[2];
    lp0[3] = c * p0[3];
}

// One side of a face whose lattice directions all lie clearly on one side
// (FaceRec::general unset): the points along s e (s the direction's sign on
// this side) come from this side alone, q = p - s dt (e.grad).  With R the
// adjoint factor of a point's velocity terms and h that of its e.u, the point
// adjoint of velocity u_t is -3/gamma R u_t + e_t h, linear in the side's p and
// grad: only the moments of R, h and the density adjoint over the directions
// are summed here, 14 sums a point in place of the 4 + 12 components' own
// (with their selections on a tie): about 970 instructions a face for the 1350
// of face_vjp, which faces with a tie keep.
struct SideMoments {
    float z0, z[3];         // density adjoint l: sum l, sum s e l
    float m0, m[3], mm[6];  // sum R, sum s e R, sum e e R (xx, yy, zz, xy, xz, yz)
    float h[3], hh[6];      // sum e h, sum s e e h
};
template <int EX, int EY, int EZ>
__device__ __forceinline__ void point_vjp(SideMoments &m, const float p[4], const float g[12], float sdt, float s,
                                          float s3, float lg, float rho0, float ig45, float ig15)
{
    float q[4];
#pragma unroll
    for (int v = 0; v < 4; v++) q[v] = fmaf(-sdt, edot<EX, EY, EZ>(g[3 * v], g[3 * v + 1], g[3 * v + 2]), p[v]);
    const float x = edot<EX, EY, EZ>(q[1], q[2], q[3]);
    const float uu = dot3(q[1], q[2], q[3], q[1], q[2], q[3]);
    const float t = fmaf(ig45, x, s3);
    const float P = fmaf(x, t, -ig15 * uu);
    const float l = fmaf(lg, P, lg), R = lg * (rho0 + q[0]), h = R * fmaf(ig45, x, t);
    m.z0 += l;
    efma<EX>(m.z[0], s, l); efma<EY>(m.z[1], s, l); efma<EZ>(m.z[2], s, l);
    m.m0 += R;
    efma<EX>(m.m[0], s, R); efma<EY>(m.m[1], s, R); efma<EZ>(m.m[2], s, R);
    eacc<EX * EX>(m.mm[0], R); eacc<EY * EY>(m.mm[1], R); eacc<EZ * EZ>(m.mm[2], R);
    eacc<EX * EY>(m.mm[3], R); eacc<EX * EZ>(m.mm[4], R); eacc<EY * EZ>(m.mm[5], R);
    eacc<EX>(m.h[0], h); eacc<EY>(m.h[1], h); eacc<EZ>(m.h[2], h);
    efma<EX * EX>(m.hh[0], s, h); efma<EY * EY>(m.hh[1], s, h); efma<EZ * EZ>(m.hh[2], s, h);
    efma<EX * EY>(m.hh[3], s, h); efma<EX * EZ>(m.hh[4], s, h); efma<EY * EZ>(m.hh[5], s, h);
}
template <class L, int K>
__device__ __forceinline__ void pair_vjp_clear(SideMoments &mo, SideMoments &mn, const FaceAdj &fa, const float po[4],
                                               const float pn[4], const float go[12], const float gn[12],
                                               const FaceRec &fr, float rho0, float ig45, float ig15)
{
    constexpr int ex = L::ex[K], ey = L::ey[K], ez = L::ez[K];
    constexpr float w = L::w(K);
    const float en = edot<ex, ey, ez>(fr.nx, fr.ny, fr.nz);
    const float sdt = copysignf(fr.dt, en), s = copysignf(1.0f, en), s3 = copysignf(3.0f, en);
    const float lgs = w * fmaf(en, edot<ex, ey, ez>(fa.lTx, fa.lTy, fa.lTz), fa.lS0);
    const float lgd = copysignf(w, en) * edot<ex, ey, ez>(fa.lS1x, fa.lS1y, fa.lS1z);
    point_vjp<ex, ey, ez>(mo, po, go, sdt, s, s3, lgs + lgd, rho0, ig45, ig15);
    point_vjp<ex, ey, ez>(mn, pn, gn, -sdt, -s, -s3, lgs - lgd, rho0, ig45, ig15);
}
template <class L, int... P>
__device__ __forceinline__ void all_pair_vjps_clear(std::integer_sequence<int, P...>, SideMoments &mo,
                                                    SideMoments &mn, const FaceAdj &fa, const float po[4],
                                                    const float pn[4], const float go[12], const float gn[12],
                                                    const FaceRec &fr, float rho0, float ig45, float ig15)
{
    (pair_vjp_clear<L, 2 * P + 1>(mo, mn, fa, po, pn, go, gn, fr, rho0, ig45, ig15), ...);
}
// a side's state (out[0]) and gradient (out[1..3]) adjoint from its moments
// and the rest point's; d: its centroid's offset from the face
__device__ __forceinline__ void side_vjp(const SideMoments &m, const float p[4], const float g[12], const float lp0[4],
                                         float3 d, float dt, float ig, float4 out[4])
{
    const float c = -3.0f * ig, cd = c * dt, cdd = cd * dt;
    const float m0 = c * m.m0, m1[3] = {cd * m.m[0], cd * m.m[1], cd * m.m[2]};
    const float xx = cdd * m.mm[0], yy = cdd * m.mm[1], zz = cdd * m.mm[2];
    const float xy = cdd * m.mm[3], xz = cdd * m.mm[4], yz = cdd * m.mm[5];
    const float hx[3] = {m.hh[0], m.hh[3], m.hh[4]}, hy[3] = {m.hh[3], m.hh[1], m.hh[5]},
                hz[3] = {m.hh[4], m.hh[5], m.hh[2]};
    float ls[4], lg[12];
    ls[0] = m.z0 + 0.5f * lp0[0];
    lg[0] = -dt * m.z[0]; lg[1] = -dt * m.z[1]; lg[2] = -dt * m.z[2];
#pragma unroll
    for (int t = 0; t < 3; t++) {
        const float gx = g[3 * t + 3], gy = g[3 * t + 4], gz = g[3 * t + 5], u = p[t + 1];
        ls[t + 1] = m.h[t] + u * m0 - (gx * m1[0] + gy * m1[1] + gz * m1[2]) + 0.5f * lp0[t + 1];
        lg[3 * t + 3] = (gx * xx + gy * xy + gz * xz) - u * m1[0] - dt * hx[t];
        lg[3 * t + 4] = (gx * xy + gy * yy + gz * yz) - u * m1[1] - dt * hy[t];
        lg[3 * t + 5] = (gx * xz + gy * yz + gz * zz) - u * m1[2] - dt * hz[t];
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
        lg[3 * v] -= d.x * ls[v]; lg[3 * v + 1] -= d.y * ls[v]; lg[3 * v + 2] -= d.z * ls[v];
    }
    out[0] = make_float4(ls[0], ls[1], ls[2], ls[3]);
    out[1] = make_float4(lg[0], lg[1], lg[2], lg[3]);
    out[2] = make_float4(lg[4], lg[5], lg[6], lg[7]);
    out[3] = make_float4(lg[8], lg[9], lg[10], lg[11]);
}

// Adjoint of the flux of a face clear of every lattice direction (laid out as
// face_vjp's)
template <class L>
__device__ __forceinline__ void face_vjp_clear(const FluidArgs &a, const FaceLoads &in, const FaceRec &fr, int o,
                                               float4 out[8])
{
    const float sov[4] = {in.so.x, in.so.y, in.so.z, in.so.w}, snv[4] = {in.sn.x, in.sn.y, in.sn.z, in.sn.w};
    float go[12], gn[12], po[4], pn[4], p0[4], lp0[4];
    grad_array(in.go, go);
    grad_array(in.gn, gn);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        po[v] = sov[v] - (fr.d1.x * go[3 * v] + fr.d1.y * go[3 * v + 1] + fr.d1.z * go[3 * v + 2]);
        pn[v] = snv[v] - (fr.d2.x * gn[3 * v] + fr.d2.y * gn[3 * v + 1] + fr.d2.z * gn[3 * v + 2]);
        p0[v] = 0.5f * (po[v] + pn[v]);
    }
    const float4 lam = make_float4(in.mn.x - in.mo.x, in.mn.y - in.mo.y, in.mn.z - in.mo.z, in.mn.w - in.mo.w);
    const FaceAdj fj = flux_vjp<L>(a, fr, in.mom, lam, o);
    rest_vjp<L>(a, fj, p0, lp0);
    const float ig = a.inv_gamma;
    SideMoments mo = {}, mn = {};
    all_pair_vjps_clear<L>(std::make_integer_sequence<int, (L::Q - 1) / 2>{}, mo, mn, fj, po, pn, go, gn, fr, a.rho0,
                           4.5f * ig, 1.5f * ig);
    side_vjp(mo, po, go, lp0, fr.d1, fr.dt, ig, out);
    side_vjp(mn, pn, gn, lp0, fr.d2, fr.dt, ig, out + 4);
}

// Adjoint of one tile-face's flux (the forward of face_flux in
// fluid_kernels.hip, strict upwinding), from the face's moments S0, S1 as the
// forward pass computed them.  out[0] state and out[1..3] gradient
// adjoint of the owner, out[4..7] the same for the neighbour (zero for a
// boundary face, whose ghost is a function of the owner).  Boundary faces, and
// interior faces whose points may come from either side.
template <class L, bool GHOST>
__device__ __forceinline__ void face_vjp(const FluidArgs &a, const FaceLoads &in, const FaceRec &fr, int o, int nb,
                                         float4 out[8])
{
    const float3 fb = fr.d1, fcv = fr.d2;
    constexpr bool ghost = GHOST;  // boundary faces follow the interior faces in every tile list
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < 8; k++) out[k] = zero;
    const float nx = fr.nx, ny = fr.ny, nz = fr.nz, dt = fr.dt;
    const float4 so = in.so, mo = in.mo;
    float go[12], gn[12];
    grad_array(in.go, go);
    const float sov[4] = {so.x, so.y, so.z, so.w};
    float po[4], pn[4], p0[4];
    float4 lam;
    int ty[4] = {0, 0, 0, 0};
    float inv_dmag = 0.0f, dir[3] = {0.0f, 0.0f, 0.0f}, fac[3] = {1.0f, 1.0f, 1.0f};
    if (!ghost) {
        const float4 sn = in.sn, mn4 = in.mn;
        lam = make_float4(mn4.x - mo.x, mn4.y - mo.y, mn4.z - mo.z, mn4.w - mo.w);
        grad_array(in.gn, gn);
        const float snv[4] = {sn.x, sn.y, sn.z, sn.w};
#pragma unroll
        for (int v = 0; v < 4; v++) {
            po[v] = sov[v] - (fb.x * go[3 * v] + fb.y * go[3 * v + 1] + fb.z * go[3 * v + 2]);
            pn[v] = snv[v] - (fcv.x * gn[3 * v] + fcv.y * gn[3 * v + 1] + fcv.z * gn[3 * v + 2]);
            p0[v] = 0.5f * (po[v] + pn[v]);
        }
    } else {
        const int bc = nb - a.n_cells;
        const int2 t2 = a.bc_type[bc];
        if (t2.y == LBFS_BC_EMPTY) return;
        lam = make_float4(-mo.x, -mo.y, -mo.z, -mo.w);
        const float4 bv = a.bc_val[bc];
        const float bvv[4] = {bv.x, bv.y, bv.z, bv.w};
        const float d1n = sqrtf(fb.x * fb.x + fb.y * fb.y + fb.z * fb.z);
        inv_dmag = 2.0f / d1n;
        if (a.flags & LBFS_FLAG_GHOST_DIR_GPU) { dir[0] = -fb.x / d1n; dir[1] = -fb.y / d1n; dir[2] = -fb.z / d1n; }
        else { dir[0] = nx; dir[1] = ny; dir[2] = nz; }
        const float nv[3] = {nx, ny, nz};
#pragma unroll
        for (int c = 0; c < 3; c++) fac[c] = (a.flags & LBFS_FLAG_NEUMANN_SIGNED) ? 1.0f - nv[c] : 1.0f - fabsf(nv[c]);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            ty[v] = v == 0 ? t2.x : t2.y;
            if (ty[v] == 1 || ty[v] == 3) {
                const float dphi = 2.0f * (bvv[v] - sov[v]) * inv_dmag;
#pragma unroll
                for (int c = 0; c < 3; c++) gn[3 * v + c] = dphi * dir[c];
                p0[v] = ty[v] == 1 ? bvv[v] : sov[v] - (fb.x * gn[3 * v] + fb.y * gn[3 * v + 1] + fb.z * gn[3 * v + 2]);
            } else {
#pragma unroll
                for (int c = 0; c < 3; c++) gn[3 * v + c] = go[3 * v + c] * fac[c];
                p0[v] = sov[v] - (fb.x * gn[3 * v] + fb.y * gn[3 * v + 1] + fb.z * gn[3 * v + 2]);
            }
            po[v] = p0[v];
            pn[v] = p0[v];
        }
    }
    // LBFS_FLAG_GHOST_FACE_GRAD: the owner-side points of a boundary face take
    // the ghost gradient (LBFS.cu:391-394); the reverse below routes their
    // gradient adjoint into the ghost gradient's
    const bool ghost_grad_all = ghost && (a.flags & LBFS_FLAG_GHOST_FACE_GRAD);
    if (ghost_grad_all) {
#pragma unroll
        for (int t = 0; t < 12; t++) go[t] = gn[t];
    }
    float Go[12], Gn[12];
#pragma unroll
    for (int t = 0; t < 12; t++) { Go[t] = go[t] * dt; Gn[t] = gn[t] * dt; }
    const float rho0 = a.rho0, ig = a.inv_gamma;
    const FaceAdj fj = flux_vjp<L>(a, fr, in.mom, lam, o);
    float lp0[4];
    rest_vjp<L>(a, fj, p0, lp0);
    float lpo[4] = {0.0f, 0.0f, 0.0f, 0.0f}, lpn[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    float lGo[12], lGn[12];
#pragma unroll
    for (int t = 0; t < 12; t++) { lGo[t] = 0.0f; lGn[t] = 0.0f; }
    all_pair_vjps<L>(std::make_integer_sequence<int, (L::Q - 1) / 2>{}, fj, po, pn, Go, Gn, nx, ny, nz, rho0, ig, lpo,
                     lpn, lGo, lGn);
    float lso[4], lgo_[12];
    if (!ghost) {
        float lsn[4], lgn_[12];
        const float d1[3] = {fb.x, fb.y, fb.z}, d2[3] = {fcv.x, fcv.y, fcv.z};
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float a_o = lpo[v] + 0.5f * lp0[v], a_n = lpn[v] + 0.5f * lp0[v];
            lso[v] = a_o;
            lsn[v] = a_n;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                lgo_[3 * v + c] = dt * lGo[3 * v + c] - d1[c] * a_o;
                lgn_[3 * v + c] = dt * lGn[3 * v + c] - d2[c] * a_n;
            }
        }
        out[4] = make_float4(lsn[0], lsn[1], lsn[2], lsn[3]);
        out[5] = make_float4(lgn_[0], lgn_[1], lgn_[2], lgn_[3]);
        out[6] = make_float4(lgn_[4], lgn_[5], lgn_[6], lgn_[7]);
        out[7] = make_float4(lgn_[8], lgn_[9], lgn_[10], lgn_[11]);
    } else {
        const float d1[3] = {fb.x, fb.y, fb.z};
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float lp = lpo[v] + lpn[v] + lp0[v];  // every lattice point starts from the face value
            float lgv[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (ghost_grad_all) {
                    lgo_[3 * v + c] = 0.0f;
                    lgv[c] = dt * (lGn[3 * v + c] + lGo[3 * v + c]);
                } else {
                    lgo_[3 * v + c] = dt * lGo[3 * v + c];
                    lgv[c] = dt * lGn[3 * v + c];
                }
            }
            lso[v] = 0.0f;
            if (ty[v] == 1 || ty[v] == 3) {
                if (ty[v] == 3) {
                    lso[v] += lp;
#pragma unroll
                    for (int c = 0; c < 3; c++) lgv[c] -= d1[c] * lp;
                }
                const float ldphi = dir[0] * lgv[0] + dir[1] * lgv[1] + dir[2] * lgv[2];
                lso[v] -= 2.0f * inv_dmag * ldphi;
            } else {
                lso[v] += lp;
#pragma unroll
                for (int c = 0; c < 3; c++) lgo_[3 * v + c] += fac[c] * (lgv[c] - d1[c] * lp);
            }
        }
    }
    out[0] = make_float4(lso[0], lso[1], lso[2], lso[3]);
    out[1] = make_float4(lgo_[0], lgo_[1], lgo_[2], lgo_[3]);
    out[2] = make_float4(lgo_[4], lgo_[5], lgo_[6], lgo_[7]);
    out[3] = make_float4(lgo_[8], lgo_[9], lgo_[10], lgo_[11]);
}

__device__ __forceinline__ void add4(float *acc, float4 v)
{
    acc[0] += v.x; acc[1] += v.y; acc[2] += v.z; acc[3] += v.w;
}

// Bound by its waits: each chunk's loads, its faces and its sums follow one
// another behind barriers, and some 180 registers leave two wavefronts a SIMD.
// Workgroups of 256 threads put two of them on a compute unit, one's faces
// beside the other's loads and sums.  128x64x64, D3Q19, 8x8x8 tiles: 512
// threads 111 us, with the moments of face_vjp_clear (37.4 -> 29.6 M vector
// instructions) 112; 256 threads 85.  Three workgroups in 168 registers take
// 107 (spills), or 96 with one side of a face after the other; the next
// chunk's loads issued ahead gain nothing at two.  Tiles of more than 512 cells
// keep 512 threads of two cells: four cells' sums a thread spill (20 steps of
// 64x48x48 on 16x8x8 tiles reversed in 2.16 ms, 2.43 with 256 threads).
// NT: threads, and the faces per LDS chunk (8 float4 each), held as 8 planes of NT
// float4 so that a wavefront's stores are contiguous; ADJ_CELLS: cells per thread
template <class L, int NT, int ADJ_CELLS>
__global__ __launch_bounds__(NT) void k_adj_flux(FluidArgs a, AdjFluidArgs j, const float4 *__restrict__ st,
                                                 const float4 *__restrict__ grad)
{
    extern __shared__ float4 lds_adj[];
    const TileRec T = a.tiles[xcd_remap(blockIdx.x, gridDim.x)];
    const int c0 = T.c0, c1 = T.c0 + T.nc;
    int *ids = reinterpret_cast<int *>(lds_adj + 8 * NT);  // cell id of each slot
    for (int q = threadIdx.x; q < T.nc + T.nh; q += NT) ids[q] = slot_cell(a, T, q);
    float acc[ADJ_CELLS][16];
    uint32_t slot[ADJ_CELLS][3];  // two slots each; 0x7fff: none
#pragma unroll
    for (int u = 0; u < ADJ_CELLS; u++) {
#pragma unroll
        for (int k = 0; k < 16; k++) acc[u][k] = 0.0f;
        const int i = (int)threadIdx.x + u * NT;
        const uint32_t *sl = reinterpret_cast<const uint32_t *>(a.cell_slots) + 3 * (size_t)(T.pc + i);
#pragma unroll
        for (int k = 0; k < 3; k++) slot[u][k] = i < T.nc ? sl[k] : 0x7fff7fffu;
    }
    const int last = T.nc + T.nh - 1;
    __syncthreads();
    for (int cs = 0; cs < T.nf; cs += NT) {
        const int q = cs + (int)threadIdx.x;
        if (q < T.nf) {
            // (a boundary face's neighbour slot is 0xffff: some cell of the tile's, unused)
            const uint32_t gs = a.face_gslot[T.pf + q];
            const int oc = ids[gs & 0xffffu];
            const FaceLoads in = load_face(a, st, grad, j.mu, T.f0 + q, oc, ids[min((int)(gs >> 16), last)]);
            const FaceRec fr = unpack_face(in.raw);
            float4 o[8];
            if (!fr.general) face_vjp_clear<L>(a, in, fr, oc, o);
            else if (q < T.nif) face_vjp<L, false>(a, in, fr, oc, 0, o);
            else face_vjp<L, true>(a, in, fr, oc, a.n_cells + a.tile_bc[T.b0 + q - T.nif], o);
#pragma unroll
            for (int k = 0; k < 8; k++) lds_adj[k * NT + threadIdx.x] = o[k];
        }
        __syncthreads();
        const uint32_t base = (uint32_t)cs, n = (uint32_t)min(NT, T.nf - cs);
#pragma unroll
        for (int u = 0; u < ADJ_CELLS; u++)
#pragma unroll
            for (int k = 0; k < 6; k++) {
                const uint32_t s = slot[u][k / 2] >> 16 * (k & 1);
                const uint32_t r = (s & 0x7fffu) - base;
                if (r >= n) continue;
                const int side = (s & 0x8000u) ? 0 : 4;  // bit 15 set: the cell owns the face
                const float4 *src = lds_adj + side * NT + r;
#pragma unroll
                for (int v = 0; v < 4; v++) add4(&acc[u][4 * v], src[v * NT]);
            }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < ADJ_CELLS; u++) {
        const int i = c0 + (int)threadIdx.x + u * NT;
        if (i >= c1) continue;
        const float4 l = j.ls[i];
        j.ls_acc[i] = make_float4(l.x + acc[u][0], l.y + acc[u][1], l.z + acc[u][2], l.w + acc[u][3]);
        j.lam_g[3 * (size_t)i + 0] = make_float4(acc[u][4], acc[u][5], acc[u][6], acc[u][7]);
        j.lam_g[3 * (size_t)i + 1] = make_float4(acc[u][8], acc[u][9], acc[u][10], acc[u][11]);
        j.lam_g[3 * (size_t)i + 2] = make_float4(acc[u][12], acc[u][13], acc[u][14], acc[u][15]);
    }
}

// ---------------------------------------------------------------------------
// gradients
// ---------------------------------------------------------------------------
// forward: grad_i[v] = sum_k W_k(i) d_k[v], d_k = st_j - st_i (interior),
// 2 (bc - st_i) for a mirrored ghost value, 0 for a copied one
__device__ __forceinline__ void lam_grad(const float4 *__restrict__ lg, int i, float g[12])
{
    const float4 a = lg[3 * (size_t)i], b = lg[3 * (size_t)i + 1], c = lg[3 * (size_t)i + 2];
    g[0] = a.x; g[1] = a.y; g[2] = a.z; g[3] = a.w;
    g[4] = b.x; g[5] = b.y; g[6] = b.z; g[7] = b.w;
    g[8] = c.x; g[9] = c.y; g[10] = c.z; g[11] = c.w;
}

// Reverse stencil rows (set-up): slot k of cell i, neighbour c, takes the
// weights of c's slot that points back to i; where i meets c through several
// slots, the r-th of them takes the r-th of c's.  A cell's slots depend on no
// other cell's choice, so each is found by itself: on the host, in one thread,
// this was 40 ms of the 524288-cell channel's first gradient (70 -> 30 ms).
__global__ __launch_bounds__(256) void k_adj_rev_rows(FluidArgs a, float4 *__restrict__ rev_w,
                                                      unsigned int *__restrict__ lone)
{
    const int n = a.n_cells, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    int jk[6];
#pragma unroll
    for (int k = 0; k < 6; k++) jk[k] = a.stencil[(size_t)k * n + i];
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int c = jk[k];
        float4 w = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (c >= 0) {
            int r = 0, found = -1;
#pragma unroll
            for (int p = 0; p < k; p++) r += jk[p] == c;
#pragma unroll
            for (int kb = 0; kb < 6; kb++)
                if (a.stencil[(size_t)kb * n + c] == i && r-- == 0) found = kb;
            if (found >= 0) {
                const float *g = a.gw + (size_t)(3 * found) * n + c;
                w = make_float4(g[0], g[n], g[2 * (size_t)n], 0.0f);
            } else {
                *lone = 1u;
            }
        }
        rev_w[(size_t)k * n + i] = w;
    }
}

// The transpose of the gradients for cell i: its state adjoint (written to
// lam_out and returned).
__device__ __forceinline__ float4 adj_grad_cell(const FluidArgs &a, const AdjFluidArgs &j, int i)
{
    const int n = a.n_cells;
    const float4 l0 = j.ls_acc[i];
    float acc[4] = {l0.x, l0.y, l0.z, l0.w};
    float g[12];
    lam_grad(j.lam_g, i, g);
    // every stencil index and weight first, then the neighbours' rows and
    // adjoint gradients three entries at a time (a boundary entry loads the
    // cell's own, unused), so the loads are in flight together rather than
    // one index and one neighbour at a time
    int jk[6];
#pragma unroll
    for (int k = 0; k < 6; k++) jk[k] = a.stencil[(size_t)k * n + i];
    float wk[18];
#pragma unroll
    for (int k = 0; k < 18; k++) wk[k] = a.gw[(size_t)k * n + i];
#pragma unroll
    for (int k0 = 0; k0 < 6; k0 += 3) {
        float4 rk[3];
        float gk[3][12];
#pragma unroll
        for (int u = 0; u < 3; u++) {
            const int jn = jk[k0 + u];
            rk[u] = j.rev_w[(size_t)(k0 + u) * n + i];
            lam_grad(j.lam_g, jn >= 0 ? jn : i, gk[u]);
        }
#pragma unroll
        for (int u = 0; u < 3; u++) {
            const int k = k0 + u, jn = jk[k];
            const float wx = wk[3 * k], wy = wk[3 * k + 1], wz = wk[3 * k + 2];
            float c[4] = {1.0f, 1.0f, 1.0f, 1.0f};
            if (jn < 0) {
                const int2 ty = a.bc_type[-1 - jn];
                const bool mv = ty.y == 1 || ty.y == 3;
                c[0] = ty.x == 1 ? 2.0f : 0.0f;
                c[1] = c[2] = c[3] = mv ? 2.0f : 0.0f;
            }
#pragma unroll
            for (int v = 0; v < 4; v++) acc[v] -= c[v] * (wx * g[3 * v] + wy * g[3 * v + 1] + wz * g[3 * v + 2]);
            if (jn >= 0) {
                // the neighbour's stencil row that points back here
                const float4 r = rk[u];
                const float *gc = gk[u];
#pragma unroll
                for (int v = 0; v < 4; v++) acc[v] += r.x * gc[3 * v] + r.y * gc[3 * v + 1] + r.z * gc[3 * v + 2];
            }
        }
    }
    if (j.acc_rw) {
        // the interpolation adjoint is held as v 2^(40 - e), e the binary
        // exponent of the largest adjoint node velocity component
        const double inv_scale = adj_fix_inv_scale(*j.umax);
        unsigned long long *p = j.acc_rw + 3 * (size_t)i;
#pragma unroll
        for (int t = 0; t < 3; t++) {
            const long long v = (long long)p[t];
            if (v != 0) {
                acc[1 + t] += (float)((double)v * inv_scale);
                p[t] = 0ull;
            }
        }
    }
    const float4 L = make_float4(acc[0], acc[1], acc[2], acc[3]);
    j.lam_out[i] = L;
    return L;
}

// UPD: the update adjoint of the step before follows in the same pass (its
// state adjoint is the one just computed; every reader of the update
// adjoint's outputs of this step has finished): one launch fewer per step
template <bool UPD>
__global__ __launch_bounds__(256) void k_adj_grad(FluidArgs a, AdjFluidArgs j, AdjPrevStep prev)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    double p[3] = {0.0, 0.0, 0.0};
    if (i < a.n_cells) {
        const float4 L = adj_grad_cell(a, j, i);
        if (UPD) adj_update_cell(a, j, prev.cf, i, L, prev.st[i], prev.res[i], p);
    }
    if (UPD) adj_force_partials(j, p);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_adj_rev_rows(const FluidArgs &a, float4 *rev_w, unsigned int *lone, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_rev_rows, dim3((a.n_cells + 255) / 256), dim3(256), 0, s, a, rev_w, lone);
    return hipGetLastError();
}

hipError_t launch_adj_update(const FluidArgs &a, const AdjFluidArgs &j, const float4 *st, const float4 *res,
                             hipStream_t s)
{
    const int blocks = (a.n_cells + 255) / 256;
    hipLaunchKernelGGL(k_adj_update, dim3(blocks), dim3(256), 0, s, a, j, st, res);
    return hipGetLastError();
}

hipError_t launch_adj_force_sum(const AdjFluidArgs &j, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_force_sum, dim3(1), dim3(256), 0, s, j);
    return hipGetLastError();
}

template <class L, int NT, int ADJ_CELLS>
static void launch_adj_flux_as(const FluidArgs &a, const AdjFluidArgs &j, const float4 *st, const float4 *grad, hipStream_t s)
{
    const size_t lds = sizeof(float4) * 8 * NT + sizeof(int) * (size_t)a.max_grad_slots;
    hipLaunchKernelGGL((k_adj_flux<L, NT, ADJ_CELLS>), dim3(a.n_tiles), dim3(NT), lds, s, a, j, st, grad);
}

template <class L>
static void launch_adj_flux_l(const FluidArgs &a, const AdjFluidArgs &j, const float4 *st, const float4 *grad,
                              int max_tile_cells, hipStream_t s)
{
    if (max_tile_cells <= 256) launch_adj_flux_as<L, 256, 1>(a, j, st, grad, s);
    else if (max_tile_cells <= 512) launch_adj_flux_as<L, 256, 2>(a, j, st, grad, s);
    else launch_adj_flux_as<L, 512, 2>(a, j, st, grad, s);
}

hipError_t launch_adj_flux(const FluidArgs &a, const AdjFluidArgs &j, const float4 *st, const float4 *grad,
                           int max_tile_cells, hipStream_t s)
{
    switch (a.lattice) {
    case LBFS_D3Q15: launch_adj_flux_l<D3Q15>(a, j, st, grad, max_tile_cells, s); break;
    case LBFS_D3Q19: launch_adj_flux_l<D3Q19>(a, j, st, grad, max_tile_cells, s); break;
    case LBFS_D2Q9: launch_adj_flux_l<D2Q9>(a, j, st, grad, max_tile_cells, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_adj_grad(const FluidArgs &a, const AdjFluidArgs &j, const AdjPrevStep *prev, hipStream_t s)
{
    const dim3 grid((a.n_cells + 255) / 256), blk(256);
    if (prev) hipLaunchKernelGGL(k_adj_grad<true>, grid, blk, 0, s, a, j, *prev);
    else hipLaunchKernelGGL(k_adj_grad<false>, grid, blk, 0, s, a, j, AdjPrevStep{});
    return hipGetLastError();
}

}  // namespace lbfs
