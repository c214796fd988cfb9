// Device helpers shared by the fluid kernels and their adjoints: gradient
// loads, compile-time lattice direction sums and the equilibrium deviation of
// one lattice point.
#pragma once

#include <hip/hip_runtime.h>

#include <utility>

#include "fluid_kernels.hpp"
#include "lattice.hpp"
#include "xcd.hpp"

namespace lbfs {

// Multiply-adds are written out in the forward fluid path (this header up to
// the reset at its end, and the kernels that use it): which products the
// compiler fuses would otherwise depend on the kernel they are inlined into,
// and the one-pass and two-pass steps give the same bits.
#pragma clang fp contract(off)

__device__ __forceinline__ float dot3(float ax, float ay, float az, float bx, float by, float bz)
{
    return fmaf(ax, bx, fmaf(ay, by, az * bz));
}

__device__ __forceinline__ void load_grad(const float4 *__restrict__ grad, int i, float g[12])
{
    const float4 a = grad[3 * (size_t)i], b = grad[3 * (size_t)i + 1], c = grad[3 * (size_t)i + 2];
    g[0] = a.x; g[1] = a.y; g[2] = a.z; g[3] = a.w;
    g[4] = b.x; g[5] = b.y; g[6] = b.z; g[7] = b.w;
    g[8] = c.x; g[9] = c.y; g[10] = c.z; g[11] = c.w;
}

// one tile-face record: unit normal and area from the area-weighted normal
struct FaceRec {
    float nx, ny, nz, A, dt;
    float3 d1, d2;  // owner and neighbour image centroid - face centroid
    bool general;   // takes the general reconstruction (pair_step): boundary faces and faces with a
                    // lattice direction in their own plane (DeviceLayout::fA)
};
// Length and inverse length from the hardware reciprocal square root and one
// Newton step each (9 instructions where the library's square root and division
// take 24 of a face's some 500); lengths whose square leaves the normal range
// take the library's.  The inverse is that of the rounded length, as a division
// gives it: from the root's own residual, length times normal is off by two
// roundings (3.0e-8 of the area vector against 1.7e-8), the same at every step.
__device__ __forceinline__ void length_and_inverse(float s, float &len, float &inv)
{
    if (__builtin_expect(s > 1e-36f && s < 1e36f, 1)) {
        const float y = __builtin_amdgcn_rsqf(s);
        const float l = s * y, h = 0.5f * y;
        const float e = fmaf(-l, l, s);
        len = fmaf(e, h, l);
        inv = fmaf(y, fmaf(-len, y, 1.0f), y);
    } else {
        len = sqrtf(s);
        inv = len > 0.0f ? 1.0f / len : 0.0f;
    }
}
// the record as stored
struct FaceRaw {
    float4 fa, fb;
    float2 fc;
};
__device__ __forceinline__ FaceRaw load_face_raw(const FluidArgs &a, int tf) { return {a.fA[tf], a.fB[tf], a.fC[tf]}; }
__device__ __forceinline__ FaceRec unpack_face(const FaceRaw &raw)
{
    const float4 fa = raw.fa;
    FaceRec r;
    r.d1 = make_float3(raw.fb.x, raw.fb.y, raw.fb.z);
    r.d2 = make_float3(raw.fb.w, raw.fc.x, raw.fc.y);
    float iA;
    length_and_inverse(dot3(fa.x, fa.y, fa.z, fa.x, fa.y, fa.z), r.A, iA);
    r.nx = fa.x * iA;
    r.ny = fa.y * iA;
    r.nz = fa.z * iA;
    r.dt = fabsf(fa.w);
    r.general = __float_as_int(fa.w) < 0;
    return r;
}

// cell id of a slot of tile T, and the neighbour of its face q: a cell id, or
// n_cells + the boundary face's number
__device__ __forceinline__ int slot_cell(const FluidArgs &a, const TileRec &T, int slot)
{
    return slot < T.nc ? T.c0 + slot : a.halo_ids[T.h0 + slot - T.nc];
}
__device__ __forceinline__ int face_neighbour(const FluidArgs &a, const TileRec &T, uint32_t gs, int q)
{
    return q < T.nif ? slot_cell(a, T, gs >> 16) : a.n_cells + a.tile_bc[T.b0 + q - T.nif];
}

template <class L>
constexpr bool opposite_pairs()
{
    for (int k = 1; k + 1 < L::Q; k += 2)
        if (L::ex[k] != -L::ex[k + 1] || L::ey[k] != -L::ey[k + 1] || L::ez[k] != -L::ez[k + 1]) return false;
    return (L::Q % 2) == 1;
}

// Sums over the components of a lattice direction with the zero components
// dropped at compile time: 0 * x cannot be folded away at run time (x may be
// infinite or NaN), so these are written out per direction.  -0.0f is the
// exact identity of addition, so the first term folds to itself.
template <int EX, int EY, int EZ>
__device__ __forceinline__ float edot(float a, float b, float c)
{
    float s = -0.0f;
    if constexpr (EX == 1) s += a; else if constexpr (EX == -1) s -= a;
    if constexpr (EY == 1) s += b; else if constexpr (EY == -1) s -= b;
    if constexpr (EZ == 1) s += c; else if constexpr (EZ == -1) s -= c;
    return s;
}

template <int E>
__device__ __forceinline__ void eacc(float &s, float v)
{
    if constexpr (E == 1) s += v; else if constexpr (E == -1) s -= v;
}

template <int E>
__device__ __forceinline__ void efma(float &s, float a, float b)
{
    if constexpr (E == 1) s = fmaf(a, b, s); else if constexpr (E == -1) s = fmaf(-a, b, s);
}

// equilibrium deviation g / w = drho + rho P of one lattice point with state
// ph = (drho, u, v, w): P = 3 e.u + 4.5 (e.u)^2 / gamma - 1.5 u.u / gamma
template <int EX, int EY, int EZ>
__device__ __forceinline__ float eq_point(const float ph[4], float rho0, float ig)
{
    const float eu = edot<EX, EY, EZ>(ph[1], ph[2], ph[3]);
    const float uu = dot3(ph[1], ph[2], ph[3], ph[1], ph[2], ph[3]);
    const float P = fmaf(eu, fmaf(4.5f * ig, eu, 3.0f), -1.5f * ig * uu);
    return fmaf(rho0 + ph[0], P, ph[0]);
}

struct FaceSums {
    float S0, S1x, S1y, S1z, Tx, Ty, Tz;
};

// one pair of opposite directions (e, -e): one e.n and one e.grad per side
template <class L, bool BAND, int K>
__device__ __forceinline__ void pair_step(FaceSums &f, const float po[4], const float pn[4], const float p0[4],
                                          const float go[12], const float gn[12], float nx, float ny, float nz,
                                          float bw, bool ghost, float rho0, float ig)
{
    constexpr int ex = L::ex[K], ey = L::ey[K], ez = L::ez[K];
    static_assert(L::w(K) == L::w(K + 1), "opposite directions carry equal weights");
    const float en = edot<ex, ey, ez>(nx, ny, nz);
    float pk[4], pb[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const float ego = edot<ex, ey, ez>(go[3 * v], go[3 * v + 1], go[3 * v + 2]);
        const float egn = edot<ex, ey, ez>(gn[3 * v], gn[3 * v + 1], gn[3 * v + 2]);
        if (!BAND) {
            // point x_f - e dt sits on the neighbour side when e.n < 0 (ties to the owner)
            pk[v] = en < 0.0f ? pn[v] - egn : po[v] - ego;
            pb[v] = en > 0.0f ? pn[v] + egn : po[v] + ego;
        } else {
            const float avg = ghost ? egn : 0.5f * (ego + egn);
            pk[v] = en > bw ? po[v] - ego : (en < -bw ? pn[v] - egn : p0[v] - avg);
            pb[v] = en < -bw ? po[v] + ego : (en > bw ? pn[v] + egn : p0[v] + avg);
        }
    }
    // (the first point's weight within the sum and the difference: 3 % less
    // rounding in the flux than with both products rounded)
    const float g = eq_point<ex, ey, ez>(pk, rho0, ig);
    const float gb = L::w(K) * eq_point<-ex, -ey, -ez>(pb, rho0, ig);
    const float gs = fmaf(L::w(K), g, gb), gd = fmaf(L::w(K), g, -gb);
    f.S0 += gs;
    eacc<ex>(f.S1x, gd); eacc<ey>(f.S1y, gd); eacc<ez>(f.S1z, gd);
    efma<ex>(f.Tx, en, gs); efma<ey>(f.Ty, en, gs); efma<ez>(f.Tz, en, gs);
}

// The same pair on a face whose lattice directions all lie clearly on one side
// (|e.n| beyond the tie and the tie band, DeviceLayout::fA): with s = sign(e.n)
// the point along s e comes from the owner side and its opposite from the
// neighbour side, so each point is one contraction and one multiply-add per
// variable where the selection of pair_step evaluates both sides for both
// points.  g / w = drho + 3/2 (rho / gamma) (eu (3 eu + 2 s gamma) - u.u) is the
// equilibrium deviation of eq_point (u.u summed by itself: its squares taken from
// the larger first term one by one are each rounded at that term's size, 8 % more
// error in a face's flux); the signs ride in the factors of the sums: about 46
// operations a diagonal pair where pair_step takes 63.  128x64x64 channel, D3Q19, 8x8x8 tiles: face pass 34.8 -> 30.6 us,
// fused pass 45.9 -> 42.9 us (both were vector-bound, now memory).  pair_step
// stays for the faces whose points may come from either side.
template <class L, int K>
__device__ __forceinline__ void pair_fast(FaceSums &f, const float po[4], const float pn[4], const float go[12],
                                          const float gn[12], float nx, float ny, float nz, float dt, float rho15,
                                          float ig15, float gam2)
{
    constexpr int ex = L::ex[K], ey = L::ey[K], ez = L::ez[K];
    constexpr float w = L::w(K);
    const float en = edot<ex, ey, ez>(nx, ny, nz);
    const float sdt = copysignf(dt, en), sgam = copysignf(gam2, en), s = copysignf(1.0f, en);
    float qo[4], qn[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        qo[v] = fmaf(-sdt, edot<ex, ey, ez>(go[3 * v], go[3 * v + 1], go[3 * v + 2]), po[v]);
        qn[v] = fmaf(sdt, edot<ex, ey, ez>(gn[3 * v], gn[3 * v + 1], gn[3 * v + 2]), pn[v]);
    }
    const float euo = edot<ex, ey, ez>(qo[1], qo[2], qo[3]), eun = edot<ex, ey, ez>(qn[1], qn[2], qn[3]);
    const float Bo = fmaf(euo, fmaf(3.0f, euo, sgam), -dot3(qo[1], qo[2], qo[3], qo[1], qo[2], qo[3]));
    const float Bn = fmaf(eun, fmaf(3.0f, eun, -sgam), -dot3(qn[1], qn[2], qn[3], qn[1], qn[2], qn[3]));
    const float g_o = fmaf(fmaf(ig15, qo[0], rho15), Bo, qo[0]), g_n = fmaf(fmaf(ig15, qn[0], rho15), Bn, qn[0]);
    // (weighted as in pair_step; a product w e.n for the second moments would be
    // off by the same rounding at every step)
    const float gb = w * g_n, gs = fmaf(w, g_o, gb), gd = fmaf(w, g_o, -gb);
    f.S0 += gs;
    efma<ex>(f.S1x, s, gd); efma<ey>(f.S1y, s, gd); efma<ez>(f.S1z, s, gd);
    efma<ex>(f.Tx, en, gs); efma<ey>(f.Ty, en, gs); efma<ez>(f.Tz, en, gs);
}

template <class L, int... P>
__device__ __forceinline__ void all_pairs_fast(std::integer_sequence<int, P...>, FaceSums &f, const float po[4],
                                               const float pn[4], const float go[12], const float gn[12], float nx,
                                               float ny, float nz, float dt, float rho15, float ig15, float gam2)
{
    (pair_fast<L, 2 * P + 1>(f, po, pn, go, gn, nx, ny, nz, dt, rho15, ig15, gam2), ...);
}

template <class L, bool BAND, int... P>
__device__ __forceinline__ void all_pairs(std::integer_sequence<int, P...>, FaceSums &f, const float po[4],
                                          const float pn[4], const float p0[4], const float go[12],
                                          const float gn[12], float nx, float ny, float nz, float bw, bool ghost,
                                          float rho0, float ig)
{
    (pair_step<L, BAND, 2 * P + 1>(f, po, pn, p0, go, gn, nx, ny, nz, bw, ghost, rho0, ig), ...);
}

#pragma clang fp contract(fast)

}  // namespace lbfs
