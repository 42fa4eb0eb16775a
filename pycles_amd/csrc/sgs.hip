// Kinematics, Smagorinsky SGS closure and second-order diffusion.
//
//   Kinematics.update                Kinematics.pyx:41-58, kinematics.h:6-138
//   Smagorinsky.update               SGS.pyx:146-152, sgs.h:4-19
//   ScalarDiffusion.update           ScalarDiffusion.pyx:76-119,
//                                    scalar_diffusion.h:6-58, flux_divergence.h:4-32
//   MomentumDiffusion.update         MomentumDiffusion.pyx:44-66,
//                                    momentum_diffusion.h:5-118, flux_divergence.h:34-80
//
// Two kernels per stage, both with one thread per column marching a chunk of
// levels:
//  * sgs_kernel: the strain-rate magnitude from the velocity gradients at the
//    staggered points around the cell, then the eddy viscosity and
//    diffusivity.  The reference stores the nine gradients and the nine
//    strain-rate components (18 field passes written and read again); here
//    they are formed from the velocities in registers and only |S|, nu and D
//    are written.
//  * diffusion_kernel: for each cell, the diffusive fluxes of s and qt on
//    its six faces and the nine stress fluxes on the faces the momentum
//    divergence needs (each flux formed by both cells sharing the face, with
//    no flux array; the lower z faces are carried from the level below), the
//    divergences accumulated into the tendencies in the reference's
//    per-variable order, and the entropy source of the dissipation.
// A wavefront is 64 columns of one row, so every row address is scalar and
// every neighbour along x is one 32-bit lane offset formed before the march;
// a level's loads (22 and 47, in-cache re-reads of neighbours included) are
// issued together ahead of its arithmetic, and the values that the next level
// shares (its own level's centre values, its lower faces' strains and
// fluxes) stay in registers.  One thread per cell with a wrapped 64-bit
// offset per load spent its time on that address arithmetic (about 90 and
// 200 loads a cell).
// Bound: HBM (7 and 19 field passes) on large grids, 256 x 256 x 75 FP32: 47
// us (3.2 TB/s) and 93 us (4.0 TB/s) against 193 and 335 us before; latency on
// small ones, 64 x 64 x 75 FP64: 13 and 29 us against 23 and 50.
// x and y are periodic by index wrap; z reads the stored ghost levels.  In
// FP64 every expression follows the reference's operation order.
#include "common.h"

extern int pycles_check_dims(const pycles_dims *d);

namespace {

// z chunks of n levels: until the grid holds 8 wavefronts per SIMD (what a CU
// can hold), chunks of at least 4 (each chunk forms one level of faces again:
// a quarter more loads at 4, which only grids too small to fill the chip pay).
static ZSplit sgs_zsplit(const Geo &g, int n) {
    const long long cols = (long long)((g.nx + 63) / 64) * ((g.ny + 3) / 4);
    int want = 1;
    while (cols * want < 2048 && n / (want * 2) >= 4) want *= 2;
    return zsplit_ceil(n, want);
}

// The columns around a thread's own: lane offsets along x, scalar row offsets
// along y (both wrapped), and loads of a field at level offset `lev`.
struct Nbr {
    unsigned c, m1, m2, p1;      // i, i-1, i-2, i+1
    long long r, rm1, rm2, rp1;  // rows j, j-1, j-2, j+1, times nx
};
__device__ __forceinline__ Nbr neighbours(const Geo &g, int i, int j) {
    Nbr n;
    n.c = i;
    n.m1 = i >= 1 ? i - 1 : i - 1 + g.nx;
    n.m2 = i >= 2 ? i - 2 : (2 * g.nx + i - 2) % g.nx;
    n.p1 = i + 1 < g.nx ? i + 1 : i + 1 - g.nx;
    n.r = (long long)j * g.nx;
    n.rm1 = (long long)(j >= 1 ? j - 1 : j - 1 + g.ny) * g.nx;
    n.rm2 = (long long)(j >= 2 ? j - 2 : (2 * g.ny + j - 2) % g.ny) * g.nx;
    n.rp1 = (long long)(j + 1 < g.ny ? j + 1 : j + 1 - g.ny) * g.nx;
    return n;
}
// f at scalar element offset `row` (level and row) and lane offset i
template <typename T> __device__ __forceinline__ T at(const T *f, long long row, unsigned i) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(f + row) + (size_t)(i * (unsigned)sizeof(T)));
}
template <typename T> __device__ __forceinline__ T nt_at(const T *f, long long row, unsigned i) {
    return __builtin_nontemporal_load(
        reinterpret_cast<const T *>(reinterpret_cast<const char *>(f + row) + (size_t)(i * (unsigned)sizeof(T))));
}
template <typename T> __device__ __forceinline__ void nt_put(T *f, long long row, unsigned i, T v) {
    __builtin_nontemporal_store(v, reinterpret_cast<T *>(reinterpret_cast<char *>(f + row) + (size_t)(i * (unsigned)sizeof(T))));
}

template <typename T>
struct Vel {
    const T *v[3];
};

// Strain rate of an off-diagonal pair (kinematics.h:54-62) from its two
// velocity differences and inverse spacings.  A diagonal one,
// 0.5 (g + g), is its gradient g.
template <typename T> __device__ __forceinline__ T strain2(T da, T ia, T db, T ib) {
    return T(0.5) * (da * ia + db * ib);
}

template <typename T>
__global__ __launch_bounds__(256) void sgs_kernel(Geo g, Vel<T> vel, const T *bvf, T *smag_out, T *visc, T *diff,
                                                  double csd2, double prt, int kchunk) {
    const uint3 tile = xcd_tile<1>();
    const int il = tile.x * 64 + threadIdx.x;
    const int j = __builtin_amdgcn_readfirstlane(tile.y * 4 + threadIdx.y);
    if (j >= g.ny) return;
    const bool own = il < g.nx;
    const Nbr n = neighbours(g, own ? il : g.nx - 1, j);
    const T *u = vel.v[0], *v = vel.v[1], *w = vel.v[2];
    const T xi = (T)g.dxi[0], yi = (T)g.dxi[1], zi = (T)g.dxi[2];
    const long long P = g.plane;
    const int k0 = tile.z * kchunk;
    const int k1 = min(k0 + kchunk, g.nzg);
    // the reference computes |S| on [1, nlg-1) in z (0 elsewhere, and with it
    // nu and D)
    for (int e = 0; e < 2; ++e) {
        const int k = e ? g.nzg - 1 : 0;
        if (own && k >= k0 && k < k1) {
            smag_out[k * P + n.r + n.c] = T(0);
            visc[k * P + n.r + n.c] = T(0);
            diff[k * P + n.r + n.c] = T(0);
        }
    }
    const int ks = max(k0, 1), ke = min(k1, g.nzg - 1);
    if (ks >= ke) return;
    // carried: the centre values of level k and of w at k-1, and the strains
    // S02 at (i, i-1) and S12 at (j, j-1) of level k-1
    T uc, um, vc, vm, wc, wp, a02, b02, a12, b12;
    {
        const long long o = (ks - 1) * P;
        const T u0 = at(u, o + n.r, n.c), u1 = at(u, o + n.r, n.m1);
        const T v0 = at(v, o + n.r, n.c), v1 = at(v, o + n.rm1, n.c);
        const T w0 = at(w, o + n.r, n.c), wm = at(w, o + n.r, n.m1), wx = at(w, o + n.r, n.p1);
        const T wj = at(w, o + n.rm1, n.c), wy = at(w, o + n.rp1, n.c);
        uc = at(u, o + P + n.r, n.c);
        um = at(u, o + P + n.r, n.m1);
        vc = at(v, o + P + n.r, n.c);
        vm = at(v, o + P + n.rm1, n.c);
        wc = at(w, o + P + n.r, n.c);
        wp = w0;
        a02 = strain2(uc - u0, zi, wx - w0, xi);
        b02 = strain2(um - u1, zi, w0 - wm, xi);
        a12 = strain2(vc - v0, zi, wy - w0, yi);
        b12 = strain2(vm - v1, zi, w0 - wj, yi);
    }
    for (int kk = ks; kk < ke; ++kk) {
        const int k = __builtin_amdgcn_readfirstlane(kk);
        const long long o = k * P, c = o + n.r, d = o + n.rm1, e = o + n.rp1;
        const T um2 = at(u, c, n.m2), up = at(u, c, n.p1);
        const T ue = at(u, e, n.c), uem = at(u, e, n.m1), ud = at(u, d, n.c), udm = at(u, d, n.m1);
        const T vm2 = at(v, o + n.rm2, n.c), vp = at(v, e, n.c);
        const T vx = at(v, c, n.p1), vw = at(v, c, n.m1), vdx = at(v, d, n.p1), vdw = at(v, d, n.m1);
        const T wx = at(w, c, n.p1), wm = at(w, c, n.m1), wy = at(w, e, n.c), wj = at(w, d, n.c);
        const T un = at(u, c + P, n.c), unm = at(u, c + P, n.m1);
        const T vn = at(v, c + P, n.c), vnm = at(v, d + P, n.c);
        const T wn = at(w, c + P, n.c);
        const T n2 = nt_at(bvf, c, n.c);
        // on-diagonal components at ijk - s_d (kinematics.h:96-108)
        T m = T(0);
        const T g0 = (uc - um) * xi, g1 = (vc - vm) * yi, g2 = (wc - wp) * zi;
        m += g0 * g0;
        m += g1 * g1;
        m += g2 * g2;
        // the (v1, d) pairs with d from v1 to 2 (kinematics.h:111-128): four
        // points ijk, ijk - s_v1, ijk - s_d, ijk - s_d - s_v1
        T si = T(0.25) * ((up - uc) * xi + g0 + g0 + (um - um2) * xi);
        m += T(2.0) * si * si;
        si = T(0.25) * (strain2(ue - uc, yi, vx - vc, xi) + strain2(uem - um, yi, vc - vw, xi) +
                        strain2(uc - ud, yi, vdx - vm, xi) + strain2(um - udm, yi, vm - vdw, xi));
        m += T(2.0) * si * si;
        const T s02 = strain2(un - uc, zi, wx - wc, xi), t02 = strain2(unm - um, zi, wc - wm, xi);
        si = T(0.25) * (s02 + t02 + a02 + b02);
        m += T(2.0) * si * si;
        si = T(0.25) * ((vp - vc) * yi + g1 + g1 + (vm - vm2) * yi);
        m += T(2.0) * si * si;
        const T s12 = strain2(vn - vc, zi, wy - wc, yi), t12 = strain2(vnm - vm, zi, wc - wj, yi);
        si = T(0.25) * (s12 + t12 + a12 + b12);
        m += T(2.0) * si * si;
        const T S = sqrt(T(2.0) * m);
        // smagorinsky_update (sgs.h:4-19); csd2 = cs*cs*delta*delta as the
        // reference evaluates it left to right
        T nu = (T)csd2 * S;
        if (n2 > T(0)) {
            const T fb = sqrt(fmax(T(1.0) - n2 / ((T)prt * S * S), T(0.0)));
            nu = nu * fb;
        }
        if (own) {
            nt_put(smag_out, c, n.c, S);
            nt_put(visc, c, n.c, nu);
            nt_put(diff, c, n.c, nu / (T)prt);
        }
        a02 = s02;
        b02 = t02;
        a12 = s12;
        b12 = t12;
        uc = un;
        um = unm;
        vc = vn;
        vm = vnm;
        wp = wc;
        wc = wn;
    }
}

template <typename T>
struct DiffArgs {
    Vel<T> vel;
    T *tv[3];
    const T *phi[2];
    T *tphi[2];
    const T *visc, *diff, *smag, *temp;
};
// Profiles as restricted kernel arguments: read through the scalar cache
// (the field stores cannot alias them).
#define DIFF_PROFILES                                                                                       \
    const double *__restrict__ rho0, const double *__restrict__ rho0_half, const double *__restrict__ alpha0, \
        const double *__restrict__ alpha0_half, const double *__restrict__ base0, const double *__restrict__ base1

// Stress flux (compute_diffusive_flux_m, momentum_diffusion.h:5-88) from its
// strain rate, viscosity (the sum of the four corner values for an
// off-diagonal pair, in the reference's order) and density.
template <typename T> __device__ __forceinline__ T stress(T S, T nu, T rho) { return T(-2.0) * S * nu * rho; }
template <typename T> __device__ __forceinline__ T corner(T a, T b, T c, T d) { return T(0.25) * (a + b + c + d); }
// Scalar flux -interp_2(D[p], D[p+s]) (phi[p+s] - phi[p]) rho dxi
// (scalar_diffusion.h:21-43)
template <typename T> __device__ __forceinline__ T scalar_flux(T Dp, T Dq, T dphi, T rho, T dxi) {
    const T K = T(0.5) * (Dp + Dq);
    return T(-1.0) * K * dphi * rho * dxi;
}

// NSC: scalars diffused (0: none); MOM: the stress divergence; SRC: the
// entropy source into the first scalar's tendency.
template <typename T, int NSC, bool MOM, bool SRC>
__global__ __launch_bounds__(256) void diffusion_kernel(Geo g, DiffArgs<T> a, DIFF_PROFILES, int kchunk) {
    const uint3 tile = xcd_tile<1>();
    const int il = tile.x * 64 + threadIdx.x;
    const int j = __builtin_amdgcn_readfirstlane(tile.y * 4 + threadIdx.y);
    if (j >= g.ny) return;
    const bool own = il < g.nx;
    const Nbr n = neighbours(g, own ? il : g.nx - 1, j);
    const T *u = a.vel.v[0], *v = a.vel.v[1], *w = a.vel.v[2];
    const T xi = (T)g.dxi[0], yi = (T)g.dxi[1], zi = (T)g.dxi[2];
    const T sx = (T)(1.0 / g.dx[0]), sy = (T)(1.0 / g.dx[1]), sz = (T)(1.0 / g.dx[2]);
    const long long P = g.plane;
    const int k0 = g.gw + tile.z * kchunk;
    const int k1 = min(k0 + kchunk, g.nz + g.gw);
    const double *base[2] = {base0, base1};
    // z difference of a scalar; FP32 deviations from the level profile take
    // the profile's difference in FP64
    auto dz_phi = [&](int sc, T hi, T lo, int kp) {
        if (sizeof(T) == 4 && base[sc]) return (T)((base[sc][kp + 1] - base[sc][kp]) + (double)(hi - lo));
        return hi - lo;
    };
    // carried: centre values of level k, and the fluxes of the face below
    T uc = 0, um = 0, vc = 0, vm = 0, wc = 0, nc = 0, nm = 0, nx_ = 0, nj = 0, ny_ = 0, Dc = 0;
    T f02 = 0, f12 = 0, f22 = 0, pc[2] = {}, fz[2] = {};
    {
        const long long c = k0 * P + n.r, d = k0 * P + n.rm1, e = k0 * P + n.rp1;
        if (MOM) {
            uc = at(u, c, n.c);
            um = at(u, c, n.m1);
            vc = at(v, c, n.c);
            vm = at(v, d, n.c);
            wc = at(w, c, n.c);
            nc = at(a.visc, c, n.c);
            nm = at(a.visc, c, n.m1);
            nx_ = at(a.visc, c, n.p1);
            nj = at(a.visc, d, n.c);
            ny_ = at(a.visc, e, n.c);
        } else if (SRC) {
            nc = at(a.visc, c, n.c);
        }
        if (NSC > 0) Dc = at(a.diff, c, n.c);
#pragma unroll
        for (int sc = 0; sc < NSC; ++sc) pc[sc] = at(a.phi[sc], c, n.c);
        // the face below the chunk (zero on the surface face, k0 = gw)
        if (k0 > g.gw) {
            const int kp = k0 - 1;
            if (MOM) {
                const T w0 = at(w, c - P, n.c), wx = at(w, c - P, n.p1), wy = at(w, e - P, n.c);
                const T u0 = at(u, c - P, n.c), v0 = at(v, c - P, n.c);
                const T q0 = at(a.visc, c - P, n.c), qx = at(a.visc, c - P, n.p1), qy = at(a.visc, e - P, n.c);
                const T r0 = (T)rho0[kp];
                f02 = stress(strain2(uc - u0, zi, wx - w0, xi), corner(q0, qx, nc, nx_), r0);
                f12 = stress(strain2(vc - v0, zi, wy - w0, yi), corner(q0, qy, nc, ny_), r0);
                f22 = stress((wc - w0) * zi, nc, (T)rho0_half[kp + 1]);
            }
#pragma unroll
            for (int sc = 0; sc < NSC; ++sc)
                fz[sc] = scalar_flux(at(a.diff, c - P, n.c), Dc, dz_phi(sc, pc[sc], at(a.phi[sc], c - P, n.c), kp),
                                     (T)rho0[kp], sz);
        }
    }
    for (int kk = k0; kk < k1; ++kk) {
        const int k = __builtin_amdgcn_readfirstlane(kk);
        const long long c = k * P + n.r, d = k * P + n.rm1, e = k * P + n.rp1;
        // this level's loads, all ahead of its arithmetic and stores
        T up = 0, ue = 0, uem = 0, ud = 0, vp = 0, vx = 0, vdx = 0, vw = 0, wm = 0, wx = 0, wj = 0, wy = 0;
        T nxy = 0, ndx = 0, nwy = 0, un = 0, unm = 0, vn = 0, vnm = 0, wn = 0;
        T qn = 0, qnm = 0, qnx = 0, qnj = 0, qny = 0;
        T Dm = 0, Dx = 0, Dj = 0, Dy = 0, Dn = 0, pm[2] = {}, px[2] = {}, pj[2] = {}, py[2] = {}, pn[2] = {};
        T tv[3] = {}, tp[2] = {}, S = 0, Tt = 0;
        if (NSC > 0) {
            Dm = at(a.diff, c, n.m1);
            Dx = at(a.diff, c, n.p1);
            Dj = at(a.diff, d, n.c);
            Dy = at(a.diff, e, n.c);
            Dn = at(a.diff, c + P, n.c);
        }
#pragma unroll
        for (int sc = 0; sc < NSC; ++sc) {
            pm[sc] = at(a.phi[sc], c, n.m1);
            px[sc] = at(a.phi[sc], c, n.p1);
            pj[sc] = at(a.phi[sc], d, n.c);
            py[sc] = at(a.phi[sc], e, n.c);
            pn[sc] = at(a.phi[sc], c + P, n.c);
            tp[sc] = nt_at(a.tphi[sc], c, n.c);
        }
        if (SRC) {
            if (NSC == 0) tp[0] = nt_at(a.tphi[0], c, n.c);
            S = nt_at(a.smag, c, n.c);
            Tt = nt_at(a.temp, c, n.c);
        }
        if (MOM) {
            up = at(u, c, n.p1);
            ue = at(u, e, n.c);
            uem = at(u, e, n.m1);
            ud = at(u, d, n.c);
            vp = at(v, e, n.c);
            vx = at(v, c, n.p1);
            vdx = at(v, d, n.p1);
            vw = at(v, c, n.m1);
            wm = at(w, c, n.m1);
            wx = at(w, c, n.p1);
            wj = at(w, d, n.c);
            wy = at(w, e, n.c);
            nxy = at(a.visc, e, n.p1);
            ndx = at(a.visc, d, n.p1);
            nwy = at(a.visc, e, n.m1);
            un = at(u, c + P, n.c);
            unm = at(u, c + P, n.m1);
            vn = at(v, c + P, n.c);
            vnm = at(v, d + P, n.c);
            wn = at(w, c + P, n.c);
            qn = at(a.visc, c + P, n.c);
            qnm = at(a.visc, c + P, n.m1);
            qnx = at(a.visc, c + P, n.p1);
            qnj = at(a.visc, d + P, n.c);
            qny = at(a.visc, e + P, n.c);
#pragma unroll
            for (int q = 0; q < 3; ++q) tv[q] = nt_at(a.tv[q], c, n.c);
        } else if (SRC) {
            qn = at(a.visc, c + P, n.c);
        }
        const T rh = (T)rho0_half[k], r0 = (T)rho0[k];
        const T ah = (T)alpha0_half[k], af = (T)alpha0[k];
        // ScalarDiffusion: each scalar, directions x, y, z (flux_divergence.h:4-32)
#pragma unroll
        for (int sc = 0; sc < NSC; ++sc) {
            T t = tp[sc];
            t -= ah * (scalar_flux(Dc, Dx, px[sc] - pc[sc], rh, sx) - scalar_flux(Dm, Dc, pc[sc] - pm[sc], rh, sx)) * xi;
            t -= ah * (scalar_flux(Dc, Dy, py[sc] - pc[sc], rh, sy) - scalar_flux(Dj, Dc, pc[sc] - pj[sc], rh, sy)) * yi;
            const T f = scalar_flux(Dc, Dn, dz_phi(sc, pn[sc], pc[sc], k), r0, sz);
            t -= ah * (f - fz[sc]) * zi;
            fz[sc] = f;
            tp[sc] = t;
        }
        // MomentumDiffusion: component i1, directions i2 (flux_divergence.h:34-80)
        if (MOM) {
            const T rn = (T)rho0_half[k + 1];
            const T s01 = strain2(ue - uc, yi, vx - vc, xi);
            const T s02 = strain2(un - uc, zi, wx - wc, xi), s12 = strain2(vn - vc, zi, wy - wc, yi);
            T t = tv[0];
            t -= ah * (stress((up - uc) * xi, nx_, rh) - stress((uc - um) * xi, nc, rh)) * xi;
            t -= ah * (stress(s01, corner(nc, nx_, ny_, nxy), rh) -
                       stress(strain2(uc - ud, yi, vdx - vm, xi), corner(nj, ndx, nc, nx_), rh)) * yi;
            T f = stress(s02, corner(nc, nx_, qn, qnx), r0);
            t -= ah * (f - f02) * zi;
            f02 = f;
            tv[0] = t;
            t = tv[1];
            t -= ah * (stress(s01, corner(nc, ny_, nx_, nxy), rh) -
                       stress(strain2(uem - um, yi, vc - vw, xi), corner(nm, nwy, nc, ny_), rh)) * xi;
            t -= ah * (stress((vp - vc) * yi, ny_, rh) - stress((vc - vm) * yi, nc, rh)) * yi;
            f = stress(s12, corner(nc, ny_, qn, qny), r0);
            t -= ah * (f - f12) * zi;
            f12 = f;
            tv[1] = t;
            t = tv[2];
            t -= af * (stress(s02, corner(nc, qn, nx_, qnx), r0) -
                       stress(strain2(unm - um, zi, wc - wm, xi), corner(nm, qnm, nc, qn), r0)) * xi;
            t -= af * (stress(s12, corner(nc, qn, ny_, qny), r0) -
                       stress(strain2(vnm - vm, zi, wc - wj, yi), corner(nj, qnj, nc, qn), r0)) * yi;
            f = stress((wn - wc) * zi, qn, rn);
            t -= af * (f - f22) * zi;
            f22 = f;
            tv[2] = t;
        }
        // compute_entropy_source (momentum_diffusion.h:90-118) into the s tendency
        if (SRC) tp[0] += S * S * nc / Tt;
        if (own) {
#pragma unroll
            for (int sc = 0; sc < NSC; ++sc) nt_put(a.tphi[sc], c, n.c, tp[sc]);
            if (SRC && NSC == 0) nt_put(a.tphi[0], c, n.c, tp[0]);
            if (MOM) {
#pragma unroll
                for (int q = 0; q < 3; ++q) nt_put(a.tv[q], c, n.c, tv[q]);
            }
        }
        uc = un;
        um = unm;
        vc = vn;
        vm = vnm;
        wc = wn;
        nc = qn;
        nm = qnm;
        nx_ = qnx;
        nj = qnj;
        ny_ = qny;
        Dc = Dn;
#pragma unroll
        for (int sc = 0; sc < NSC; ++sc) pc[sc] = pn[sc];
    }
}

}  // namespace

extern "C" int pycles_sgs_smagorinsky(const pycles_dims *dims, const void *const vel[3], const void *bvf, double cs,
                                      double prt, void *strain_mag, void *visc, void *diff, int precision,
                                      void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!vel || !vel[0] || !vel[1] || !vel[2] || !bvf || !strain_mag || !visc || !diff) {
        pycles_set_error("sgs_smagorinsky: NULL argument");
        return PYCLES_ERR_ARG;
    }
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("sgs_smagorinsky: bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    if (!(prt > 0.0)) {
        pycles_set_error("sgs_smagorinsky: the turbulent Prandtl number must be positive");
        return PYCLES_ERR_ARG;
    }
    const Geo g = make_geo(dims);
    // sgs.h:7 on the host: cbrt and the product in the reference's order
    const double delta = cbrt(g.dx[0] * g.dx[1] * g.dx[2]);
    const double csd2 = cs * cs * delta * delta;
    const ZSplit zs = sgs_zsplit(g, g.nzg);
    const dim3 grid((g.nx + 63) / 64, (g.ny + 3) / 4, zs.nch), blk(64, 4);
    hipStream_t st = (hipStream_t)stream;
    if (precision == PYCLES_F64) {
        Vel<double> v{{(const double *)vel[0], (const double *)vel[1], (const double *)vel[2]}};
        hipLaunchKernelGGL(sgs_kernel<double>, grid, blk, 0, st, g, v, (const double *)bvf, (double *)strain_mag,
                           (double *)visc, (double *)diff, csd2, prt, zs.len);
    } else {
        Vel<float> v{{(const float *)vel[0], (const float *)vel[1], (const float *)vel[2]}};
        hipLaunchKernelGGL(sgs_kernel<float>, grid, blk, 0, st, g, v, (const float *)bvf, (float *)strain_mag,
                           (float *)visc, (float *)diff, csd2, prt, zs.len);
    }
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

template <typename T>
static int launch_diffusion(const Geo &g, const pycles_ref *ref, const void *const vel[3], void *const tend_vel[3],
                            int nscal, const void *const *scal, void *const *tend_scal,
                            const pycles_scalar_base *base, const void *visc, const void *diff,
                            const void *strain_mag, const void *T_, int flags, hipStream_t st) {
    DiffArgs<T> a;
    for (int q = 0; q < 3; ++q) {
        a.vel.v[q] = (const T *)vel[q];
        a.tv[q] = tend_vel ? (T *)tend_vel[q] : nullptr;
    }
    for (int q = 0; q < 2; ++q) {
        a.phi[q] = q < nscal ? (const T *)scal[q] : nullptr;
        a.tphi[q] = q < nscal ? (T *)tend_scal[q] : nullptr;
    }
    a.visc = (const T *)visc;
    a.diff = (const T *)diff;
    a.smag = (const T *)strain_mag;
    a.temp = (const T *)T_;
    const double *b0 = (sizeof(T) == 4 && base && nscal > 0) ? base->base[0] : nullptr;
    const double *b1 = (sizeof(T) == 4 && base && nscal > 1) ? base->base[1] : nullptr;
    const ZSplit zs = sgs_zsplit(g, g.nz);
    const dim3 grid((g.nx + 63) / 64, (g.ny + 3) / 4, zs.nch), blk(64, 4);
    const int nsc = (flags & PYCLES_DIFF_SCALARS) ? nscal : 0;
    const bool mom = flags & PYCLES_DIFF_MOMENTUM, src = flags & PYCLES_DIFF_ENTROPY_SOURCE;
#define DIFF_LAUNCH(NSC_, MOM_, SRC_)                                                                          \
    if (nsc == NSC_ && mom == MOM_ && src == SRC_)                                                             \
        hipLaunchKernelGGL((diffusion_kernel<T, NSC_, MOM_, SRC_>), grid, blk, 0, st, g, a, ref->rho0,         \
                           ref->rho0_half, ref->alpha0, ref->alpha0_half, b0, b1, zs.len);
#define DIFF_LAUNCH_SC(MOM_, SRC_) DIFF_LAUNCH(0, MOM_, SRC_) DIFF_LAUNCH(1, MOM_, SRC_) DIFF_LAUNCH(2, MOM_, SRC_)
    DIFF_LAUNCH_SC(false, true)
    DIFF_LAUNCH_SC(true, false)
    DIFF_LAUNCH_SC(true, true)
    DIFF_LAUNCH(1, false, false)
    DIFF_LAUNCH(2, false, false)
#undef DIFF_LAUNCH_SC
#undef DIFF_LAUNCH
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

extern "C" int pycles_diffusion(const pycles_dims *dims, const pycles_ref *ref, const void *const vel[3],
                                void *const tend_vel[3], int nscal, const void *const *scal, void *const *tend_scal,
                                const pycles_scalar_base *base, const void *visc, const void *diff,
                                const void *strain_mag, const void *temperature, int flags, int precision,
                                void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    const int known = PYCLES_DIFF_SCALARS | PYCLES_DIFF_MOMENTUM | PYCLES_DIFF_ENTROPY_SOURCE;
    if ((flags & ~known) || !flags) {
        pycles_set_error("diffusion: flags %d", flags);
        return PYCLES_ERR_ARG;
    }
    if (!ref || !ref->rho0 || !ref->rho0_half || !ref->alpha0 || !ref->alpha0_half || !vel || !vel[0] || !vel[1] ||
        !vel[2]) {
        pycles_set_error("diffusion: NULL reference profile or velocity");
        return PYCLES_ERR_ARG;
    }
    if (nscal < 0 || nscal > 2 || (nscal > 0 && (!scal || !tend_scal))) {
        pycles_set_error("diffusion: nscal = %d", nscal);
        return PYCLES_ERR_ARG;
    }
    for (int q = 0; q < nscal; ++q)
        if (!scal[q] || !tend_scal[q]) {
            pycles_set_error("diffusion: NULL scalar %d", q);
            return PYCLES_ERR_ARG;
        }
    if ((flags & PYCLES_DIFF_SCALARS) && (!diff || nscal == 0)) {
        pycles_set_error("diffusion: scalar diffusion needs the diffusivity and a scalar");
        return PYCLES_ERR_ARG;
    }
    if ((flags & PYCLES_DIFF_MOMENTUM) && (!tend_vel || !tend_vel[0] || !tend_vel[1] || !tend_vel[2] || !visc)) {
        pycles_set_error("diffusion: momentum diffusion needs the three tendencies and the viscosity");
        return PYCLES_ERR_ARG;
    }
    if ((flags & PYCLES_DIFF_ENTROPY_SOURCE) && (nscal == 0 || !strain_mag || !temperature || !visc)) {
        pycles_set_error("diffusion: the entropy source needs s, |S|, the viscosity and T");
        return PYCLES_ERR_ARG;
    }
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("diffusion: bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    if (dims->gw < 2) {
        pycles_set_error("diffusion: gw must be at least 2");
        return PYCLES_ERR_ARG;
    }
    const Geo g = make_geo(dims);
    hipStream_t st = (hipStream_t)stream;
    if (precision == PYCLES_F64)
        return launch_diffusion<double>(g, ref, vel, tend_vel, nscal, scal, tend_scal, base, visc, diff, strain_mag,
                                        temperature, flags, st);
    return launch_diffusion<float>(g, ref, vel, tend_vel, nscal, scal, tend_scal, base, visc, diff, strain_mag,
                                   temperature, flags, st);
}
