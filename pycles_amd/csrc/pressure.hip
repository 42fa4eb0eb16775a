// Anelastic pressure projection on one GPU (whole domain).
//
// The reference (PressureSolver.pyx:38-81, PressureFFTParallel.pyx:150-220)
// removes the level mean of w, forms div(rho0 u) with second-order
// differences, takes complex FFTs of the real divergence along x then y
// (scipy.fftpack.fft), solves one real tridiagonal system per (kx, ky) for the
// real and imaginary parts (SparseSolvers.pyx:24-43), zeroes the (0,0) mode,
// inverts the FFTs, keeps the real part, fills the pressure halo and
// subtracts grad p from u, v, w.  MPI pencil transposes move data between the
// FFT and solve directions.
//
// Here the domain is whole on one GPU, so there are no transposes: the
// divergence of a row is computed and Fourier-transformed in LDS in one
// kernel, and because the input is real only the half spectrum
// kx = 0..nx/2 is kept (the other half is its complex conjugate, so the
// solves there are redundant).  The y transform, the per-column Thomas
// sweep and the inverse transforms each take one pass over the half
// spectrum [nz][ny][nx/2+1] (kx fastest).  The Thomas recurrence runs in FP64
// in both precisions (its low-wavenumber systems are the ill-conditioned
// ones).  The correction marches each column in z so it can also fill the z
// ghost levels of u, v, w and reduce the CFL number.
#include <math.h>
#include <string.h>

#include <vector>

#include "common.h"

extern int pycles_check_dims(const pycles_dims *d);
// Partial sums of every level, MEAN_SPLITS per level (timestep.hip)
constexpr int MEAN_SPLITS = 16;
extern int pycles_level_partials(const Geo &g, const void *field, double *partial, int precision, hipStream_t st);

struct pycles_pressure_plan {
    Geo g;
    int precision;
    int nxh;
    int nxp;         // row stride of the spectrum: nxh rounded up to 16 (128-byte rows in FP32)
    int gx;          // kx columns per y-FFT block
    void *mem;       // the one allocation that the arrays below lie in
    void *spec;      // [nz][ny][nxp] complex, field precision (columns nxh..nxp-1 unused)
    double *ck;      // Thomas segment carries: [nz / S][3][ny][nxp] (S levels per segment)
    double *pm;      // or, with few columns, reciprocal pivots [nz][ny nxh] and
    void *pc;        // the coefficients c' (field precision)
    void *twx;       // exp(-2 pi i m / nx), m < nx/2, interleaved (field precision)
    void *twy;
    double *kx2, *ky2, *rho_h, *dd, *a, *c;
    double *mean, *partial;
    int logx, logy, loggx;
    bool thomas_lds;  // few columns: the z solve with stored pivots, in LDS
    int planes;       // fewer still: y transforms and z solve of a kx plane in one
                      // kernel (1; 2: with its pivots staged in LDS)
    size_t plane_lds;
};

static int ilog2(long long n) {
    int l = 0;
    while ((1LL << l) < n) ++l;
    return ((1LL << l) == n) ? l : -1;
}

template <typename T> struct C2 { T x, y; };

template <typename T>
__device__ __forceinline__ C2<T> cmul(C2<T> a, C2<T> b) {
    return C2<T>{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ __forceinline__ void bfly(C2<T> &a, C2<T> &b) {
    const C2<T> t = a;
    a = C2<T>{t.x + b.x, t.y + b.y};
    b = C2<T>{t.x - b.x, t.y - b.y};
}
// times -i (forward) or +i (inverse)
template <typename T, bool INV>
__device__ __forceinline__ C2<T> rot90(C2<T> a) {
    return INV ? C2<T>{-a.y, a.x} : C2<T>{a.y, -a.x};
}

// In-register DFTs of size 2, 4, 8, natural order in and out, kernel
// exp(-+2 pi i n k / R) (forward: minus).
template <typename T, bool INV>
__device__ __forceinline__ void dft2(C2<T> *v) {
    bfly(v[0], v[1]);
}
template <typename T, bool INV>
__device__ __forceinline__ void dft4(C2<T> *v) {
    bfly(v[0], v[2]);
    bfly(v[1], v[3]);
    v[3] = rot90<T, INV>(v[3]);
    bfly(v[0], v[1]);
    bfly(v[2], v[3]);
    const C2<T> t = v[1];
    v[1] = v[2];
    v[2] = t;
}
template <typename T, bool INV>
__device__ __forceinline__ void dft8(C2<T> *v) {
    C2<T> e[4] = {v[0], v[2], v[4], v[6]};
    C2<T> o[4] = {v[1], v[3], v[5], v[7]};
    dft4<T, INV>(e);
    dft4<T, INV>(o);
    const T h = T(0.70710678118654752440);
    // o[k] *= exp(-+ i pi k / 4)
    o[1] = INV ? C2<T>{h * (o[1].x - o[1].y), h * (o[1].x + o[1].y)}
               : C2<T>{h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)};
    o[2] = rot90<T, INV>(o[2]);
    o[3] = INV ? C2<T>{-h * (o[3].x + o[3].y), h * (o[3].x - o[3].y)}
               : C2<T>{h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y)};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = C2<T>{e[k].x + o[k].x, e[k].y + o[k].y};
        v[k + 4] = C2<T>{e[k].x - o[k].x, e[k].y - o[k].y};
    }
}
template <typename T, int R, bool INV>
__device__ __forceinline__ void dft(C2<T> *v) {
    if (R == 2) dft2<T, INV>(v);
    else if (R == 4) dft4<T, INV>(v);
    else dft8<T, INV>(v);
}

// One radix-R pass of a Stockham autosort FFT over S interleaved length-N
// sequences in LDS (element e of sequence b at buf[e * S + b]).  Thread t
// (0 .. N/8-1) of sequence b does the 8/R butterflies q = t + s N/8: it reads
// x[q + r N/R], twiddles by w_N^{k r N/(Ns R)} with k = q mod Ns, transforms,
// and writes to (q - k) R + k + r Ns.  Ns is the length of the sub-transforms
// already combined.  All threads of the block take part in the two barriers;
// those without a butterfly (act false) do nothing else.
template <typename T, int R, bool INV>
__device__ __forceinline__ void stockham_pass(C2<T> *buf, int S, int b, int t, int N, int Ns, const C2<T> *tw,
                                              bool act) {
    constexpr int NB = 8 / R;
    const int NR = N / R, N8 = N >> 3;
    C2<T> v[NB][R];
    if (act)
#pragma unroll
        for (int s = 0; s < NB; ++s) {
            const int q = t + s * N8;
#pragma unroll
            for (int r = 0; r < R; ++r) v[s][r] = buf[(q + r * NR) * S + b];
        }
    __syncthreads();
    if (act)
#pragma unroll
    for (int s = 0; s < NB; ++s) {
        const int q = t + s * N8;
        const int k = q & (Ns - 1);
        if (Ns > 1) {
            const int step = k * (N / (Ns * R));
#pragma unroll
            for (int r = 1; r < R; ++r) {
                C2<T> w = tw[step * r];
                if (INV) w.y = -w.y;
                v[s][r] = cmul(v[s][r], w);
            }
        }
        dft<T, R, INV>(v[s]);
        const int base = (q - k) * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) buf[(base + r * Ns) * S + b] = v[s][r];
    }
    __syncthreads();
}

// Unnormalised DFT (forward: exp(-2 pi i n k/N); inverse: +) of the S
// sequences in buf, N = 2^logN >= 8, in natural order in and out.
// tw[m] = exp(-2 pi i m/N), m < N.
template <typename T, bool INV>
__device__ __forceinline__ void stockham_fft(C2<T> *buf, int S, int b, int t, int N, int logN, const C2<T> *tw, bool act = true) {
    int Ns = 1;
    const int rem = logN % 3;
    if (rem == 1) {
        stockham_pass<T, 2, INV>(buf, S, b, t, N, Ns, tw, act);
        Ns = 2;
    } else if (rem == 2) {
        stockham_pass<T, 4, INV>(buf, S, b, t, N, Ns, tw, act);
        Ns = 4;
    }
    for (int p = 0; p < logN / 3; ++p) {
        stockham_pass<T, 8, INV>(buf, S, b, t, N, Ns, tw, act);
        Ns *= 8;
    }
}

// ---------------------------------------------------------------------------
// The partial sums of w's levels are computed before this kernel; every
// wavefront adds those of its level and the level below in order, and the level's first block writes the mean
// that the correction reads and, on the last stage, clears the CFL maximum.
// One block per 2S consecutive rows (j0 .. j0+2S-1) of one level: divergence
// (PressureSolver.pyx:138-175, zeroed then x, y, z contributions added in that
// order), then the forward FFT along x of the rows in pairs (row 2b as the
// real part and row 2b+1 as the imaginary part of one complex sequence),
// separated into the two half spectra.
// TR: the spectrum as planes [kx][level][y] (plane_solve_kernel) instead of rows
// [level][y][kx]; the block's 2S rows are then consecutive.
// V consecutive cells per access (16 bytes; 1 where a field is off a 16-byte
// boundary): a third of the addresses and more bytes in flight per thread than
// with single cells, 512 x 512 x 256 FP64 560 -> 467 us (4.6 TB/s), FP32 267 ->
// 250.  The phases of the few blocks that fit a CU bound it (memory, then LDS:
// the real values' writes meet in a few banks).  Neighbouring lanes on 8
// neighbouring rows have no such conflicts, but a row's share is then 128 bytes
// and the memory slower (562 and 329).
template <typename TS, bool TR, int V>
__global__ __launch_bounds__(512) void div_fftx_kernel(Geo g, const TS *u, const TS *v, const TS *w,
                                                       const double *alpha0, const double *alpha0_half,
                                                       const double *partial, double *mean, double *cfl, TS *div_out,
                                                       C2<TS> *spec, const C2<TS> *tw, int logx, int nxh, int nxp,
                                                       int logS) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int S = 1 << logS;
    C2<TS> *buf = reinterpret_cast<C2<TS> *>(smem_raw);
    TS *bufr = reinterpret_cast<TS *>(smem_raw);
    const int kk = blockIdx.y;
    const int k = kk + g.gw;
    const int j0 = blockIdx.x << (logS + 1);
    const double ah = alpha0_half[k];
    const double a0 = alpha0[k], a0m = alpha0[k - 1];
    // multiplied by 1/(n0*n1) as the reference does
    const double rn = 1.0 / (double)((long long)g.ny * g.nx);
    double mk = 0.0, mkm = 0.0;
    if (blockDim.x >= 2 * MEAN_SPLITS) {
        // lanes 0..15: the partials of level k, 16..31: of level k - 1
        const int ml = threadIdx.x % (2 * MEAN_SPLITS);
        const double ms = partial[(long long)(ml < MEAN_SPLITS ? k : k - 1) * MEAN_SPLITS + ml % MEAN_SPLITS];
#pragma unroll
        for (int o = 0; o < MEAN_SPLITS; ++o) {
            mk += __shfl(ms, o, 64);
            mkm += __shfl(ms, MEAN_SPLITS + o, 64);
        }
    } else {  // blocks below half a wavefront (nx = 8 or 16 with few rows)
        for (int o = 0; o < MEAN_SPLITS; ++o) {
            mk += partial[(long long)k * MEAN_SPLITS + o];
            mkm += partial[(long long)(k - 1) * MEAN_SPLITS + o];
        }
    }
    mk *= rn;
    mkm *= rn;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        mean[k] = mk;
        if (kk == 0 && cfl) *cfl = 0.0;
    }
    const double dxi0 = 1.0 / g.dx[0], dxi1 = 1.0 / g.dx[1], dxi2 = 1.0 / g.dx[2];
    // Q accesses per field and thread at a time: all their loads are issued
    // before the arithmetic and the stores (a store in between would hold back
    // the next cells' loads, which the compiler must assume it aliases)
    typedef TS VT __attribute__((ext_vector_type(V)));
    constexpr int Q = V == 1 ? 4 : 2, LV = V == 1 ? 0 : (V == 2 ? 1 : 2);
    const int B = blockDim.x, nt = (g.nx / V) << (logS + 1);
    auto get = [](const TS *f) { return *reinterpret_cast<const VT *>(f); };
    for (int t0 = threadIdx.x; t0 < nt; t0 += Q * B) {
        VT uc[Q], vc[Q], vm[Q], wc[Q], wm[Q];
        TS ue[Q];  // u of the cell before the first
        long long oo[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int t = min(t0 + q * B, nt - 1);  // a clamped duplicate past the end: loaded, not stored
            const int i = (t & (g.nx / V - 1)) * V;
            const int j = j0 + (t >> (logx - LV));
            const int jm = j == 0 ? g.ny - 1 : j - 1;
            const long long row = gidx(g, 0, j, k), o = row + i;
            oo[q] = o;
            uc[q] = get(u + o);
            ue[q] = u[row + (i == 0 ? g.nx - 1 : i - 1)];
            vc[q] = get(v + o);
            vm[q] = get(v + gidx(g, i, jm, k));
            wc[q] = get(w + o);
            wm[q] = get(w + o - g.plane);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int t = t0 + q * B;
            if (t >= nt) continue;
            const int i = (t & (g.nx / V - 1)) * V, rb = t >> (logx - LV);
            VT d;
            TS um = ue[q];
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if (sizeof(TS) == 8) {
                    // the profiles are positive normal numbers: div64 is the
                    // IEEE quotient (common.h)
                    double dv = 0.0;
                    dv += (div64((double)uc[q][e], ah) - div64((double)um, ah)) * dxi0;
                    dv += (div64((double)vc[q][e], ah) - div64((double)vm[q][e], ah)) * dxi1;
                    const double wk = (double)wc[q][e] - mk;
                    const double wkm = (double)wm[q][e] - mkm;
                    dv += (div64(wk, a0) - div64(wkm, a0m)) * dxi2;
                    d[e] = (TS)dv;
                } else {
                    // FP32 path: rho0*u in FP32 except the level means and profiles
                    const float rh = (float)(1.0 / ah);
                    float dv = ((float)uc[q][e] - (float)um) * (float)(dxi0)*rh;
                    dv += ((float)vc[q][e] - (float)vm[q][e]) * (float)(dxi1)*rh;
                    const float wk = (float)((double)wc[q][e] - mk);
                    const float wkm = (float)((double)wm[q][e] - mkm);
                    dv += (wk * (float)(1.0 / a0) - wkm * (float)(1.0 / a0m)) * (float)dxi2;
                    d[e] = (TS)dv;
                }
                um = uc[q][e];
                bufr[2 * ((i + e) * S + (rb >> 1)) + (rb & 1)] = d[e];
            }
            if (div_out) *reinterpret_cast<VT *>(div_out + oo[q]) = d;
        }
    }
    __syncthreads();
    const int b = threadIdx.x & (S - 1), t = threadIdx.x >> logS;
    stockham_fft<TS, false>(buf, S, b, t, g.nx, logx, tw, t < g.nx / 8);
    // X_a[m] = (Z[m] + conj Z[N-m]) / 2, X_b[m] = -i (Z[m] - conj Z[N-m]) / 2
    if (TR) {
        for (int q = threadIdx.x; q < nxh * 2 * S; q += blockDim.x) {
            const int r = q & (2 * S - 1), m = q >> (logS + 1), pb = r >> 1;
            const C2<TS> z = buf[m * S + pb];
            const C2<TS> zm = buf[((g.nx - m) & (g.nx - 1)) * S + pb];
            spec[((long long)m * g.nz + kk) * g.ny + j0 + r] =
                (r & 1) ? C2<TS>{TS(0.5) * (z.y + zm.y), TS(-0.5) * (z.x - zm.x)}
                        : C2<TS>{TS(0.5) * (z.x + zm.x), TS(0.5) * (z.y - zm.y)};
        }
        return;
    }
    const int nxhalf = g.nx / 2;  // the last column after the others, which need no division
    for (int q = threadIdx.x; q < (nxh << logS); q += blockDim.x) {
        const bool last = q >= nxhalf << logS;
        const int m = last ? nxhalf : q & (nxhalf - 1);
        const int pb = last ? q - (nxhalf << logS) : q >> (logx - 1);
        const C2<TS> z = buf[m * S + pb];
        const C2<TS> zm = buf[((g.nx - m) & (g.nx - 1)) * S + pb];
        const C2<TS> xa{TS(0.5) * (z.x + zm.x), TS(0.5) * (z.y - zm.y)};
        const C2<TS> xb{TS(0.5) * (z.y + zm.y), TS(-0.5) * (z.x - zm.x)};
        spec[((long long)kk * g.ny + j0 + 2 * pb) * nxp + m] = xa;
        spec[((long long)kk * g.ny + j0 + 2 * pb + 1) * nxp + m] = xb;
    }
}

// FFT along y for gx consecutive kx columns of one level, in place
// (inverse: times 1/ny).
template <typename TS>
__global__ __launch_bounds__(1024) void ffty_kernel(Geo g, C2<TS> *spec, const C2<TS> *tw, int logy, int nxh,
                                                   int nxp, int gx, int loggx, int inverse) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    C2<TS> *buf = reinterpret_cast<C2<TS> *>(smem_raw);
    const int kx0 = blockIdx.x * gx;
    const int kk = blockIdx.y;
    const int ncol = min(gx, nxh - kx0);
    C2<TS> *lev = spec + (long long)kk * g.ny * nxp;
    // staged four elements per thread at a time, loads before LDS writes
    const int B = blockDim.x, nq = g.ny * gx;
    for (int q0 = threadIdx.x; q0 < nq; q0 += 4 * B) {
        C2<TS> z[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int q = q0 + u * B;
            const int y = q >> loggx, b = q & (gx - 1);
            z[u] = (q < nq && b < ncol) ? lev[(long long)y * nxp + kx0 + b] : C2<TS>{TS(0), TS(0)};
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (q0 + u * B < nq) buf[q0 + u * B] = z[u];
    }
    __syncthreads();
    const int b = threadIdx.x & (gx - 1), t = threadIdx.x >> loggx;
    if (inverse) stockham_fft<TS, true>(buf, gx, b, t, g.ny, logy, tw);
    else stockham_fft<TS, false>(buf, gx, b, t, g.ny, logy, tw);
    const TS sc = inverse ? TS(1.0 / (double)g.ny) : TS(1);
    for (int q = threadIdx.x; q < g.ny * gx; q += blockDim.x) {
        const int y = q >> loggx, bb = q & (gx - 1);
        if (bb < ncol) {
            C2<TS> z = buf[q];
            if (inverse) {
                z.x *= sc;
                z.y *= sc;
            }
            lev[(long long)y * nxp + kx0 + bb] = z;
        }
    }
}

// Largest nz of the pressure solve: the Thomas kernel holds four FP64 level
// profiles in LDS (64 KB at this size).
constexpr int PRESSURE_MAX_NZ = 2048;

// Levels per segment of the checkpointed Thomas solve: the right-hand sides
// of two segments are held in registers, twice the registers per level in FP64.
template <typename TS> constexpr int thomas_seg() { return sizeof(TS) == 4 ? 16 : 8; }

// 1/d in FP64 from the hardware reciprocal and two Newton steps (within an
// ulp or two of the division; no special values occur: d is a pivot of a
// diagonally dominant system).
__device__ __forceinline__ double rcp64(double d) {
    double r = __builtin_amdgcn_rcp(d);
    double e = __builtin_fma(-d, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-d, r, 1.0);
    return __builtin_fma(r, e, r);
}

// One thread per (kx, ky) column: TDMA of SparseSolvers.pyx:24-43 on the real
// and imaginary parts, with the diagonal of compute_diagonal
// (PressureFFTParallel.pyx:129-148); the (0,0) mode is set to zero (:196-200).
// The recurrence runs in FP64 whatever the storage type TS.  No per-level
// scratch: the forward sweep streams the right-hand sides and keeps only the
// FP64 carry (c', x'r, x'i) at the last level of every S-level segment (3
// doubles per column per segment, in ck).  The back substitution walks the
// segments from the top: it recomputes a segment's forward values from the
// carry below it and the right-hand sides, which are still in place (the
// solution overwrites a segment only after its forward values are
// recomputed), then substitutes down the segment.  The next segment's
// right-hand sides and carry are loaded while the current one is worked on.
// Per column-level: the right-hand side read twice and the solution written
// (24 B in FP32, 48 B in FP64), where a stored scratch of forward values
// would add its write and read back (40 and 80 B).  Both sweeps evaluate the
// same FP64 expressions, so the recomputed values are the forward sweep's,
// bit for bit; the reciprocal is rcp64, not an IEEE division.  The forward
// values enter the back substitution rounded to TS, as the reference's
// in-place arrays would hold them in that precision.
template <typename TS, int S>
__global__ __launch_bounds__(256, 3) void thomas_kernel(Geo g, C2<TS> *spec, double *ck, const double *kx2,
                                                        const double *ky2, const double *rho_h, const double *dd,
                                                        const double *a, const double *c, int nxh, int nxp) {
    // The level profiles (rho_h, dd, a, c) in LDS, 4 nz doubles: read from
    // global memory in the level loops they are vector loads (the stores
    // keep the compiler from the scalar cache), and each wait for one would
    // also wait for every older load and store, right-hand sides included.
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double *lv = reinterpret_cast<double *>(smem_raw);
    const int nz = g.nz;
    for (int t = threadIdx.x; t < nz; t += blockDim.x) {
        lv[t] = rho_h[t];
        lv[nz + t] = dd[t];
        lv[2 * nz + t] = a[t];
        lv[3 * nz + t] = c[t];
    }
    __syncthreads();
    const double *lrho = lv, *ldd = lv + nz, *la = lv + 2 * nz, *lc = lv + 3 * nz;
    const long long ncol = (long long)g.ny * nxp;
    const long long col = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= ncol) return;
    const int kx = (int)(col % nxp);
    const int ky = (int)(col / nxp);
    if (kx >= nxh) return;
    if (kx == 0 && ky == 0) {
        for (int k = 0; k < nz; ++k) spec[(long long)k * ncol + col] = C2<TS>{TS(0), TS(0)};
        return;
    }
    const double kk = kx2[kx] + ky2[ky];
    auto at = [&](int k) { return spec + (long long)k * ncol + col; };
    // one forward step: the carry of level k - 1 to level k
    auto fstep = [&](int k, C2<TS> z, double &sc, double &xr, double &xi) {
        const double b = lrho[k] * kk - ldd[k];
        if (k == 0) {
            const double ib = rcp64(b);
            sc = lc[0] * ib;
            xr = (double)z.x * ib;
            xi = (double)z.y * ib;
        } else {
            const double m = rcp64(b - la[k] * sc);
            sc = lc[k] * m;
            xr = ((double)z.x - la[k] * xr) * m;
            xi = ((double)z.y - la[k] * xi) * m;
        }
    };
    // forward sweep: right-hand sides S levels ahead, loaded at every level
    // (clamped), a carry stored at the end of every whole segment
    double sc = 0.0, xr = 0.0, xi = 0.0;
    C2<TS> zq[S];
#pragma unroll
    for (int u = 0; u < S; ++u) zq[u] = *at(min(u, nz - 1));
    int k0 = 0;
    for (; k0 + S <= nz; k0 += S) {
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const int k = k0 + u;
            const C2<TS> z = zq[u];
            zq[u] = *at(min(k + S, nz - 1));
            fstep(k, z, sc, xr, xi);
        }
        const long long q = 3LL * (k0 / S) * ncol + col;
        ck[q] = sc;
        ck[q + ncol] = xr;
        ck[q + 2 * ncol] = xi;
    }
#pragma unroll
    for (int u = 0; u < S; ++u)
        if (k0 + u < nz) fstep(k0 + u, zq[u], sc, xr, xi);
    // the top level's solution is its forward value
    *at(nz - 1) = C2<TS>{(TS)xr, (TS)xi};
    // back substitution, segment by segment from the top; (xr, xi) carries
    // the solution of the level above, in FP64.  Segment sg needs the carry
    // of segment sg - 1 (none for sg = 0, whose first step starts afresh);
    // the loads of the next segment down use a clamped index, and with a
    // single segment no carry is read.
    const int nseg = (nz + S - 1) / S;
    const int top = nz - 2 < 0 ? 0 : nz - 2;  // the highest level still holding its right-hand side
    C2<TS> zs[S];
    double csc = 0.0, cxr = 0.0, cxi = 0.0;
    auto load_seg = [&](int sg, C2<TS> *z, double &lsc, double &lxr, double &lxi) {
#pragma unroll
        for (int u = 0; u < S; ++u) z[u] = *at(min(sg * S + u, top));
        if (nseg > 1) {
            const long long q = 3LL * max(sg - 1, 0) * ncol + col;
            lsc = ck[q];
            lxr = ck[q + ncol];
            lxi = ck[q + 2 * ncol];
        }
    };
    load_seg(nseg - 1, zs, csc, cxr, cxi);
    for (int sg = nseg - 1; sg >= 0; --sg) {
        const int lo = sg * S;
        C2<TS> zn[S];
        double nsc = 0.0, nxr = 0.0, nxi = 0.0;
        load_seg(max(sg - 1, 0), zn, nsc, nxr, nxi);
        TS sT[S], rT[S], iT[S];
#pragma unroll
        for (int u = 0; u < S; ++u) {
            if (lo + u < nz - 1) {
                fstep(lo + u, zs[u], csc, cxr, cxi);
                sT[u] = (TS)csc;
                rT[u] = (TS)cxr;
                iT[u] = (TS)cxi;
            }
        }
#pragma unroll
        for (int u = S - 1; u >= 0; --u) {
            const int k = lo + u;
            if (k < nz - 1) {
                xr = (double)rT[u] - (double)sT[u] * xr;
                xi = (double)iT[u] - (double)sT[u] * xi;
                *at(k) = C2<TS>{(TS)xr, (TS)xi};
            }
        }
#pragma unroll
        for (int u = 0; u < S; ++u) zs[u] = zn[u];
        csc = nsc;
        cxr = nxr;
        cxi = nxi;
    }
}

// The same solve for grids with few columns, where one thread per column is one
// dependent chain (a reciprocal and seven more FP64 operations per level and
// sweep) on a few SIMDs.  The chain of the pivots depends on the plan only, so
// pivot_kernel forms the reciprocal pivots m and the coefficients c' once, when
// the plan is made, with thomas_kernel's expressions.  A block of 16 columns
// then loads all their levels' right-hand sides, m and c' into LDS together
// (every load in flight at once) and one wavefront runs the two sweeps, the
// real parts on lanes 0..15 and the imaginary parts on lanes 16..31: three
// dependent operations per level forward and two back.  The same bits.
// 64^3 FP64: 21 -> 11.5 us, 256 x 64 x 75 FP32 26 -> 17 (holding the columns
// in LDS without stored pivots: 19.6 and 21).
constexpr int TL_COLS = 16, TL_U = 8;
template <typename TS> constexpr size_t thomas_lds_bytes(int nz) {
    return (size_t)nz * (TL_COLS * (sizeof(C2<TS>) + sizeof(double) + sizeof(TS)) + sizeof(double));
}
// m and c' (rounded to TS, as the forward values are) of column (kx, ky) at
// level k, at k sk + ky sy + kx sx
template <typename TS>
__global__ __launch_bounds__(64) void pivot_kernel(Geo g, const double *kx2, const double *ky2, const double *rho_h,
                                                   const double *dd, const double *a, const double *c, int nxh,
                                                   long long sk, long long sy, long long sx, double *pm, TS *pc) {
    const long long ncol = (long long)g.ny * nxh;
    const long long col = (long long)blockIdx.x * 64 + threadIdx.x;
    if (col >= ncol) return;
    const int kx = (int)(col % nxh), ky = (int)(col / nxh);
    const double kk = kx2[kx] + ky2[ky];
    const long long o = ky * sy + kx * sx;
    double sc = 0.0;
    for (int k = 0; k < g.nz; ++k) {
        const double b = rho_h[k] * kk - dd[k];
        const double m = k == 0 ? rcp64(b) : rcp64(b - a[k] * sc);
        sc = c[k] * m;
        pm[k * sk + o] = m;
        pc[k * sk + o] = (TS)sc;
    }
}
// Both sweeps of one part (real or imaginary) of one column from the stored
// pivots: x[k xs] in LDS holds the right-hand side and becomes the solution,
// m[k ms] and c[k ms] (LDS or global) are the pivots' arrays, la the lower
// diagonal.  A batch of TL_U levels is read while the one before is worked on.
template <typename TS>
__device__ __forceinline__ void column_sweeps(TS *x, int xs, const double *m, const TS *c, long long ms, const double *la,
                                              int nz) {
    double xr = 0.0;
    TS q[2][TL_U];
    double pm[2][TL_U], pa[2][TL_U];
    auto fetch = [&](int b, int k0) {
#pragma unroll
        for (int u = 0; u < TL_U; ++u) {
            const int k = min(k0 + u, nz - 1);
            q[b][u] = x[k * xs];
            pm[b][u] = m[k * ms];
            pa[b][u] = la[k];
        }
    };
    auto fwd = [&](int b, int k0) {
#pragma unroll
        for (int u = 0; u < TL_U; ++u)
            if (k0 + u < nz) {
                xr = k0 + u == 0 ? (double)q[b][u] * pm[b][u] : ((double)q[b][u] - pa[b][u] * xr) * pm[b][u];
                x[(k0 + u) * xs] = (TS)xr;
            }
    };
    fetch(0, 0);
    for (int k0 = 0; k0 < nz; k0 += 2 * TL_U) {
        fetch(1, k0 + TL_U);
        fwd(0, k0);
        fetch(0, k0 + 2 * TL_U);
        fwd(1, k0 + TL_U);
    }
    // back substitution from the level below the top, whose solution is its
    // forward value, carried unrounded
    TS f[2][TL_U];
    auto bfetch = [&](int b, int k0) {
#pragma unroll
        for (int u = 0; u < TL_U; ++u) {
            const int k = max(k0 - u, 0);
            q[b][u] = x[k * xs];
            f[b][u] = c[k * ms];
        }
    };
    auto bwd = [&](int b, int k0) {
#pragma unroll
        for (int u = 0; u < TL_U; ++u)
            if (k0 - u >= 0) {
                xr = (double)q[b][u] - (double)f[b][u] * xr;
                x[(k0 - u) * xs] = (TS)xr;
            }
    };
    bfetch(0, nz - 2);
    for (int k0 = nz - 2; k0 >= 0; k0 -= 2 * TL_U) {
        bfetch(1, k0 - TL_U);
        bwd(0, k0);
        bfetch(0, k0 - 2 * TL_U);
        bwd(1, k0 - TL_U);
    }
}
template <typename TS>
__global__ __launch_bounds__(256) void thomas_lds_kernel(Geo g, C2<TS> *spec, const double *pm, const TS *pc,
                                                         const double *a, int nxh, int nxp) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int nz = g.nz;
    double *la = reinterpret_cast<double *>(smem_raw);               // [nz]
    double *lm = la + nz;                                            // [nz][16]
    C2<TS> *z = reinterpret_cast<C2<TS> *>(lm + (size_t)nz * TL_COLS);  // [nz][16]
    TS *lc = reinterpret_cast<TS *>(z + (size_t)nz * TL_COLS);       // [nz][16]
    for (int t = threadIdx.x; t < nz; t += 256) la[t] = a[t];
    const long long ncol = (long long)g.ny * nxh, plane = (long long)g.ny * nxp;
    const int cl = threadIdx.x % TL_COLS, lv = threadIdx.x / TL_COLS;
    const long long cc = (long long)blockIdx.x * TL_COLS + cl;
    const bool live = cc < ncol;
    const long long col = live ? cc : ncol - 1;
    C2<TS> *sp = spec + (col / nxh) * nxp + col % nxh;
    constexpr int LV = 256 / TL_COLS, NB = 4;
    for (int k0 = lv; k0 < nz; k0 += NB * LV) {
        C2<TS> q[NB];
        double m[NB];
        TS f[NB];
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const long long k = min(k0 + u * LV, nz - 1);
            q[u] = sp[k * plane];
            m[u] = pm[k * ncol + col];
            f[u] = pc[k * ncol + col];
        }
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int k = k0 + u * LV;
            if (k < nz) {
                z[k * TL_COLS + cl] = q[u];
                lm[k * TL_COLS + cl] = m[u];
                lc[k * TL_COLS + cl] = f[u];
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < 2 * TL_COLS) {
        column_sweeps<TS>(reinterpret_cast<TS *>(z) + 2 * cl + threadIdx.x / TL_COLS, 2 * TL_COLS, lm + cl, lc + cl, TL_COLS,
                          la, nz);
    }
    __syncthreads();
    // the (0,0) mode is set to zero
    const bool zero = col == 0;
    if (live)
        for (int k = lv; k < nz; k += LV)
            sp[(long long)k * plane] = zero ? C2<TS>{TS(0), TS(0)} : z[k * TL_COLS + cl];
}

// The transform along y, the z solve and the inverse transform of one
// wavenumber kx in one kernel, where a plane of ny x nz complex values fits in
// LDS and the nxh planes' blocks are all resident at once: three kernels of
// little work each (two transforms and the solve, 22 us at 64^3 FP64) become one
// and the spectrum is read and written once instead of three times.  The
// spectrum is laid out as planes [kx][level][y].  In LDS level b of row y is
// element y S + b, S = nz made odd, so that accesses along either index spread
// over the banks.  The transforms run over as many levels at a time as the
// block has threads (ny / 8 each), the sweeps on one lane per column and part.
// The same bits as the separate kernels.  64^3 FP64 22.5 -> 17.7 us, 256 x 64 x 75
// FP32 29 -> 19, and two launches less.
// ST: the plane's pivots are staged in LDS too, loaded with the spectrum (read
// from global memory the sweeps wait for them).
template <typename TS, bool ST> size_t plane_lds_bytes(int ny, int nz) {
    return sizeof(C2<TS>) * (size_t)ny * (nz | 1) + sizeof(double) * (size_t)nz +
           (ST ? (sizeof(double) + sizeof(TS)) * (size_t)ny * nz : 0);
}
template <typename TS, bool ST>
__global__ __launch_bounds__(1024) void plane_solve_kernel(Geo g, C2<TS> *spec, const double *pm, const TS *pc,
                                                           const double *a, const C2<TS> *tw, int logy) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int ny = g.ny, nz = g.nz, S = nz | 1, B = blockDim.x, tid = threadIdx.x;
    C2<TS> *buf = reinterpret_cast<C2<TS> *>(smem_raw);
    double *la = reinterpret_cast<double *>(buf + (size_t)ny * S);
    double *lm = la + nz;                                        // ST: [nz][ny]
    TS *lc = reinterpret_cast<TS *>(lm + (ST ? (size_t)nz * ny : 0));
    const long long plane = (long long)blockIdx.x * nz * ny;
    C2<TS> *sp = spec + plane;
    for (int t = tid; t < nz; t += B) la[t] = a[t];
    const int n = ny * nz;
    for (int q0 = tid; q0 < n; q0 += 4 * B) {
        C2<TS> z[4];
        double m[4];
        TS f[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int q = min(q0 + u * B, n - 1);
            z[u] = sp[q];
            if (ST) {
                m[u] = pm[plane + q];
                f[u] = pc[plane + q];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int q = q0 + u * B;
            if (q < n) {
                buf[(q & (ny - 1)) * S + (q >> logy)] = z[u];
                if (ST) {
                    lm[q] = m[u];
                    lc[q] = f[u];
                }
            }
        }
    }
    __syncthreads();
    const int n8 = ny >> 3;
    const int per = min(B / n8, nz);  // levels transformed at a time
    const int b = tid % per, t = tid / per;
    for (int l0 = 0; l0 < nz; l0 += per)
        stockham_fft<TS, false>(buf + l0, S, b, t, ny, logy, tw, t < n8 && l0 + b < nz);
    for (int c = tid; c < 2 * ny; c += B) {
        const int ky = c & (ny - 1);
        column_sweeps<TS>(reinterpret_cast<TS *>(buf + (size_t)ky * S) + (c >> logy), 2, (ST ? lm : pm + plane) + ky,
                          (ST ? lc : pc + plane) + ky, ny, la, nz);
    }
    __syncthreads();
    if (blockIdx.x == 0) {  // the (0,0) mode is set to zero
        for (int k = tid; k < nz; k += B) buf[k] = C2<TS>{TS(0), TS(0)};
        __syncthreads();
    }
    for (int l0 = 0; l0 < nz; l0 += per)
        stockham_fft<TS, true>(buf + l0, S, b, t, ny, logy, tw, t < n8 && l0 + b < nz);
    const TS sc = TS(1.0 / (double)ny);
    for (int q = tid; q < n; q += B) {
        C2<TS> z = buf[(q & (ny - 1)) * S + (q >> logy)];
        z.x *= sc;
        z.y *= sc;
        sp[q] = z;
    }
}

// Inverse x transform of 2S rows in pairs: Z[m] = X_a[m] + i X_b[m] with the
// Hermitian extension X[N-m] = conj X[m], one inverse FFT, real part -> row
// 2b and imaginary part -> row 2b+1, times 1/nx, written to p at level k'+gw
// together with the mirrored z ghost level (sym, as communicate_variable does).
template <typename TS, bool TR>
__global__ __launch_bounds__(512) void ifftx_kernel(Geo g, const C2<TS> *spec, TS *p, const C2<TS> *tw, int logx,
                                                    int nxh, int nxp, int logS) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int S = 1 << logS;
    C2<TS> *buf = reinterpret_cast<C2<TS> *>(smem_raw);
    const TS *bufr = reinterpret_cast<const TS *>(smem_raw);
    const int kk = blockIdx.y;
    const int j0 = blockIdx.x << (logS + 1);
    // staged four elements per thread at a time: their loads are all issued
    // before the LDS writes (one memory round trip per four, not per one)
    const int B = blockDim.x, nq = g.nx << logS;
    for (int q0 = threadIdx.x; q0 < nq; q0 += 4 * B) {
        C2<TS> xa[4], xb[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int q = q0 + u * B;
            if (q < nq) {
                const int m = TR ? q >> logS : q & (g.nx - 1);
                const int pb = TR ? q & (S - 1) : q >> logx;
                const int mm = m < nxh ? m : g.nx - m;
                if (TR) {  // rows 2 pb and 2 pb + 1 of wavenumber mm are neighbours
                    const C2<TS> *ra = spec + ((long long)mm * g.nz + kk) * g.ny + j0 + 2 * pb;
                    xa[u] = ra[0];
                    xb[u] = ra[1];
                } else {
                    const C2<TS> *ra = spec + ((long long)kk * g.ny + j0 + 2 * pb) * nxp;
                    xa[u] = ra[mm];
                    xb[u] = ra[nxp + mm];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int q = q0 + u * B;
            if (q < nq) {
                const int m = TR ? q >> logS : q & (g.nx - 1);
                const int pb = TR ? q & (S - 1) : q >> logx;
                if (m >= nxh) {  // Hermitian extension X[N-m] = conj X[m]
                    xa[u].y = -xa[u].y;
                    xb[u].y = -xb[u].y;
                }
                buf[m * S + pb] = C2<TS>{xa[u].x - xb[u].y, xa[u].y + xb[u].x};
            }
        }
    }
    __syncthreads();
    const int b = threadIdx.x & (S - 1), t = threadIdx.x >> logS;
    stockham_fft<TS, true>(buf, S, b, t, g.nx, logx, tw);
    const TS sc = TS(1.0 / (double)g.nx);
    const int k = kk + g.gw;
    for (int q = threadIdx.x; q < (g.nx << (logS + 1)); q += blockDim.x) {
        const int i = q & (g.nx - 1);
        const int rb = q >> logx;
        const int j = j0 + rb;
        const TS val = bufr[2 * (i * S + (rb >> 1)) + (rb & 1)] * sc;
        p[gidx(g, i, j, k)] = val;
        if (kk < g.gw) p[gidx(g, i, j, g.gw - 1 - kk)] = val;
        if (kk >= g.nz - g.gw) p[gidx(g, i, j, 2 * g.gw + 2 * g.nz - 1 - k)] = val;
    }
}

// second_order_pressure_correction (PressureSolver.pyx:83-110) after the mean
// removal of w, with the z ghost levels of u, v (sym) and w (asym) that each
// corrected level feeds, and the CFL maximum of the corrected interior.  V
// consecutive columns per thread (16-byte accesses; nx is a power of two), a
// z chunk per block row; p at level k comes from the level below's step.
// Bound: HBM, 7 field passes; u, v and w, read and written once, through
// non-temporal accesses.  512 x 512 x 256: FP64 764 -> 699 us (5.4 TB/s; 813
// with ordinary accesses), FP32 378 -> 345 us; 64^3 FP64 10 -> 6.5 (one column
// per thread and one row per block before).
template <typename TS, int V>
__global__ __launch_bounds__(256) void correct_kernel(Geo g, TS *u, TS *v, TS *w, const TS *p,
                                                      const double *__restrict__ mean, double dt, double *cfl,
                                                      int kchunk) {
    typedef TS VT __attribute__((ext_vector_type(V)));
    const long long e = ((long long)blockIdx.x * 256 + threadIdx.x) * V;
    const int k0 = g.gw + blockIdx.y * kchunk;
    const int k1 = blockIdx.y + 1 == gridDim.y ? g.nz + g.gw : k0 + kchunk;
    const int gw = g.gw, nzg = g.nzg;
    const long long P = g.plane;
    auto get = [](const TS *f) { return *reinterpret_cast<const VT *>(f); };
    auto getn = [](const TS *f) { return __builtin_nontemporal_load(reinterpret_cast<const VT *>(f)); };
    auto put = [](TS *f, VT x) { __builtin_nontemporal_store(x, reinterpret_cast<VT *>(f)); };
    double cm = 0.0;
    if (e < P) {
        const int i = (int)(e & (g.nx - 1));
        const long long r = e - i;
        const long long ce = i + V == g.nx ? r : e + V;          // the column east of the last one
        const long long cn = r + g.nx == P ? (long long)i : e + g.nx;  // the row to the north
        VT pc = get(p + (long long)k0 * P + e);
        // four levels at a time: all their loads before their stores (a store
        // would hold back the next level's loads, which it may alias)
        for (int kb = k0; kb < k1; kb += 4) {
            VT uq[4], vq[4], wq[4], pnq[4], ptq[4];
            TS peq[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int k = min(kb + q, k1 - 1);  // a clamped duplicate past the end: loaded, not stored
                const long long lo = (long long)k * P;
                peq[q] = p[lo + ce];
                pnq[q] = get(p + lo + cn);
                ptq[q] = get(p + lo + P + e);
                uq[q] = getn(u + lo + e);
                vq[q] = getn(v + lo + e);
                wq[q] = getn(w + lo + e);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int k = kb + q;
                if (k >= k1) break;
                const long long o = (long long)k * P + e;
                const double mk = mean[k];
                VT un, vn, wn;
#pragma unroll
                for (int c = 0; c < V; ++c) {
                    const TS pcc = pc[c], pe = c + 1 < V ? pc[c + 1 < V ? c + 1 : c] : peq[q], pn = pnq[q][c], pt = ptq[q][c];
                    if (sizeof(TS) == 8) {
                        un[c] = uq[q][c] - (pe - pcc) * g.dxi[0];
                        vn[c] = vq[q][c] - (pn - pcc) * g.dxi[1];
                        const double wm = (double)wq[q][c] - mk;
                        wn[c] = (TS)(wm - ((double)pt - (double)pcc) * g.dxi[2]);
                    } else {
                        un[c] = uq[q][c] - (pe - pcc) * (TS)g.dxi[0];
                        vn[c] = vq[q][c] - (pn - pcc) * (TS)g.dxi[1];
                        wn[c] = (TS)((double)wq[q][c] - mk) - (pt - pcc) * (TS)g.dxi[2];
                    }
                    if (cfl) {
                        const double x = dt * (fabs((double)un[c]) * g.dxi[0] + fabs((double)vn[c]) * g.dxi[1] +
                                               fabs((double)wn[c]) * g.dxi[2]);
                        cm = cfl_fold(cm, x);
                    }
                }
                put(u + o, un);
                put(v + o, vn);
                put(w + o, wn);
                // the ghost levels this level feeds (as rk_store in advection_impl.h)
                if (k < 2 * gw) {
                    put(u + (long long)(2 * gw - 1 - k) * P + e, un);
                    put(v + (long long)(2 * gw - 1 - k) * P + e, vn);
                    if (k == gw) put(w + (long long)(gw - 1) * P + e, VT(TS(0)));
                    if (k <= 2 * gw - 2) put(w + (long long)(2 * gw - 2 - k) * P + e, -wn);
                }
                if (k >= nzg - 2 * gw) {
                    put(u + (long long)(2 * (nzg - gw) - 1 - k) * P + e, un);
                    put(v + (long long)(2 * (nzg - gw) - 1 - k) * P + e, vn);
                    if (k == nzg - gw - 1) put(w + (long long)(nzg - gw) * P + e, VT(TS(0)));
                    if (k >= nzg - 2 * gw + 1) put(w + (long long)(2 * (nzg - gw) - k) * P + e, -wn);
                }
                pc = ptq[q];
            }
        }
    }
    // + 1e-11 as compute_cfl_max: rounding is monotonic, so adding it to every
    // block's maximum gives the maximum plus it
    if (cfl) cfl_block_max(cm + 1e-11, cfl);
}

// Standalone divergence (interior) in the field precision.
template <typename TS>
__global__ void divergence_kernel(Geo g, const TS *u, const TS *v, const TS *w, const double *alpha0,
                                  const double *alpha0_half, TS *div) {
    const long long n = g.plane * g.nz;
    const double dxi0 = 1.0 / g.dx[0], dxi1 = 1.0 / g.dx[1], dxi2 = 1.0 / g.dx[2];
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(t % g.nx);
        const int j = (int)((t / g.nx) % g.ny);
        const int k = (int)(t / g.plane) + g.gw;
        const int im1 = i == 0 ? g.nx - 1 : i - 1;
        const int jm = j == 0 ? g.ny - 1 : j - 1;
        const long long o = gidx(g, i, j, k);
        const double ah = alpha0_half[k];
        double dv = 0.0;
        dv += ((double)u[o] / ah - (double)u[gidx(g, im1, j, k)] / ah) * dxi0;
        dv += ((double)v[o] / ah - (double)v[gidx(g, i, jm, k)] / ah) * dxi1;
        dv += (((double)w[o]) / alpha0[k] - ((double)w[o - g.plane]) / alpha0[k - 1]) * dxi2;
        div[o] = (TS)dv;
    }
}

// ---------------------------------------------------------------------------
// The form of a plan's z solve (PYCLES_PRESSURE_*) and the LDS of its blocks.
// The plane form where its blocks are all resident at once (with staged pivots,
// or else without) and, by the us of a projection with it and without:
// - fewer blocks than half the CUs: a plane of at most 5120 values.  64 x 64 x 75
//   FP64 49 and 53, 64 x 128 x 40 48 and 49, x 50 55 and 53, x 70 81 and 59;
// - a block per CU at most: any plane that fits.  256 x 64 x 75 FP32 57 and 62, 256 x
//   256 x 60 104 and 116, FP64 164 and 165;
// - more: the other kernels fill the chip too, and read and write the spectrum
//   as fast once it is large.  At most 2^17 columns and 2^21 cells (FP32 rows
//   of 1024 or more: 3 2^19), or 2^14 columns of any depth.  512 x 128 x 25 FP64 91
//   and 99, x 38 123 and 116; 512 x 32 x 150 138 and 146; 2048 x 64 x 20 141 and 125;
//   1024 x 64 x 20 FP32 60 and 62, x 30 86 and 80; 1024 x 128 x 40 161 and 127.
// Then stored pivots for few columns, their blocks all resident at once.
static bool planes_pay(const Geo &g, bool f64) {
    const int nxh = g.nx / 2 + 1;
    if (nxh < 128) return (long long)g.ny * g.nz <= 5120;
    if (nxh <= 256) return true;
    return g.plane <= 1 << 17 &&
           (g.plane <= 1 << 14 || g.plane * g.nz <= (!f64 && g.nx >= 1024 ? 3 << 19 : 1 << 21));
}
static int pressure_form(const Geo &g, int precision, size_t *lds) {
    const bool f64 = precision == PYCLES_F64;
    const int nxh = g.nx / 2 + 1;
    const long long cu = 160 * 1024;  // LDS of a CU
    if (planes_pay(g, f64)) {
        *lds = f64 ? plane_lds_bytes<double, true>(g.ny, g.nz) : plane_lds_bytes<float, true>(g.ny, g.nz);
        if ((long long)*lds <= cu && nxh <= 256 * (cu / (long long)*lds)) return PYCLES_PRESSURE_PLANES_STAGED;
        *lds = f64 ? plane_lds_bytes<double, false>(g.ny, g.nz) : plane_lds_bytes<float, false>(g.ny, g.nz);
        if ((long long)*lds <= cu && nxh <= 256 * (cu / (long long)*lds)) return PYCLES_PRESSURE_PLANES;
    }
    *lds = f64 ? thomas_lds_bytes<double>(g.nz) : thomas_lds_bytes<float>(g.nz);
    const long long blocks = ((long long)g.ny * nxh + TL_COLS - 1) / TL_COLS;
    if ((long long)*lds <= cu && blocks <= 256 * (cu / (long long)*lds) && blocks <= 2048) return PYCLES_PRESSURE_COLUMNS;
    *lds = 0;
    return PYCLES_PRESSURE_GENERAL;
}

// Whether a plan can be made for these sizes, and their logarithms
static int pressure_check(const pycles_dims *dims, int precision, int *logx, int *logy) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("pressure: bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    const Geo g = make_geo(dims);
    *logx = ilog2(g.nx);
    *logy = ilog2(g.ny);
    if (*logx < 3 || *logy < 3 || g.nx > 4096 || g.ny > 4096) {
        pycles_set_error("pressure: nx, ny must be powers of two in [8, 4096] (got %d, %d)", g.nx, g.ny);
        return PYCLES_ERR_UNSUPPORTED;
    }
    if (g.nz < 2 || g.nz > PRESSURE_MAX_NZ) {
        pycles_set_error("pressure: nz must be in [2, %d] (got %d)", PRESSURE_MAX_NZ, g.nz);
        return PYCLES_ERR_UNSUPPORTED;
    }
    return PYCLES_OK;
}

extern "C" int pycles_pressure_form(const pycles_dims *dims, int precision) {
    int logx, logy;
    const int rc = pressure_check(dims, precision, &logx, &logy);
    if (rc) return rc;
    size_t lds;
    return pressure_form(make_geo(dims), precision, &lds);
}

extern "C" int pycles_pressure_plan_create(const pycles_dims *dims, const double *rho0, const double *rho0_half,
                                           int precision, pycles_pressure_plan **out) {
    if (!out || !rho0 || !rho0_half) {
        pycles_set_error("pressure_plan_create: bad arguments");
        return PYCLES_ERR_ARG;
    }
    int logx, logy;
    const int rc = pressure_check(dims, precision, &logx, &logy);
    if (rc) return rc;
    const Geo g = make_geo(dims);
    pycles_pressure_plan *P = new pycles_pressure_plan();
    memset(P, 0, sizeof(*P));
    P->g = g;
    P->precision = precision;
    P->nxh = g.nx / 2 + 1;
    P->nxp = (P->nxh + 15) & ~15;
    P->logx = logx;
    P->logy = logy;
    const size_t cs = precision == PYCLES_F64 ? 16 : 8;
    const size_t es = cs / 2;
    // y transform: gx kx columns per block (16 makes 128-byte row segments in
    // FP32), at most 1024 threads and 64 KB
    int gx = 16;
    while (gx > 1 && ((size_t)gx * g.ny / 8 > 1024 || (size_t)gx * g.ny * cs > 64 * 1024)) gx >>= 1;
    P->gx = gx;
    P->loggx = ilog2(gx);
    const long long nspec = (long long)g.nz * g.ny * P->nxp;
    const int gw = g.gw, nz = g.nz;
    // host tables (same expressions as the reference initializers)
    std::vector<double> kx2(P->nxh), ky2(g.ny), rh(nz), dd(nz), a(nz), c(nz);
    for (int i = 0; i < P->nxh; ++i) {
        const double xi = (i <= g.nx / 2) ? (double)i : (double)(i - g.nx);
        kx2[i] = (2.0 * cos((2.0 * PC_PI / g.nx) * xi) - 2.0) / g.dx[0] / g.dx[0];
    }
    kx2[0] = 0.0;
    for (int j = 0; j < g.ny; ++j) {
        const double yi = (j <= g.ny / 2) ? (double)j : (double)(j - g.ny);
        ky2[j] = (2.0 * cos((2.0 * PC_PI / g.ny) * yi) - 2.0) / g.dx[1] / g.dx[1];
    }
    ky2[0] = 0.0;
    const double dzi = g.dxi[2];
    for (int k = 0; k < nz; ++k) {
        rh[k] = rho0_half[k + gw];
        if (k == 0) dd[k] = (rho0[gw]) * dzi * dzi;
        else if (k == nz - 1) dd[k] = (rho0[k + gw - 1]) * dzi * dzi;
        else dd[k] = (rho0[k + gw] + rho0[k + gw - 1]) * dzi * dzi;
        a[k] = (k == 0) ? 0.0 : dzi * dzi * rho0[k + gw - 1];
        c[k] = (k == nz - 1) ? 0.0 : dzi * dzi * rho0[k + gw];
    }
    // twiddles exp(-2 pi i m / N), m < N, interleaved (re, im)
    std::vector<double> twx(2 * g.nx), twy(2 * g.ny);
    for (int m = 0; m < g.nx; ++m) {
        const double ang = -2.0 * PC_PI * (double)m / (double)g.nx;
        twx[2 * m] = cos(ang);
        twx[2 * m + 1] = sin(ang);
    }
    for (int m = 0; m < g.ny; ++m) {
        const double ang = -2.0 * PC_PI * (double)m / (double)g.ny;
        twy[2 * m] = cos(ang);
        twy[2 * m + 1] = sin(ang);
    }
    // one allocation for the tables, the spectrum and the z solve's arrays (14 of
    // them and 8 copies made a plan take 130 to 190 us) and one copy of the tables
    struct Part {
        void **ptr;
        size_t off;
    } parts[14];
    int nparts = 0;
    size_t total = 0;
    auto part = [&](auto &ptr, size_t bytes) {
        parts[nparts++] = Part{(void **)&ptr, total};
        total += (bytes + 255) & ~(size_t)255;
    };
    part(P->spec, nspec * cs);
    {
        // the LDS limit is raised for every plan of the form, not to this one's size
        size_t lds;
        int form = pressure_form(g, precision, &lds);
        const bool f64 = precision == PYCLES_F64;
        const void *fn = form == PYCLES_PRESSURE_COLUMNS ? (f64 ? (const void *)thomas_lds_kernel<double> : (const void *)thomas_lds_kernel<float>)
                       : form == PYCLES_PRESSURE_PLANES ? (f64 ? (const void *)plane_solve_kernel<double, false> : (const void *)plane_solve_kernel<float, false>)
                                                        : (f64 ? (const void *)plane_solve_kernel<double, true> : (const void *)plane_solve_kernel<float, true>);
        if (form != PYCLES_PRESSURE_GENERAL && lds > 64 * 1024 &&
            hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess) {
            (void)hipGetLastError();
            form = PYCLES_PRESSURE_GENERAL;
        }
        P->thomas_lds = form == PYCLES_PRESSURE_COLUMNS;
        P->planes = form == PYCLES_PRESSURE_PLANES ? 1 : form == PYCLES_PRESSURE_PLANES_STAGED ? 2 : 0;
        P->plane_lds = lds;
        if (P->planes || P->thomas_lds) {
            part(P->pm, sizeof(double) * (size_t)g.nz * g.ny * P->nxh);
            part(P->pc, es * (size_t)g.nz * g.ny * P->nxh);
        } else {
            const int seg = precision == PYCLES_F64 ? thomas_seg<double>() : thomas_seg<float>();
            part(P->ck, 3 * sizeof(double) * (size_t)(g.nz / seg + 1) * g.ny * P->nxp);
        }
    }
    part(P->mean, (size_t)g.nzg * 8);
    part(P->partial, (size_t)g.nzg * MEAN_SPLITS * 8);
    const size_t tab0 = total;
    part(P->twx, (size_t)g.nx * cs);
    part(P->twy, (size_t)g.ny * cs);
    part(P->kx2, P->nxh * 8);
    part(P->ky2, g.ny * 8);
    part(P->rho_h, nz * 8);
    part(P->dd, nz * 8);
    part(P->a, nz * 8);
    part(P->c, nz * 8);
    std::vector<unsigned char> tables(total - tab0);
    if (hipMalloc(&P->mem, total) != hipSuccess) {
        (void)hipGetLastError();
        pycles_set_error("pressure: hipMalloc of %zu bytes failed", total);
        pycles_pressure_plan_destroy(P);
        return PYCLES_ERR_HIP;
    }
    for (int q = 0; q < nparts; ++q) *parts[q].ptr = (char *)P->mem + parts[q].off;
    auto put = [&](const void *dev, const double *v, int n, bool field) {
        unsigned char *h = tables.data() + ((const char *)dev - (const char *)P->mem - tab0);
        if (field && precision == PYCLES_F32)
            for (int m = 0; m < n; ++m) ((float *)h)[m] = (float)v[m];
        else
            memcpy(h, v, n * sizeof(double));
    };
    put(P->twx, twx.data(), 2 * g.nx, true);
    put(P->twy, twy.data(), 2 * g.ny, true);
    put(P->kx2, kx2.data(), P->nxh, false);
    put(P->ky2, ky2.data(), g.ny, false);
    put(P->rho_h, rh.data(), nz, false);
    put(P->dd, dd.data(), nz, false);
    put(P->a, a.data(), nz, false);
    put(P->c, c.data(), nz, false);
    hipError_t e = hipMemcpy((char *)P->mem + tab0, tables.data(), tables.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        pycles_set_error("pressure: table upload failed: %s", hipGetErrorString(e));
        pycles_pressure_plan_destroy(P);
        return PYCLES_ERR_HIP;
    }
    if (P->planes || P->thomas_lds) {
        const dim3 grid((unsigned)(((long long)g.ny * P->nxh + 63) / 64));
        // planes: [kx][level][ky]; otherwise [level][ky][kx]
        const long long sk = P->planes ? g.ny : (long long)g.ny * P->nxh, sy = P->planes ? 1 : P->nxh,
                        sx = P->planes ? (long long)g.nz * g.ny : 1;
        if (precision == PYCLES_F64)
            hipLaunchKernelGGL(pivot_kernel<double>, grid, dim3(64), 0, 0, g, P->kx2, P->ky2, P->rho_h, P->dd, P->a, P->c,
                               P->nxh, sk, sy, sx, P->pm, (double *)P->pc);
        else
            hipLaunchKernelGGL(pivot_kernel<float>, grid, dim3(64), 0, 0, g, P->kx2, P->ky2, P->rho_h, P->dd, P->a, P->c,
                               P->nxh, sk, sy, sx, P->pm, (float *)P->pc);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(0);  // any stream may use the plan
        if (e != hipSuccess) {
            pycles_set_error("pressure: pivots: %s", hipGetErrorString(e));
            pycles_pressure_plan_destroy(P);
            return PYCLES_ERR_HIP;
        }
    }
    *out = P;
    return PYCLES_OK;
}

extern "C" void pycles_pressure_plan_destroy(pycles_pressure_plan *P) {
    if (!P) return;
    if (P->mem) (void)hipFree(P->mem);
    delete P;
}

template <typename TS>
static int run_pressure(pycles_pressure_plan *P, const pycles_ref *ref, void *u, void *v, void *w, void *p,
                        void *div, double dt, double *cfl_out, hipStream_t st) {
    const Geo &g = P->g;
    int rc = pycles_level_partials(g, w, P->partial, P->precision, st);
    if (rc) return rc;
    // x transforms: S complex sequences (2S rows) per block, S nx/8 threads; as
    // many sequences as 2048 points hold, fewer on grids below 2 blocks per CU.
    // With less than four wavefronts per SIMD the divergence takes four times
    // the threads, four cells each (16 with S nx/8 threads, in four rounds of
    // loads and divisions); the transform's S nx/8 are the first of them.
    // 64^3 FP64: 11.4 us and 4.8 for the means' kernel -> 7.7 for both.
    int logS = 0;
    while ((g.nx << (logS + 1)) <= 2048 && (2 << (logS + 1)) <= g.ny) ++logS;
    while (logS > 0 && (long long)(g.ny >> (logS + 1)) * g.nz < 512 && (g.nx << logS) / 8 > 64) --logS;
    const int S = 1 << logS;
    const size_t rowsmem = sizeof(C2<TS>) * (size_t)g.nx * S;
    const int bx = S * g.nx / 8;
    const long long waves = (long long)(g.ny / (2 * S)) * g.nz * ((bx + 63) / 64);
    const int dbx = waves < 4096 && bx >= 32 && bx <= 128 ? 4 * bx : bx;
    constexpr int V = 16 / sizeof(TS);
    const bool wdiv = (((uintptr_t)u | (uintptr_t)v | (uintptr_t)w | (uintptr_t)div) & 15) == 0;
#define DIV_FFTX(TR_, V_)                                                                                      \
    hipLaunchKernelGGL((div_fftx_kernel<TS, TR_, V_>), dim3(g.ny / (2 * S), g.nz), dim3(dbx), rowsmem, st, g,       \
                       (const TS *)u, (const TS *)v, (const TS *)w, ref->alpha0, ref->alpha0_half, P->partial,  \
                       P->mean, cfl_out, (TS *)div, (C2<TS> *)P->spec, (const C2<TS> *)P->twx, P->logx, P->nxh, \
                       P->nxp, logS)
    // the plane form's small grids have four cells per thread: single cells there
    // (256 x 64 x 75 FP32, a projection and its RK3 stage: 73.5 us against 74.2)
    if (P->planes) DIV_FFTX(true, 1);
    else if (wdiv) DIV_FFTX(false, V);
    else DIV_FFTX(false, 1);
#undef DIV_FFTX
    PYCLES_CHECK_LAUNCH();
    if (P->planes) {
        // threads for all levels' transforms, or for the sweeps, up to 1024
        int pb = g.nz * (g.ny / 8);
        if (pb < 2 * g.ny) pb = 2 * g.ny;
        pb = pb > 1024 ? 1024 : (pb + 63) / 64 * 64;
        if (P->planes == 2)
            hipLaunchKernelGGL((plane_solve_kernel<TS, true>), dim3(P->nxh), dim3(pb), P->plane_lds, st, g,
                               (C2<TS> *)P->spec, P->pm, (const TS *)P->pc, P->a, (const C2<TS> *)P->twy, P->logy);
        else
            hipLaunchKernelGGL((plane_solve_kernel<TS, false>), dim3(P->nxh), dim3(pb), P->plane_lds, st, g,
                               (C2<TS> *)P->spec, P->pm, (const TS *)P->pc, P->a, (const C2<TS> *)P->twy, P->logy);
        PYCLES_CHECK_LAUNCH();
    } else {
        const size_t ysmem = sizeof(C2<TS>) * (size_t)g.ny * P->gx;
        const dim3 ygrid((P->nxh + P->gx - 1) / P->gx, g.nz);
        const int by = P->gx * g.ny / 8;
        hipLaunchKernelGGL(ffty_kernel<TS>, ygrid, dim3(by), ysmem, st, g, (C2<TS> *)P->spec,
                           (const C2<TS> *)P->twy, P->logy, P->nxh, P->nxp, P->gx, P->loggx, 0);
        PYCLES_CHECK_LAUNCH();
        const long long ncol = (long long)g.ny * P->nxp;
        if (P->thomas_lds)
            hipLaunchKernelGGL(thomas_lds_kernel<TS>, dim3((unsigned)(((long long)g.ny * P->nxh + TL_COLS - 1) / TL_COLS)),
                               dim3(256), thomas_lds_bytes<TS>(g.nz), st, g, (C2<TS> *)P->spec, P->pm, (const TS *)P->pc,
                               P->a, P->nxh, P->nxp);
        else
            hipLaunchKernelGGL((thomas_kernel<TS, thomas_seg<TS>()>), dim3((unsigned)((ncol + 255) / 256)), dim3(256),
                               4 * sizeof(double) * (size_t)g.nz, st, g, (C2<TS> *)P->spec, P->ck, P->kx2, P->ky2,
                               P->rho_h, P->dd, P->a, P->c, P->nxh, P->nxp);
        PYCLES_CHECK_LAUNCH();
        hipLaunchKernelGGL(ffty_kernel<TS>, ygrid, dim3(by), ysmem, st, g, (C2<TS> *)P->spec,
                           (const C2<TS> *)P->twy, P->logy, P->nxh, P->nxp, P->gx, P->loggx, 1);
        PYCLES_CHECK_LAUNCH();
    }
#define IFFTX(TR_)                                                                                             \
    hipLaunchKernelGGL((ifftx_kernel<TS, TR_>), dim3(g.ny / (2 * S), g.nz), dim3(bx), rowsmem, st, g,           \
                       (const C2<TS> *)P->spec, (TS *)p, (const C2<TS> *)P->twx, P->logx, P->nxh, P->nxp, logS)
    if (P->planes) IFFTX(true);
    else IFFTX(false);
#undef IFFTX
    PYCLES_CHECK_LAUNCH();
    const ZSplit zs = correct_zsplit(g.plane, g.nz, g.gw);
    const bool wide = (((uintptr_t)u | (uintptr_t)v | (uintptr_t)w | (uintptr_t)p) & 15) == 0;
    const dim3 cgrid((unsigned)((g.plane / (wide ? V : 1) + 255) / 256), zs.nch);
    if (wide)
        hipLaunchKernelGGL((correct_kernel<TS, V>), cgrid, dim3(256), 0, st, g, (TS *)u, (TS *)v, (TS *)w, (const TS *)p,
                           P->mean, dt, cfl_out, zs.len);
    else
        hipLaunchKernelGGL((correct_kernel<TS, 1>), cgrid, dim3(256), 0, st, g, (TS *)u, (TS *)v, (TS *)w, (const TS *)p,
                           P->mean, dt, cfl_out, zs.len);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

extern "C" int pycles_pressure_update(pycles_pressure_plan *P, const pycles_ref *ref, void *u, void *v, void *w,
                                      void *p, void *div, double dt, double *cfl_out, void *stream) {
    if (!P || !ref || !u || !v || !w || !p) {
        pycles_set_error("pressure_update: NULL argument");
        return PYCLES_ERR_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
    if (P->precision == PYCLES_F64) return run_pressure<double>(P, ref, u, v, w, p, div, dt, cfl_out, st);
    return run_pressure<float>(P, ref, u, v, w, p, div, dt, cfl_out, st);
}

extern "C" int pycles_divergence(const pycles_dims *dims, const pycles_ref *ref, const void *u, const void *v,
                                 const void *w, void *div, int precision, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!ref || !u || !v || !w || !div) {
        pycles_set_error("divergence: NULL argument");
        return PYCLES_ERR_ARG;
    }
    Geo g = make_geo(dims);
    hipStream_t st = (hipStream_t)stream;
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(divergence_kernel<double>, dim3(2048), dim3(256), 0, st, g, (const double *)u,
                           (const double *)v, (const double *)w, ref->alpha0, ref->alpha0_half, (double *)div);
    else
        hipLaunchKernelGGL(divergence_kernel<float>, dim3(2048), dim3(256), 0, st, g, (const float *)u,
                           (const float *)v, (const float *)w, ref->alpha0, ref->alpha0_half, (float *)div);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}
