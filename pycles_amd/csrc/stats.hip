// On-device horizontal statistics: per-level moments, maxima and minima of a
// field or of a product of two fields, optionally conditional on a mask, and
// the liquid-water statistics of the saturation adjustment.
//
//   HorizontalMean / MeanofSquares / MeanofCubes  ParallelMPI.pyx:196-326
//   HorizontalMaximum / HorizontalMinimum         ParallelMPI.pyx:327-389
//   HorizontalMeanConditional (+ofSquares)        ParallelMPI.pyx:430-540
//   ThermodynamicsSA.liquid_stats                 ThermodynamicsSA.pyx:395-492
//
// Every level is split over STAT_SPLITS blocks; each block reduces its share
// of the level in a fixed order into FP64 partials, and a second kernel adds
// the partials in split order, so the result does not depend on scheduling.
// The partials live in a caller-provided workspace.
#include <mutex>

#include "common.h"
#include "thermo_funcs.h"

extern int pycles_check_dims(const pycles_dims *d);

#define STAT_SPLITS 16
#define STAT_NQ 6  // sum v m, sum v^2 m, sum v^3 m, max, min, sum m
#define STAT_BLOCK 256

namespace {

// Moments and extremes of one share of a level.  B: the second factor is
// given; M: the mask is given (without one every weight is 1 and the count is
// the share's size); V cells per access (16 bytes where the level, the shares
// and the pointers allow it), four accesses per thread in flight.
// Bound: HBM, one read of the field(s).  512 x 512 x 262 levels FP32: 122 -> 50
// us (5.5 TB/s; one 4-byte load a thread in flight before), with a product 88.
template <typename T, bool B, bool M, int V>
__global__ __launch_bounds__(STAT_BLOCK) void stats_partial_kernel(Geo g, const T *a, const double *base_a,
                                                                   const T *b, const double *base_b,
                                                                   const T *mask, double *partial, long long per) {
    typedef T VT __attribute__((ext_vector_type(V)));
    constexpr int U = 4;
    const int k = blockIdx.x;
    const int sp = blockIdx.y;
    const long long n = g.plane;
    const long long lo = sp * per < n ? sp * per : n;
    const long long hi = lo + per < n ? lo + per : n;
    const long long off = (long long)k * n;
    const double ba = base_a ? base_a[k] : 0.0;
    const double bb = B && base_b ? base_b[k] : 0.0;
    double s1 = 0.0, s2 = 0.0, s3 = 0.0, sm = 0.0;
    double mx = -9e12, mn = 9e12;  // the reference's initial extremes
    auto add = [&](T av, T bv, T mv) {
        double v = (double)av + ba;
        if (B) v *= (double)bv + bb;
        if (M) {
            const double m = (double)mv;
            s1 += v * m;
            s2 += v * v * m;
            s3 += v * v * v * m;
            sm += m;
            if (m != 0.0) {
                mx = fmax(mx, v);
                mn = fmin(mn, v);
            }
        } else {
            s1 += v;
            s2 += v * v;
            s3 += v * v * v;
            mx = fmax(mx, v);
            mn = fmin(mn, v);
        }
    };
    for (long long c = lo + threadIdx.x * V; c < hi; c += U * STAT_BLOCK * V) {
        VT av[U], bv[U], mv[U];
#pragma unroll
        for (int q = 0; q < U; ++q) {
            // clamped to the share's first access past its end: loaded, not used
            const long long o = off + (c + q * STAT_BLOCK * V < hi ? c + q * STAT_BLOCK * V : lo);
            av[q] = __builtin_nontemporal_load(reinterpret_cast<const VT *>(a + o));
            if (B) bv[q] = __builtin_nontemporal_load(reinterpret_cast<const VT *>(b + o));
            if (M) mv[q] = __builtin_nontemporal_load(reinterpret_cast<const VT *>(mask + o));
        }
#pragma unroll
        for (int q = 0; q < U; ++q) {
            if (c + q * STAT_BLOCK * V >= hi) break;
#pragma unroll
            for (int e = 0; e < V; ++e) add(av[q][e], B ? bv[q][e] : T(0), M ? mv[q][e] : T(0));
        }
    }
    // fixed-order sums: over the lanes by shuffles, then over the wavefronts
    double r[STAT_NQ] = {s1, s2, s3, mx, mn, sm};
    for (int s = 32; s > 0; s >>= 1) {
#pragma unroll
        for (int q = 0; q < STAT_NQ; ++q) {
            const double o = __shfl_down(r[q], s, 64);
            r[q] = q == 3 ? fmax(r[q], o) : (q == 4 ? fmin(r[q], o) : r[q] + o);
        }
    }
    __shared__ double red[STAT_NQ][STAT_BLOCK / 64];
    if (threadIdx.x % 64 == 0)
#pragma unroll
        for (int q = 0; q < STAT_NQ; ++q) red[q][threadIdx.x / 64] = r[q];
    __syncthreads();
    if (threadIdx.x < STAT_NQ) {
        const int q = threadIdx.x;
        const double *w = red[q];
        double v = q == 3 ? fmax(fmax(w[0], w[1]), fmax(w[2], w[3]))
                          : (q == 4 ? fmin(fmin(w[0], w[1]), fmin(w[2], w[3])) : (w[0] + w[1]) + (w[2] + w[3]));
        if (!M && q == 5) v = (double)(hi - lo);
        partial[((long long)k * STAT_SPLITS + sp) * STAT_NQ + q] = v;
    }
}

// One thread per level and quantity; the shares in order.
__global__ void stats_final_kernel(Geo g, const double *partial, int masked, double *out) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)g.nzg * STAT_NQ) return;
    const int k = (int)(t / STAT_NQ), q = (int)(t % STAT_NQ);
    double v[STAT_SPLITS], m[STAT_SPLITS];
#pragma unroll
    for (int sp = 0; sp < STAT_SPLITS; ++sp) {
        const double *p = partial + ((long long)k * STAT_SPLITS + sp) * STAT_NQ;
        v[sp] = p[q];
        m[sp] = p[5];
    }
    double s = q == 3 ? -9e12 : (q == 4 ? 9e12 : 0.0), sm = 0.0;
#pragma unroll
    for (int sp = 0; sp < STAT_SPLITS; ++sp) {
        s = q == 3 ? fmax(s, v[sp]) : (q == 4 ? fmin(s, v[sp]) : s + v[sp]);
        sm += m[sp];
    }
    // unconditional means multiply by 1/(n0*n1) as the reference does;
    // conditional ones divide by max(sum m, 1)
    if (q < 3) s = masked ? s / fmax(sm, 1.0) : s * (1.0 / (double)((long long)g.ny * g.nx));
    out[(long long)q * g.nzg + k] = s;
}

// Liquid-water statistics.  A block takes groups of 64 columns; each of its
// four wavefronts marches a quarter of the levels, eight loads at a time.  A
// level's cloudy cells are counted by ballot (one wavefront owns a level, so
// the LDS counter needs no atomic) and added to the global counters once per
// block (integer adds are exact, so the order does not matter); the liquid
// water path is summed per column over the quarters in order, per block over
// its groups and columns in a fixed order, and over the blocks in
// cloud_final_kernel.  Dynamic LDS: nz + 1 counters.
// Bound: HBM, one read of ql.  512 x 512 x 256 FP32: 141 -> 85 us
// (one thread per column, one load at a time before), and the block sums 105
// -> 6 us (one thread before).
constexpr int CLOUD_COLS = 64, CLOUD_Q = STAT_BLOCK / CLOUD_COLS, CLOUD_MAX_BLOCKS = 2048;
static int cloud_blocks(const Geo &g) {
    const long long n = (g.plane + CLOUD_COLS - 1) / CLOUD_COLS;
    return (int)(n < CLOUD_MAX_BLOCKS ? n : CLOUD_MAX_BLOCKS);
}
template <typename T>
__global__ __launch_bounds__(STAT_BLOCK) void cloud_kernel(Geo g, const T *ql, const double *__restrict__ rho0_half,
                                                           unsigned long long *counts, double *lwp_part) {
    extern __shared__ unsigned int lcount[];
    __shared__ double red[CLOUD_Q][CLOUD_COLS];
    __shared__ int wet[CLOUD_Q][CLOUD_COLS];
    for (int k = threadIdx.x; k <= g.nz; k += STAT_BLOCK) lcount[k] = 0u;
    __syncthreads();
    const int lane = threadIdx.x % CLOUD_COLS;
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / CLOUD_COLS);
    const int len = (g.nz + CLOUD_Q - 1) / CLOUD_Q;
    const int k0 = min(part * len, g.nz), k1 = min(k0 + len, g.nz);
    const long long groups = (g.plane + CLOUD_COLS - 1) / CLOUD_COLS;
    double total = 0.0;  // this lane's columns, first wavefront
    for (long long grp = blockIdx.x; grp < groups; grp += gridDim.x) {
        const long long c = grp * CLOUD_COLS + lane;
        const bool in = c < g.plane;
        const T *col = ql + (long long)g.gw * g.plane + (in ? c : 0);
        double lwp = 0.0;
        int cloudy = 0;
        for (int kb = k0; kb < k1; kb += 8) {
            T v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = __builtin_nontemporal_load(col + (long long)min(kb + q, k1 - 1) * g.plane);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int k = kb + q;
                if (k >= k1) break;
                const double x = (double)v[q];
                const bool w = in && x > 0.0;
                cloudy |= w;
                const unsigned long long m = __ballot(w);
                if (m && lane == 0) lcount[k] += (unsigned)__popcll(m);
                // ThermodynamicsSA.pyx:478-480 weights interior level k with
                // rho0_half[k], the ghosted array's k-th entry
                lwp += rho0_half[k] * x * g.dx[2];
            }
        }
        red[part][lane] = in ? lwp : 0.0;
        wet[part][lane] = cloudy;
        __syncthreads();
        if (part == 0) {
            int any = 0;
            for (int q = 0; q < CLOUD_Q; ++q) {
                total += red[q][lane];
                any |= wet[q][lane];
            }
            const unsigned long long m = __ballot(any);
            if (m && lane == 0) lcount[g.nz] += (unsigned)__popcll(m);
        }
        __syncthreads();
    }
    if (part == 0) {
        for (int s = 32; s > 0; s >>= 1) total += __shfl_down(total, s, 64);
        if (lane == 0) lwp_part[blockIdx.x] = total;
    }
    for (int k = threadIdx.x; k <= g.nz; k += STAT_BLOCK)
        if (lcount[k]) atomicAdd(&counts[k], (unsigned long long)lcount[k]);
}

__global__ void zero_u64_kernel(unsigned long long *p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

// out: cloud fraction profile [nz], then cloud cover, cloud base, cloud top,
// liquid water path (ThermodynamicsSA.pyx:433-489).  Base and top are the
// centre heights z_half = (k + 1/2) dz of the lowest and highest level with a
// cloudy cell; 99999.9 and -99999.9 when there is none, as the reference's
// initial values.
// One block: the levels and the block sums are dealt over its threads.
__global__ __launch_bounds__(STAT_BLOCK) void cloud_final_kernel(Geo g, const unsigned long long *counts,
                                                                 const double *lwp_part, int nblk, double *out) {
    __shared__ double rb[STAT_BLOCK], rt[STAT_BLOCK], rl[STAT_BLOCK];
    const int t = threadIdx.x;
    const double inv = 1.0 / (double)((long long)g.ny * g.nx);
    double cb = 99999.9, ct = -99999.9, lwp = 0.0;
    for (int k = t; k < g.nz; k += STAT_BLOCK) {
        out[k] = (double)counts[k] * inv;
        if (counts[k]) {
            const double z = ((double)k + 0.5) * g.dx[2];
            cb = fmin(cb, z);
            ct = fmax(ct, z);
        }
    }
    for (int b = t; b < nblk; b += STAT_BLOCK) lwp += lwp_part[b];
    rb[t] = cb;
    rt[t] = ct;
    rl[t] = lwp;
    __syncthreads();
    for (int s = STAT_BLOCK / 2; s > 0; s >>= 1) {
        if (t < s) {
            rb[t] = fmin(rb[t], rb[t + s]);
            rt[t] = fmax(rt[t], rt[t + s]);
            rl[t] += rl[t + s];
        }
        __syncthreads();
    }
    if (t != 0) return;
    // the column counts and the path are divided by n0*n1 as the reference
    // does (:461, :484); the fraction profile adds 1/(n0*n1) per cloudy cell
    // there, which the count times that reciprocal gives to a few ulps
    const double div = (double)((long long)g.ny * g.nx);
    out[g.nz] = (double)counts[g.nz] / div;
    out[g.nz + 1] = rb[0];
    out[g.nz + 2] = rt[0];
    out[g.nz + 3] = rl[0] / div;
}

// Fields of ThermodynamicsSA.stats_io (ThermodynamicsSA.pyx:256-389) at
// every stored point: the entropy potential temperature thetas_c(s, qt), the
// dry potential temperature theta_c(p0_half, T) and the relative humidity
// pv_c(p0_half, qt, qv) / pv*(T) (thermodynamic_functions.h:9-12, 23-25,
// 39-41; lookup.h:48-54), in the field precision.
template <typename TS>
__global__ __launch_bounds__(256) void sa_stat_fields_kernel(Geo g, const double *p0_half, thermo::Table lt,
                                                             const TS *s, const TS *qt, const TS *T, const TS *qv,
                                                             const double *sbase, const double *qbase,
                                                             TS *thetas, TS *theta, TS *rh) {
    const long long n = g.plane * g.nzg;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x) {
        const int k = (int)(t / g.plane);
        const double sv = (double)s[t] + (sbase ? sbase[k] : 0.0);
        const double q = (double)qt[t] + (qbase ? qbase[k] : 0.0);
        const double Tv = (double)T[t];
        if (thetas)
            thetas[t] = (TS)(PC_T_TILDE * exp((sv - (1.0 - q) * PC_SD_TILDE - q * PC_SV_TILDE) / thermo::cpm_c(q)));
        if (theta) theta[t] = (TS)(Tv / thermo::exner_c(p0_half[k]));
        if (rh) {
            const double pv_star = thermo::lookup(lt, Tv);
            const double pv = thermo::pv_c(p0_half[k], q, (double)qv[t]);
            rh[t] = (TS)(pv / pv_star);
        }
    }
}

}  // namespace

extern "C" int pycles_sa_stat_fields(const pycles_dims *dims, const pycles_ref *ref, const pycles_lookup *lt,
                                     const void *s, const void *qt, const void *T, const void *qv,
                                     const pycles_scalar_base *base, int precision, void *thetas, void *theta,
                                     void *rh, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!ref || !ref->p0_half || !lt || !lt->y || !s || !qt || !T || !qv) {
        pycles_set_error("sa_stat_fields: NULL argument");
        return PYCLES_ERR_ARG;
    }
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("sa_stat_fields: bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    const Geo g = make_geo(dims);
    thermo::Table t{lt->y, lt->x_min, lt->dx, lt->dxi, (int)lt->n};
    const double *sb = (precision == PYCLES_F32 && base) ? base->base[0] : nullptr;
    const double *qb = (precision == PYCLES_F32 && base) ? base->base[1] : nullptr;
    hipStream_t st = (hipStream_t)stream;
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(sa_stat_fields_kernel<double>, dim3(4096), dim3(256), 0, st, g, ref->p0_half, t,
                           (const double *)s, (const double *)qt, (const double *)T, (const double *)qv, sb, qb,
                           (double *)thetas, (double *)theta, (double *)rh);
    else
        hipLaunchKernelGGL(sa_stat_fields_kernel<float>, dim3(4096), dim3(256), 0, st, g, ref->p0_half, t,
                           (const float *)s, (const float *)qt, (const float *)T, (const float *)qv, sb, qb,
                           (float *)thetas, (float *)theta, (float *)rh);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

static size_t stats_ws_bytes(const Geo &g) { return sizeof(double) * (size_t)g.nzg * STAT_SPLITS * STAT_NQ; }

extern "C" size_t pycles_horizontal_stats_workspace_bytes(const pycles_dims *dims) {
    if (pycles_check_dims(dims)) return 0;
    const Geo g = make_geo(dims);
    return stats_ws_bytes(g);
}

static int stats_args(const pycles_dims *dims, const void *a, int precision, double *out) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!a || !out) {
        pycles_set_error("horizontal_stats: NULL field or output");
        return PYCLES_ERR_ARG;
    }
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("horizontal_stats: bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    return PYCLES_OK;
}

template <typename T, int V>
static void stats_partials(const Geo &g, const T *a, const double *base_a, const T *b, const double *base_b, const T *mask,
                           double *partial, hipStream_t st) {
    const dim3 grid(g.nzg, STAT_SPLITS), blk(STAT_BLOCK);
    // equal shares of a level, whole accesses each
    const long long per = ((g.plane + STAT_SPLITS - 1) / STAT_SPLITS + V - 1) / V * V;
#define STATS(B_, M_) \
    hipLaunchKernelGGL((stats_partial_kernel<T, B_, M_, V>), grid, blk, 0, st, g, a, base_a, b, base_b, mask, partial, per)
    if (b && mask) STATS(true, true);
    else if (b) STATS(true, false);
    else if (mask) STATS(false, true);
    else STATS(false, false);
#undef STATS
}

static int stats_launch(const Geo &g, const void *a, const double *base_a, const void *b, const double *base_b,
                        const void *mask, int precision, double *out, double *partial, hipStream_t st) {
    // 16-byte accesses where every level of every field starts on 16 bytes
    const int vmax = precision == PYCLES_F64 ? 2 : 4;
    const bool wide = g.plane % vmax == 0 && (((uintptr_t)a | (uintptr_t)b | (uintptr_t)mask) & 15) == 0;
    if (precision == PYCLES_F64) {
        if (wide) stats_partials<double, 2>(g, (const double *)a, base_a, (const double *)b, base_b, (const double *)mask, partial, st);
        else stats_partials<double, 1>(g, (const double *)a, base_a, (const double *)b, base_b, (const double *)mask, partial, st);
    } else {
        if (wide) stats_partials<float, 4>(g, (const float *)a, base_a, (const float *)b, base_b, (const float *)mask, partial, st);
        else stats_partials<float, 1>(g, (const float *)a, base_a, (const float *)b, base_b, (const float *)mask, partial, st);
    }
    PYCLES_CHECK_LAUNCH();
    const unsigned fb = (unsigned)(((long long)g.nzg * STAT_NQ + 63) / 64);
    hipLaunchKernelGGL(stats_final_kernel, dim3(fb), dim3(64), 0, st, g, partial, mask ? 1 : 0, out);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

extern "C" int pycles_horizontal_stats(const pycles_dims *dims, const void *a, const double *base_a, const void *b,
                                       const double *base_b, const void *mask, int precision, double *out,
                                       void *workspace, void *stream) {
    int rc = stats_args(dims, a, precision, out);
    if (rc) return rc;
    if (!workspace) {
        pycles_set_error("horizontal_stats: NULL workspace");
        return PYCLES_ERR_ARG;
    }
    const Geo g = make_geo(dims);
    return stats_launch(g, a, base_a, b, base_b, mask, precision, out, (double *)workspace, (hipStream_t)stream);
}

// No-allocation variant of pycles_horizontal_stats for callers that cannot
// allocate device memory.  Its partials live in a file-scope device array,
// one copy per GPU, whose address each device resolves once (with that
// device current) by hipGetSymbolAddress; host code passes only that
// address, never the array's name.  Every (level, split) slot is written by
// stats_partial_kernel before stats_final_kernel reads it, so nothing needs
// clearing between calls.  All calls on one GPU share the array: calls that
// overlap on one GPU (two streams, two host threads) race.
#define STATS_NOALLOC_MAX_LEVELS 2048
#define STATS_NOALLOC_MAX_DEVICES 64
static __device__ __align__(256) double scratch[(size_t)STATS_NOALLOC_MAX_LEVELS * STAT_SPLITS * STAT_NQ];
static double *g_scratch_dev[STATS_NOALLOC_MAX_DEVICES];
static std::mutex g_scratch_mu;

static int stats_scratch(double **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= STATS_NOALLOC_MAX_DEVICES) {
        pycles_set_error("horizontal_stats_noalloc: no usable current device (%d, %s)", dev, hipGetErrorString(e));
        return PYCLES_ERR_HIP;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            pycles_set_error("horizontal_stats_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
            return PYCLES_ERR_HIP;
        }
        g_scratch_dev[dev] = (double *)ptr;
    }
    *out = g_scratch_dev[dev];
    return PYCLES_OK;
}

extern "C" int pycles_horizontal_stats_noalloc(const pycles_dims *dims, const void *a, const double *base_a,
                                               const void *b, const double *base_b, const void *mask,
                                               int precision, double *out, void *stream) {
    int rc = stats_args(dims, a, precision, out);
    if (rc) return rc;
    const Geo g = make_geo(dims);
    if (g.nzg > STATS_NOALLOC_MAX_LEVELS) {
        pycles_set_error("horizontal_stats_noalloc: %d levels (with ghosts) exceed the scratch limit of %d",
                         g.nzg, STATS_NOALLOC_MAX_LEVELS);
        return PYCLES_ERR_UNSUPPORTED;
    }
    double *partial = nullptr;
    rc = stats_scratch(&partial);
    if (rc) return rc;
    return stats_launch(g, a, base_a, b, base_b, mask, precision, out, partial, (hipStream_t)stream);
}

extern "C" size_t pycles_cloud_stats_workspace_bytes(const pycles_dims *dims) {
    if (pycles_check_dims(dims)) return 0;
    const Geo g = make_geo(dims);
    return sizeof(unsigned long long) * (size_t)(g.nz + 1) + sizeof(double) * (size_t)cloud_blocks(g);
}

extern "C" int pycles_cloud_stats(const pycles_dims *dims, const double *rho0_half, const void *ql, int precision,
                                  double *out, void *workspace, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!rho0_half || !ql || !out || !workspace) {
        pycles_set_error("cloud_stats: NULL argument");
        return PYCLES_ERR_ARG;
    }
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("cloud_stats: bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    const Geo g = make_geo(dims);
    hipStream_t st = (hipStream_t)stream;
    unsigned long long *counts = (unsigned long long *)workspace;
    double *part = (double *)(counts + (g.nz + 1));
    const int nblk = cloud_blocks(g);
    hipLaunchKernelGGL(zero_u64_kernel, dim3((g.nz + 1 + 255) / 256), dim3(256), 0, st, counts, g.nz + 1);
    const size_t lds = sizeof(unsigned int) * (size_t)(g.nz + 1);
    if (lds > 48 * 1024) {
        pycles_set_error("cloud_stats: %d levels exceed the kernel's LDS counters", g.nz);
        return PYCLES_ERR_UNSUPPORTED;
    }
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(cloud_kernel<double>, dim3(nblk), dim3(STAT_BLOCK), lds, st, g, (const double *)ql,
                           rho0_half, counts, part);
    else
        hipLaunchKernelGGL(cloud_kernel<float>, dim3(nblk), dim3(STAT_BLOCK), lds, st, g, (const float *)ql,
                           rho0_half, counts, part);
    PYCLES_CHECK_LAUNCH();
    hipLaunchKernelGGL(cloud_final_kernel, dim3(1), dim3(STAT_BLOCK), 0, st, g, counts, part, nblk, out);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}
