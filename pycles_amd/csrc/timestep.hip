// SSP-RK3 stage update with the z boundary fill, the z boundary fill alone,
// level means, CFL maximum and layout conversion.
//
//   TimeStepping.update_third     TimeStepping.pyx:131-151
//   set_bcs (sym / asym)          prognostic_variables.h:205-270
//   ParallelMPI.HorizontalMean    ParallelMPI.pyx:196-241
//   compute_cfl_max               TimeStepping.pyx:222-263
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include "common.h"

static thread_local char g_err[1024] = "";

void pycles_set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

extern "C" const char *pycles_last_error(void) { return g_err; }
extern "C" const char *pycles_version(void) { return "pycles_amd 0.1 (gfx950)"; }
extern "C" int pycles_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int pycles_check_dims(const pycles_dims *d) {
    if (!d) {
        pycles_set_error("dims is NULL");
        return PYCLES_ERR_ARG;
    }
    for (int i = 0; i < 3; ++i)
        if (d->n[i] < 1 || d->n[i] > (1 << 20)) {
            pycles_set_error("dims.n[%d] = %lld out of range", i, (long long)d->n[i]);
            return PYCLES_ERR_ARG;
        }
    if (d->gw < 2 || d->gw > 8 || d->gw > d->n[2]) {
        pycles_set_error("dims.gw = %lld out of range", (long long)d->gw);
        return PYCLES_ERR_ARG;
    }
    const long long npts = d->n[0] * d->n[1] * (d->n[2] + 2 * d->gw);
    if (npts >= (1LL << 40)) {
        pycles_set_error("domain too large");
        return PYCLES_ERR_ARG;
    }
    return PYCLES_OK;
}

// Mirror one column's ghost levels after its interior is final.
template <typename T>
__device__ __forceinline__ void fill_column_bcs(T *f, long long col, long long plane, int gw, int nzg,
                                                double bc) {
    if (bc == 1.0) {
        for (int m = 0; m < gw; ++m) {
            f[(long long)(gw - 1 - m) * plane + col] = f[(long long)(gw + m) * plane + col];
            f[(long long)(nzg - gw + m) * plane + col] = f[(long long)(nzg - gw - 1 - m) * plane + col];
        }
    } else if (bc == 2.0) {
        for (int m = 0; m < gw; ++m) {
            f[(long long)(gw - 1 - m) * plane + col] = f[(long long)gw * plane + col];
            f[(long long)(nzg - gw + m) * plane + col] = f[(long long)(nzg - gw - 1) * plane + col];
        }
    } else {
        const T fac = (T)bc;
        f[(long long)(gw - 1) * plane + col] = T(0);
        f[(long long)(nzg - gw) * plane + col] = T(0);
        for (int m = 1; m < gw; ++m) {
            f[(long long)(gw - 1 - m) * plane + col] = fac * f[(long long)(gw - 1 + m) * plane + col];
            f[(long long)(nzg - gw + m) * plane + col] = fac * f[(long long)(nzg - gw - m) * plane + col];
        }
    }
}

struct PtrPack {
    void *v[8];
    void *t[8];
    void *c[8];
    double bc[8];
};

// RK3 stage of the interior, V consecutive cells of one level per thread, with
// the z ghost levels that the cell feeds (the values fill_column_bcs gives:
// every ghost level's source is an interior level).  Grid: a level's blocks in
// x, the levels in y (looped over where they exceed the grid's limit), the
// variables in z, so that each array is swept from end to end (with the
// variables inside the levels the 512 x 512 x 256 FP64 stage took 1.93 ms).
// Bound: HBM, 4 field passes (value, tendency and copy read, value written; a
// stage 0 writes the copy instead of reading it).  Accesses are 16 bytes wide
// where the plane and every pointer allow it (V = 16 / sizeof(T)), and a level
// is split over blocks so that a small grid fills the chip: one thread per
// column marching all levels left a 64 x 64 grid on 16 CUs per variable.
// 512 x 512 x 256 FP64, five fields: 2.24 -> 1.71 ms (6.3 TB/s, what a copy
// reaches); 256 x 64 x 75 FP32 19 -> 18 us (5.4).
template <typename T, int V> struct RkVec {
    typedef T type __attribute__((ext_vector_type(V)));
};
template <typename T, int RK, int V>
__global__ __launch_bounds__(256) void rk3_kernel(Geo g, PtrPack pk, double dtd, int zero_tend) {
    using VT = typename RkVec<T, V>::type;
    const int v = blockIdx.z;
    const long long e = ((long long)blockIdx.x * 256 + threadIdx.x) * V;
    if (e >= g.plane) return;
    const long long P = g.plane;
    const int gw = g.gw, nzg = g.nzg;
    const T dt = (T)dtd;
    T *val = (T *)pk.v[v];
    T *ten = (T *)pk.t[v];
    T *cpy = (T *)pk.c[v];
    auto get = [](const T *p) { return __builtin_nontemporal_load(reinterpret_cast<const VT *>(p)); };
    auto put = [](T *p, VT x) { __builtin_nontemporal_store(x, reinterpret_cast<VT *>(p)); };
    const double bc = pk.bc[v];
    for (int k = gw + blockIdx.y; k < gw + g.nz; k += gridDim.y) {
        const long long o = (long long)k * P + e;
        const VT phi = get(val + o), tn = get(ten + o);
        VT cp = VT(T(0));
        if (RK > 0) cp = get(cpy + o);
        VT x;
#pragma unroll
        for (int q = 0; q < V; ++q) x[q] = rk_update<T, RK>(phi[q], tn[q], cp[q], dt);
        put(val + o, x);
        if (RK == 0) put(cpy + o, phi);
        if (zero_tend) {
            // the reference zeroes every tendency, ghost levels included (the SA
            // buoyancy writes w tendencies on low ghost levels)
            put(ten + o, VT(T(0)));
            if (k < 2 * gw) {
                put(ten + (long long)(k - gw) * P + e, VT(T(0)));
                put(ten + (long long)(nzg - 1 - (k - gw)) * P + e, VT(T(0)));
            }
        }
        if (k >= 2 * gw && k < nzg - 2 * gw) continue;
        if (bc == 1.0) {
            if (k < 2 * gw) put(val + (long long)(2 * gw - 1 - k) * P + e, x);
            if (k >= nzg - 2 * gw) put(val + (long long)(2 * (nzg - gw) - 1 - k) * P + e, x);
        } else if (bc == 2.0) {
            for (int m = 0; m < gw; ++m) {
                if (k == gw) put(val + (long long)m * P + e, x);
                if (k == nzg - gw - 1) put(val + (long long)(nzg - 1 - m) * P + e, x);
            }
        } else {
            const VT y = (T)bc * x;
            if (k == gw) put(val + (long long)(gw - 1) * P + e, VT(T(0)));
            if (k == nzg - gw - 1) put(val + (long long)(nzg - gw) * P + e, VT(T(0)));
            if (k <= 2 * gw - 2) put(val + (long long)(2 * gw - 2 - k) * P + e, y);
            if (k >= nzg - 2 * gw + 1) put(val + (long long)(2 * (nzg - gw) - k) * P + e, y);
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void bcs_kernel(Geo g, int nv, PtrPack pk) {
    const long long col = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= g.plane) return;
    for (int v = 0; v < nv; ++v) fill_column_bcs((T *)pk.v[v], col, g.plane, g.gw, g.nzg, pk.bc[v]);
}

static int pack(int nv, void *const *values, void *const *tend, void *const *copies, const double *bc,
                PtrPack *pk) {
    if (nv < 1 || nv > 8) {
        pycles_set_error("nv = %d out of range [1, 8]", nv);
        return PYCLES_ERR_ARG;
    }
    memset(pk, 0, sizeof(*pk));
    for (int v = 0; v < nv; ++v) {
        pk->v[v] = values[v];
        pk->t[v] = tend ? tend[v] : nullptr;
        pk->c[v] = copies ? copies[v] : nullptr;
        pk->bc[v] = bc[v];
        if (!pk->v[v] || (tend && !pk->t[v]) || (copies && !pk->c[v])) {
            pycles_set_error("NULL field pointer for variable %d", v);
            return PYCLES_ERR_ARG;
        }
    }
    return PYCLES_OK;
}

extern "C" int pycles_rk3_stage(const pycles_dims *dims, int nv, void *const *values, void *const *tend,
                                void *const *copies, const double *bc_type, int rk_step, double dt,
                                int precision, int zero_tendencies, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (rk_step < 0 || rk_step > 2 || !tend || !copies || !values || !bc_type) {
        pycles_set_error("rk3_stage: bad arguments");
        return PYCLES_ERR_ARG;
    }
    PtrPack pk;
    if ((rc = pack(nv, values, tend, copies, bc_type, &pk))) return rc;
    Geo g = make_geo(dims);
    hipStream_t st = (hipStream_t)stream;
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    const int zt = zero_tendencies ? 1 : 0;
    // 16-byte accesses where every level of every array starts on 16 bytes
    const int vmax = precision == PYCLES_F64 ? 2 : 4;
    bool wide = g.plane % vmax == 0;
    for (int v = 0; v < nv; ++v)
        wide = wide && (((uintptr_t)pk.v[v] | (uintptr_t)pk.t[v] | (uintptr_t)pk.c[v]) & 15) == 0;
    const long long per = 256LL * (wide ? vmax : 1);
    const dim3 grid((unsigned)((g.plane + per - 1) / per), g.nz < 65535 ? g.nz : 65535, nv);
#define RK_LAUNCH(T, R)                                                                              \
    do {                                                                                             \
        if (wide)                                                                                    \
            hipLaunchKernelGGL((rk3_kernel<T, R, 16 / sizeof(T)>), grid, dim3(256), 0, st, g, pk, dt, zt); \
        else                                                                                         \
            hipLaunchKernelGGL((rk3_kernel<T, R, 1>), grid, dim3(256), 0, st, g, pk, dt, zt);    \
    } while (0)
    if (precision == PYCLES_F64) {
        if (rk_step == 0) RK_LAUNCH(double, 0);
        else if (rk_step == 1) RK_LAUNCH(double, 1);
        else RK_LAUNCH(double, 2);
    } else {
        if (rk_step == 0) RK_LAUNCH(float, 0);
        else if (rk_step == 1) RK_LAUNCH(float, 1);
        else RK_LAUNCH(float, 2);
    }
#undef RK_LAUNCH
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

extern "C" int pycles_apply_z_bcs(const pycles_dims *dims, int nv, void *const *values,
                                  const double *bc_type, int precision, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!values || !bc_type) {
        pycles_set_error("apply_z_bcs: NULL argument");
        return PYCLES_ERR_ARG;
    }
    PtrPack pk;
    if ((rc = pack(nv, values, nullptr, nullptr, bc_type, &pk))) return rc;
    Geo g = make_geo(dims);
    const int B = 256;
    const unsigned grid = (unsigned)((g.plane + B - 1) / B);
    hipStream_t st = (hipStream_t)stream;
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(bcs_kernel<double>, dim3(grid), dim3(B), 0, st, g, nv, pk);
    else if (precision == PYCLES_F32)
        hipLaunchKernelGGL(bcs_kernel<float>, dim3(grid), dim3(B), 0, st, g, nv, pk);
    else {
        pycles_set_error("bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

// ---------------------------------------------------------------------------
// Level sums: partial sums per (level, split) in FP64, in a fixed order, so the
// result does not depend on scheduling; the projection adds the splits in order.
#define MEAN_SPLITS 16

template <typename T>
__global__ __launch_bounds__(256) void level_partial_kernel(Geo g, const T *f, double *partial) {
    const int k = blockIdx.x;
    const int sp = blockIdx.y;
    const long long n = g.plane;
    const long long per = (n + MEAN_SPLITS - 1) / MEAN_SPLITS;
    const long long lo = sp * per;
    const long long hi = lo + per < n ? lo + per : n;
    const T *row = f + (long long)k * n;
    // four independent sums in flight per thread (fixed order: deterministic)
    const int B = blockDim.x;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    long long c = lo + threadIdx.x;
    for (; c + 3 * B < hi; c += 4 * B) {
        a0 += (double)row[c];
        a1 += (double)row[c + B];
        a2 += (double)row[c + 2 * B];
        a3 += (double)row[c + 3 * B];
    }
    for (; c < hi; c += B) a0 += (double)row[c];
    double acc = (a0 + a1) + (a2 + a3);
    // wavefront sum by lane shuffles, then the block's four wavefronts
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[(long long)k * MEAN_SPLITS + sp] = (red[0] + red[1]) + (red[2] + red[3]);
}

// partial[k][MEAN_SPLITS]: the split sums of every level (pressure.hip)
int pycles_level_partials(const Geo &g, const void *field, double *partial, int precision, hipStream_t st) {
    const dim3 grid(g.nzg, MEAN_SPLITS);
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(level_partial_kernel<double>, grid, dim3(256), 0, st, g, (const double *)field, partial);
    else
        hipLaunchKernelGGL(level_partial_kernel<float>, grid, dim3(256), 0, st, g, (const float *)field, partial);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

// Standalone entries: one block per level and field (no workspace needed).
// Each thread adds its cells in order, eight loads ahead of their additions,
// then the block's sums in a fixed tree.  Bound: latency (a launch and one
// round of loads) on small planes: one call for the five prognostic fields of
// 64 x 64 x 81 levels instead of five,
// 4 us against 5 x 6.
struct MeanPack {
    const void *f[8];
};
template <typename T>
__global__ __launch_bounds__(256) void level_mean_kernel(Geo g, MeanPack pk, double *mean) {
    constexpr int U = 8, B = 256;
    const int k = blockIdx.x, v = blockIdx.y;
    const T *row = (const T *)pk.f[v] + (long long)k * g.plane;
    double acc = 0.0;
    long long c = threadIdx.x;
    for (; c + (U - 1) * B < g.plane; c += U * B) {
        T x[U];
#pragma unroll
        for (int q = 0; q < U; ++q) x[q] = row[c + q * B];
#pragma unroll
        for (int q = 0; q < U; ++q) acc += (double)x[q];
    }
    for (; c < g.plane; c += B) acc += (double)row[c];
    __shared__ double red[B];
    red[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x < 128) red[threadIdx.x] += red[threadIdx.x + 128];
    __syncthreads();
    if (threadIdx.x < 64) {
        double s = red[threadIdx.x] + red[threadIdx.x + 64];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
        if (threadIdx.x == 0) mean[(long long)v * g.nzg + k] = s * (1.0 / (double)((long long)g.ny * g.nx));
    }
}

extern "C" int pycles_level_means(const pycles_dims *dims, int nv, const void *const *fields, double *means,
                                  int precision, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (nv < 1 || nv > 8 || !fields || !means || (precision != PYCLES_F64 && precision != PYCLES_F32)) {
        pycles_set_error("level_means: bad arguments");
        return PYCLES_ERR_ARG;
    }
    MeanPack pk;
    for (int v = 0; v < 8; ++v) {
        pk.f[v] = v < nv ? fields[v] : nullptr;
        if (v < nv && !pk.f[v]) {
            pycles_set_error("level_means: NULL field %d", v);
            return PYCLES_ERR_ARG;
        }
    }
    Geo g = make_geo(dims);
    hipStream_t st = (hipStream_t)stream;
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(level_mean_kernel<double>, dim3(g.nzg, nv), dim3(256), 0, st, g, pk, means);
    else
        hipLaunchKernelGGL(level_mean_kernel<float>, dim3(g.nzg, nv), dim3(256), 0, st, g, pk, means);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

extern "C" int pycles_level_mean(const pycles_dims *dims, const void *field, double *mean, int precision,
                                 void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!field || !mean || (precision != PYCLES_F64 && precision != PYCLES_F32)) {
        pycles_set_error("level_mean: bad arguments");
        return PYCLES_ERR_ARG;
    }
    return pycles_level_means(dims, 1, &field, mean, precision, stream);
}

// ---------------------------------------------------------------------------
// CFL maximum.  Values are non-negative, so their IEEE bit patterns order
// like unsigned integers and an integer atomic max is exact.
__global__ void cfl_init_kernel(double *out) { *out = 0.0; }

__global__ void cfl_finish_kernel(double *out) { *out = *out + 1e-11; }

template <typename T>
__global__ __launch_bounds__(256) void cfl_kernel(Geo g, const T *u, const T *v, const T *w, double dt,
                                                  double *out) {
    const long long n = g.plane * g.nz;
    double m = 0.0;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long long)gridDim.x * blockDim.x) {
        const long long o = t + (long long)g.gw * g.plane;
        const double c = dt * (fabs((double)u[o]) * g.dxi[0] + fabs((double)v[o]) * g.dxi[1] +
                               fabs((double)w[o]) * g.dxi[2]);
        m = cfl_fold(m, c);
    }
    cfl_block_max(m, out);
}

extern "C" int pycles_cfl_max(const pycles_dims *dims, const void *u, const void *v, const void *w, double dt,
                              double *out, int precision, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!u || !v || !w || !out) {
        pycles_set_error("cfl_max: NULL argument");
        return PYCLES_ERR_ARG;
    }
    Geo g = make_geo(dims);
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(cfl_init_kernel, dim3(1), dim3(1), 0, st, out);
    const long long n = g.plane * g.nz;
    unsigned grid = (unsigned)((n + 255) / 256);
    if (grid > 4096) grid = 4096;
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(cfl_kernel<double>, dim3(grid), dim3(256), 0, st, g, (const double *)u,
                           (const double *)v, (const double *)w, dt, out);
    else if (precision == PYCLES_F32)
        hipLaunchKernelGGL(cfl_kernel<float>, dim3(grid), dim3(256), 0, st, g, (const float *)u,
                           (const float *)v, (const float *)w, dt, out);
    else {
        pycles_set_error("bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    hipLaunchKernelGGL(cfl_finish_kernel, dim3(1), dim3(1), 0, st, out);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

// ---------------------------------------------------------------------------
// Layout conversion.  Reference layout index: (i*nlg1 + j)*nlg2 + k with
// i, j, k ghosted; device (k*ny + j)*nx + i over x/y interior.  For one j both
// are matrices over (i, k), one contiguous along k, the other along i, so each
// is a transpose: a block moves a tile of 64 i by 32 k of one row j through
// LDS, reading and writing along the contiguous direction of either side, all
// of a thread's eight loads before its LDS writes.  32 k (256 bytes of the
// reference's array) rather than 64 because the ghosted columns are short and
// not a multiple of either (81 levels: 84% of a 32-wide tiling in use, 63% of
// a 64-wide one).  Tiles that share the partial cache lines of a column run
// are neighbours on one XCD (xcd_band).
// Bound: HBM.  256 x 256 x 128 FP64, one field in and out: 65 us (283 MB, 4.4
// TB/s) against 253 us (85 + 168) for one element per thread, whose reads
// (ingress) or reads of the other array (egress) along i or k were a column or
// a plane apart.
constexpr int LT_I = 64, LT_K = 32, LT_N = LT_I * LT_K / 256;

// Tile of linear index t: k tiles fastest, then i tiles, then rows j.
struct LayoutTile {
    int k0, i0;
    long long j;
};
__device__ __forceinline__ LayoutTile layout_tile(long long t, int nkt, int nit) {
    LayoutTile r;
    r.k0 = (int)(t % nkt) * LT_K;
    t /= nkt;
    r.i0 = (int)(t % nit) * LT_I;
    r.j = t / nit;
    return r;
}

template <typename T>
__global__ __launch_bounds__(256) void ingress_kernel(Geo g, const double *src, T *dst, const double *base, int nkt,
                                                      int nit, long long ntiles) {
    __shared__ T tile[LT_I][LT_K + 1];
    const long long nlg1 = g.ny + 2 * g.gw, nlg2 = g.nzg;
    const int tk = threadIdx.x % LT_K, tr = threadIdx.x / LT_K;  // read: 32 k of 8 rows i
    const int ti = threadIdx.x % LT_I, tq = threadIdx.x / LT_I;  // write: 64 i of 4 levels k
    for (long long b = blockIdx.x; b < ntiles; b += gridDim.x) {
        const LayoutTile l = layout_tile(gridDim.x == ntiles ? xcd_band(b, ntiles) : b, nkt, nit);
        const int k = l.k0 + tk;
        double v[LT_N];
        const double bk = base && k < g.nzg ? base[k] : 0.0;
#pragma unroll
        for (int q = 0; q < LT_N; ++q) {
            const int i = l.i0 + tr + q * (256 / LT_K);
            v[q] = k < g.nzg && i < g.nx ? src[((i + g.gw) * nlg1 + (l.j + g.gw)) * nlg2 + k] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < LT_N; ++q) tile[tr + q * (256 / LT_K)][tk] = (T)(base ? v[q] - bk : v[q]);
        __syncthreads();
        const int i = l.i0 + ti;
#pragma unroll
        for (int q = 0; q < LT_N; ++q) {
            const int kk = tq + q * (256 / LT_I);
            if (i < g.nx && l.k0 + kk < g.nzg)
                dst[((long long)(l.k0 + kk) * g.ny + l.j) * g.nx + i] = tile[ti][kk];
        }
        __syncthreads();  // before the next tile is written
    }
}

// Tiles over the ghosted (destination) i and j: the periodic images read the
// wrapped columns again.
template <typename T>
__global__ __launch_bounds__(256) void egress_kernel(Geo g, const T *src, double *dst, const double *base, int nkt,
                                                     int nit, long long ntiles) {
    __shared__ double tile[LT_I][LT_K + 1];
    const int nlg0 = g.nx + 2 * g.gw;
    const long long nlg1 = g.ny + 2 * g.gw, nlg2 = g.nzg;
    const int tk = threadIdx.x % LT_K, tr = threadIdx.x / LT_K;
    const int ti = threadIdx.x % LT_I, tq = threadIdx.x / LT_I;
    for (long long b = blockIdx.x; b < ntiles; b += gridDim.x) {
        const LayoutTile l = layout_tile(gridDim.x == ntiles ? xcd_band(b, ntiles) : b, nkt, nit);
        int ii = (l.i0 + ti - g.gw) % g.nx;
        if (ii < 0) ii += g.nx;
        int jj = (int)((l.j - g.gw) % g.ny);
        if (jj < 0) jj += g.ny;
        T v[LT_N];
#pragma unroll
        for (int q = 0; q < LT_N; ++q) {
            const int k = l.k0 + tq + q * (256 / LT_I);
            v[q] = k < g.nzg ? src[gidx(g, ii, jj, k)] : T(0);
        }
#pragma unroll
        for (int q = 0; q < LT_N; ++q) tile[ti][tq + q * (256 / LT_I)] = (double)v[q];
        __syncthreads();
        const int k = l.k0 + tk;
        if (k < g.nzg) {
            const double bk = base ? base[k] : 0.0;
#pragma unroll
            for (int q = 0; q < LT_N; ++q) {
                const int i = l.i0 + tr + q * (256 / LT_K);
                const double w = tile[i - l.i0][tk];
                if (i < nlg0) dst[(i * nlg1 + l.j) * nlg2 + k] = base ? w + bk : w;
            }
        }
        __syncthreads();
    }
}

// Tile counts and grid of a conversion over ni x nj columns (a block per
// tile; larger domains loop over them).
struct LayoutGrid {
    int nkt, nit;
    long long ntiles;
    unsigned blocks;
};
static LayoutGrid layout_grid(const Geo &g, int ni, long long nj) {
    LayoutGrid l;
    l.nkt = (g.nzg + LT_K - 1) / LT_K;
    l.nit = (ni + LT_I - 1) / LT_I;
    l.ntiles = (long long)l.nkt * l.nit * nj;
    l.blocks = (unsigned)(l.ntiles < (1 << 22) ? l.ntiles : (1 << 22));
    return l;
}

extern "C" int pycles_layout_ingress(const pycles_dims *dims, const double *ref_layout, void *dev,
                                     const double *base, int precision, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!ref_layout || !dev) {
        pycles_set_error("layout_ingress: NULL array");
        return PYCLES_ERR_ARG;
    }
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("layout_ingress: bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    Geo g = make_geo(dims);
    const LayoutGrid l = layout_grid(g, g.nx, g.ny);
    hipStream_t st = (hipStream_t)stream;
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(ingress_kernel<double>, dim3(l.blocks), dim3(256), 0, st, g, ref_layout, (double *)dev, base,
                           l.nkt, l.nit, l.ntiles);
    else
        hipLaunchKernelGGL(ingress_kernel<float>, dim3(l.blocks), dim3(256), 0, st, g, ref_layout, (float *)dev, base,
                           l.nkt, l.nit, l.ntiles);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

extern "C" int pycles_layout_egress(const pycles_dims *dims, const void *dev, double *ref_layout,
                                    const double *base, int precision, void *stream) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!ref_layout || !dev) {
        pycles_set_error("layout_egress: NULL array");
        return PYCLES_ERR_ARG;
    }
    if (precision != PYCLES_F64 && precision != PYCLES_F32) {
        pycles_set_error("layout_egress: bad precision %d", precision);
        return PYCLES_ERR_ARG;
    }
    Geo g = make_geo(dims);
    const LayoutGrid l = layout_grid(g, g.nx + 2 * g.gw, (long long)g.ny + 2 * g.gw);
    hipStream_t st = (hipStream_t)stream;
    if (precision == PYCLES_F64)
        hipLaunchKernelGGL(egress_kernel<double>, dim3(l.blocks), dim3(256), 0, st, g, (const double *)dev, ref_layout,
                           base, l.nkt, l.nit, l.ntiles);
    else
        hipLaunchKernelGGL(egress_kernel<float>, dim3(l.blocks), dim3(256), 0, st, g, (const float *)dev, ref_layout,
                           base, l.nkt, l.nit, l.ntiles);
    PYCLES_CHECK_LAUNCH();
    return PYCLES_OK;
}

// ---------------------------------------------------------------------------
// The CFL value on the host, after the stream's work: the time-step
// adjustment's one synchronisation per step (TimeStepping.pyx:265-266).
extern "C" int pycles_cfl_read(const double *dev_cfl, double *host_cfl, void *stream) {
    if (!dev_cfl || !host_cfl) {
        pycles_set_error("cfl_read: NULL argument");
        return PYCLES_ERR_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
    hipError_t e = hipMemcpyAsync(host_cfl, dev_cfl, sizeof(double), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
        pycles_set_error("cfl_read: %s", hipGetErrorString(e));
        return PYCLES_ERR_HIP;
    }
    const double h = *host_cfl;
    if (!(h - h == 0.0)) {  // NaN or infinite
        pycles_set_error("CFL number is not finite (%g): a velocity is NaN or infinite", *host_cfl);
        return PYCLES_ERR_NONFINITE;
    }
    return PYCLES_OK;
}

// Chunk layout of the z-chunked kernels (see the header).
extern "C" int pycles_launch_chunks(int kernel, const pycles_dims *dims, int *nchunks, int *chunk_len) {
    int rc = pycles_check_dims(dims);
    if (rc) return rc;
    if (!nchunks || !chunk_len) {
        pycles_set_error("launch_chunks: NULL argument");
        return PYCLES_ERR_ARG;
    }
    const Geo g = make_geo(dims);
    ZSplit z;
    switch (kernel) {
    case 0: z = correct_zsplit(g.plane, g.nz, g.gw); break;
    case 1: z = advy_zsplit(g.nx, g.ny, g.nz); break;
    case 2: z = advz_zsplit(g.nx, g.ny, g.nz); break;
    case 3: z = thermo_zsplit(g.nx, g.ny, g.nzg); break;
    case 4: z = advyz_zsplit(g.nx, g.ny, g.nz); break;
    default:
        pycles_set_error("launch_chunks: unknown kernel %d", kernel);
        return PYCLES_ERR_ARG;
    }
    *nchunks = z.nch;
    *chunk_len = z.len;
    return PYCLES_OK;
}
