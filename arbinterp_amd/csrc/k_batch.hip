// Many fields in one launch, and the RK4 particle push.
//
// No reference counterpart: the reference evaluates one field per Query call
// and dropped its particle integrator in v1.8 (CHANGELOG.md:8, "Created for
// simulating particle motion in magnetic fields", CHANGELOG.md:22).
//
// Batched query: one persistent grid; each workgroup pulls work items
// (field, chunk of `chunk` queries) from a queue counter until the queue is
// empty, finds the field by binary search over the per-field item offsets,
// and evaluates its chunk lane-per-query from that field's table.  Every wave
// exits once the counter passes the item count, so the grid always drains.
//
// RK4 push: each lane advances one particle (x, v) by `nsteps` classical RK4
// steps under a = -grad U; the current cell's coefficients stay in registers
// and are reloaded only when a stage lands in another cell.  Positions that
// leave the interpolation box turn NaN (as the reference's batch query does)
// and the NaN then propagates through position and velocity.
#include <type_traits>

#include "arb_internal.h"

namespace {

struct BatchField {
    ArbGeom g;
    const void* table;
    int64_t q0;          // first query row of this field
    int64_t nq;          // its number of queries
    int64_t item0;       // first work item of this field
};

template <typename TO, typename T>
__device__ __forceinline__ void put(void* p, int64_t idx, T v) {
    reinterpret_cast<TO*>(p)[idx] = (TO)v;
}

template <int D, typename T, typename TC, typename TO>
__global__ void __launch_bounds__(256)
k_batch_query(const BatchField* __restrict__ fields, int32_t nfields, int64_t nitems, int32_t chunk,
              int32_t ninterp, int32_t has_comps, int32_t has_norm, const double* __restrict__ q,
              int64_t ldq, void* comps, void* norms, void* grads, int32_t* flag,
              unsigned int* counter) {
    constexpr int K = (D == 3) ? 64 : 256;
    __shared__ long long item_s;
    for (;;) {
        if (threadIdx.x == 0) item_s = (long long)atomicAdd(counter, 1u);
        __syncthreads();
        const int64_t item = item_s;
        __syncthreads();
        if (item >= nitems) return;                 // uniform: every wave leaves
        int lo = 0, hi = nfields - 1;
        while (lo < hi) {                           // last field with item0 <= item
            const int mid = (lo + hi + 1) >> 1;
            if (fields[mid].item0 <= item) lo = mid; else hi = mid - 1;
        }
        const BatchField& F = fields[lo];
        const int64_t base = (item - F.item0) * chunk;
        for (int r = threadIdx.x; r < chunk; r += blockDim.x) {
            const int64_t j = base + r;
            if (j >= F.nq) break;
            const int64_t i = F.q0 + j;
            double loc[D];
            bool oob;
            int64_t flat = arb_reduce<D>(q + i * ldq, F.g, loc, &oob);
            if (flat > F.g.nc) { flag[0] = 1; flat = F.g.nc; }
            const TC* a = reinterpret_cast<const TC*>(F.table) + flat * (int64_t)ninterp * K;
            T x[D];
#pragma unroll
            for (int d = 0; d < D; ++d) x[d] = (T)loc[d];
            int k = 0;
            if (has_comps) {
                for (int c = 0; c < 3; ++c) {
                    T v;
                    if constexpr (D == 3) v = arb_val3<T, TC>(a + c * K, x[0], x[1], x[2]);
                    else v = arb_val4<T, TC>(a + c * K, x[0], x[1], x[2], x[3]);
                    put<TO>(comps, i * 3 + c, v);
                }
                k = 3;
            }
            if (has_norm) {
                T v, gr[D];
                if constexpr (D == 3) arb_valgrad3<T, TC>(a + k * K, x[0], x[1], x[2], v, gr);
                else arb_valgrad4<T, TC>(a + k * K, x[0], x[1], x[2], x[3], v, gr);
                put<TO>(norms, i, v);
#pragma unroll
                for (int d = 0; d < D; ++d) put<TO>(grads, i * D + d, gr[d] / (T)F.g.h[d]);
            }
        }
    }
}

__global__ void k_zero_u32(unsigned int* p) { p[0] = 0u; }

// a / h for a finite h > 0 with rh = 1 / h correctly rounded: the residual
// correction of a rh (P. Markstein, "Computation of elementary functions on
// the IBM RISC System/6000 processor", IBM J. Res. Dev. 34, 1990).  a rh is
// within 1.5 units in the last place, the residual a - q h is exact, and the
// corrected sum is within 2^-104 of a / h before its one rounding: the IEEE
// quotient unless a / h lies that close to a midpoint, as long as nothing
// under- or overflows.  Three FP64 operations, where the general division
// takes about fourteen issue slots (it scales, starts from a quarter-rate
// reciprocal and fixes up).
__device__ __forceinline__ double div_h(double a, double h, double rh) {
    const double q = a * rh;
    return fma(fma(-q, h, a), rh, q);
}

// gr / h of the gradient, keeping an infinite one as it is.
__device__ __forceinline__ double grad_h(double gr, double h, double rh) {
    const double q0 = gr * rh, q = div_h(gr, h, rh);
    return isinf(q0) ? q0 : q;
}
// FP32: the quotient of two floats is no closer than 2^-49 (relative) to the
// midpoint of two floats, so the FP64 product, good to 2^-52, rounds to the
// IEEE float quotient.
__device__ __forceinline__ float grad_h(float gr, double, double rhf) {
    return (float)((double)gr * rhf);
}

// Grid constants of the push: cell edges, their reciprocals, and (FP32) the
// reciprocals of the edges rounded to float, which the gradient is divided by.
struct PushGeom {
    double lo[3], hi[3], h[3], rh[3], rhg[3];
    int32_t np[3];
    int32_t nc;
};

// Gradient in cuboid units, the operations of arb_valgrad3 without the value.
template <typename T>
__device__ __forceinline__ void grad3(const T* c, T u, T v, T w, T* g) {
    T q[4], qu[4], qv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        T p[4], pu[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            h4d<T>(c[16 * k + 4 * j], c[16 * k + 4 * j + 1], c[16 * k + 4 * j + 2],
                   c[16 * k + 4 * j + 3], u, p[j], pu[j]);
        h4d<T>(p[0], p[1], p[2], p[3], v, q[k], qv[k]);
        qu[k] = h4<T>(pu[0], pu[1], pu[2], pu[3], v);
    }
    T val;
    h4d<T>(q[0], q[1], q[2], q[3], w, val, g[2]);
    g[0] = h4<T>(qu[0], qu[1], qu[2], qu[3], w);
    g[1] = h4<T>(qv[0], qv[1], qv[2], qv[3], w);
}

// -grad U at x (physical units), with the lane's cell cache.  The reduction
// is arb_reduce's for a grid whose cells fit 32-bit indices and whose spacing
// div_h takes.
template <typename T, typename TC>
__device__ __forceinline__ void accel3_fast(const PushGeom& g, const TC* __restrict__ table,
                                            int32_t ninterp, int32_t kn, const double* x,
                                            int32_t& cached, T* c, double* acc) {
    bool out = false;
#pragma unroll
    for (int d = 0; d < 3; ++d) out |= !(x[d] >= g.lo[d] && x[d] <= g.hi[d]);   // NaN too
    double loc[3];
    int32_t ia[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double iu = div_h(out ? 0.0 : x[d] - g.lo[d], g.h[d], g.rh[d]);
        const double fl = floor(iu);
        loc[d] = iu - fl;
        ia[d] = (int32_t)fl;
    }
    int32_t flat = ia[0] + g.np[0] * (ia[1] + g.np[1] * ia[2]);
    if (flat > g.nc) flat = g.nc;
    if (!out && flat != cached) {
        const TC* a = table + ((int64_t)flat * ninterp + kn) * 64;
#pragma unroll
        for (int i = 0; i < 64; ++i) c[i] = (T)a[i];
        cached = flat;
    }
    T gr[3];
    grad3<T>(c, (T)loc[0], (T)loc[1], (T)loc[2], gr);
#pragma unroll
    for (int d = 0; d < 3; ++d)
        acc[d] = out ? NAN : -(double)grad_h(gr[d], g.h[d], g.rhg[d]);
}

// -grad U by the general reduction and division, for the grids that
// accel3_fast does not take.
template <typename T, typename TC>
__device__ __forceinline__ void accel3(const ArbGeom& g, const TC* __restrict__ table,
                                       int32_t ninterp, int32_t kn, const double* x,
                                       int64_t& cached, T* c, double* acc) {
    double loc[3];
    bool oob;
    int64_t flat = arb_reduce<3>(x, g, loc, &oob);
    if (flat > g.nc) flat = g.nc;
    if (flat != cached) {
        const TC* a = table + (flat * ninterp + kn) * 64;
#pragma unroll
        for (int i = 0; i < 64; ++i) c[i] = (T)a[i];
        cached = flat;
    }
    T v, gr[3];
    arb_valgrad3<T, T>(c, (T)loc[0], (T)loc[1], (T)loc[2], v, gr);
#pragma unroll
    for (int d = 0; d < 3; ++d) acc[d] = -(double)(gr[d] / (T)g.h[d]);
}

// One lane per particle, the cell's 64 coefficients in its registers.  Issue
// bounds it: about 230 instructions an evaluation, 195 of them FP64 (4.7 ms
// of the time below), then the reloads, as some lane of a wave changes cell
// in most steps.  1e6 particles, 200 steps, 64 x 56 x 72 nodes: FP64 11.5 ->
// 6.1 ms, mixed 6.4 -> 3.8 ms against the general reduction and a value with
// every gradient (the same bits where div_h gives the IEEE quotient, see
// there); FP64 holds two waves per SIMD, mixed three
// (at four it spills: 8.1 ms).
template <typename T, typename TC, bool FAST>
__global__ void __launch_bounds__(256)
k_rk4(ArbGeom g, PushGeom pg, const TC* __restrict__ table, int32_t ninterp, int32_t kn,
      double* __restrict__ X, double* __restrict__ V, int64_t n, double dt, int32_t nsteps) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    double x[3], v[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) { x[d] = X[p * 3 + d]; v[d] = V[p * 3 + d]; }
    std::conditional_t<FAST, int32_t, int64_t> cached = -1;
    T c[64];
    const double h2 = 0.5 * dt, h6 = dt / 6.0;
    for (int s = 0; s < nsteps; ++s) {
        // the four stages in one loop body (one copy of the evaluation: 4
        // copies take more than 256 registers, one wave per SIMD): at the
        // stage's position xs and velocity vs, sx and sa the sums v1 + 2 v2 + 2
        // v3 + v4 and a1 + 2 a2 + 2 a3 + a4 so far
        double xs[3], vs[3], sx[3], sa[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) { xs[d] = x[d]; vs[d] = v[d]; sx[d] = 0.0; sa[d] = 0.0; }
#pragma unroll 1
        for (int st = 0; st < 4; ++st) {
            double acc[3];
            if constexpr (FAST) accel3_fast<T, TC>(pg, table, ninterp, kn, xs, cached, c, acc);
            else accel3<T, TC>(g, table, ninterp, kn, xs, cached, c, acc);
            const double w = st == 1 || st == 2 ? 2.0 : 1.0, hs = st == 2 ? dt : h2;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                sx[d] = fma(w, vs[d], sx[d]);           // w is 1 or 2: exact products
                sa[d] = fma(w, acc[d], sa[d]);
                xs[d] = x[d] + hs * vs[d];
                vs[d] = v[d] + hs * acc[d];
            }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            x[d] += h6 * sx[d];
            v[d] += h6 * sa[d];
        }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) { X[p * 3 + d] = x[d]; V[p * 3 + d] = v[d]; }
}

inline unsigned grid1(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

size_t arb_batch_field_desc_size() { return sizeof(BatchField); }

void arb_batch_fill_desc(void* dst, const ArbGeom& g, const void* table, int64_t q0, int64_t nq,
                         int64_t item0) {
    BatchField* b = static_cast<BatchField*>(dst);
    b->g = g;
    b->table = table;
    b->q0 = q0;
    b->nq = nq;
    b->item0 = item0;
}

hipError_t arb_launch_batch_query(int32_t ndim, int32_t prec, int32_t out_f64, const void* fields,
                                  int32_t nfields, int64_t nitems, int32_t chunk, int32_t threads,
                                  int32_t nblocks, int32_t ninterp, int32_t has_comps,
                                  int32_t has_norm, const double* q, int64_t ldq, void* comps,
                                  void* norms, void* grads, int32_t* flag, unsigned int* counter,
                                  hipStream_t s) {
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(1), 0, s, counter);
    const BatchField* F = static_cast<const BatchField*>(fields);
    dim3 grid(nblocks), block(threads);
#define L_BATCH(DD, T, TC, TO)                                                                 \
    hipLaunchKernelGGL((k_batch_query<DD, T, TC, TO>), grid, block, 0, s, F, nfields, nitems,     \
                       chunk, ninterp, has_comps, has_norm, q, ldq, comps, norms, grads, flag,  \
                       counter)
    if (ndim == 3) {
        if (prec == ARB_PREC_FP64) L_BATCH(3, double, double, double);
        else if (out_f64) L_BATCH(3, float, float, double);
        else L_BATCH(3, float, float, float);
    } else {
        if (prec == ARB_PREC_FP64) L_BATCH(4, double, double, double);
        else if (out_f64) L_BATCH(4, float, float, double);
        else L_BATCH(4, float, float, float);
    }
#undef L_BATCH
    return hipGetLastError();
}

hipError_t arb_launch_rk4(const ArbGeom& g, int32_t prec, const void* table, int32_t ninterp,
                          int32_t kn, double* X, double* V, int64_t n, double dt, int32_t nsteps,
                          hipStream_t s) {
    if (n <= 0 || nsteps <= 0) return hipSuccess;
    dim3 grid(grid1(n, 256)), block(256);
    // accel3_fast: flat cell indices in 32 bits, and magnitudes that keep
    // div_h's residuals away from under- and overflow.  A position's index
    // along an axis is at most (hi - lo) / h there (one for rounding): npos on
    // an even axis, any number on one whose first spacing is its smallest
    PushGeom pg{};
    bool fast = true;
    double top = 0.0, cells = 1.0;
    for (int d = 0; d < 3; ++d) {
        pg.lo[d] = g.lo[d];
        pg.hi[d] = g.hi[d];
        pg.h[d] = g.h[d];
        pg.rh[d] = 1.0 / g.h[d];
        pg.rhg[d] = prec == ARB_PREC_FP64 ? pg.rh[d] : 1.0 / (double)(float)g.h[d];
        pg.np[d] = (int32_t)g.npos[d];
        top += ((g.hi[d] - g.lo[d]) / g.h[d] + 1.0) * cells;
        cells *= (double)g.npos[d];
        const double e = 0x1p300;
        fast &= g.h[d] > 1.0 / e && g.h[d] < e && fabs(g.lo[d]) < e && fabs(g.hi[d]) < e;
        if (prec != ARB_PREC_FP64) fast &= g.h[d] > 0x1p-100 && g.h[d] < 0x1p100;
    }
    fast &= top < 2147483647.0 && cells < 2147483647.0;
    pg.nc = (int32_t)g.nc;
#define L_RK4(T, F)                                                                             \
    hipLaunchKernelGGL((k_rk4<T, T, F>), grid, block, 0, s, g, pg, (const T*)table, ninterp, kn, \
                       X, V, n, dt, nsteps)
    if (prec == ARB_PREC_FP64) {
        if (fast) L_RK4(double, true);
        else L_RK4(double, false);
    } else {
        if (fast) L_RK4(float, true);
        else L_RK4(float, false);
    }
#undef L_RK4
    return hipGetLastError();
}
