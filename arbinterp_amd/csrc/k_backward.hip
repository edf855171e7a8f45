// Backward pass of the scalar interpolant (value + gradient outputs).
//
// No reference counterpart: the reference has no derivatives with respect to
// its inputs.  For upstream gradients gv (of U) and gg (of grad U):
//   d/dq   = gv grad U + Hess U . gg                  (per query, analytic)
//   d/df_n = sum_i sum_j c_ij A_{j, l(n, cell_i)}    (U is linear in f)
//            c_i = gv_i m(x_i) + sum_k gg_ik dm_k(x_i)/h_k
// The node adjoint is deterministic: queries are grouped per cell in
// query-index order (a stable radix sort of the cell keys, k_sort.hip), and
// every per-cell sum runs in that order over per-query records, written by
// row (3D table path) or at the queries' grouped positions (node tiles and
// 4D: a cell's records consecutive).  3D: blocks of 4^3 cells apply the
// transpose of the separable coefficient passes to their alpha_bar, giving
// partial gradients on the block's 7^3 node tile, and every node sums the
// tiles holding it in a fixed block order.  4D does the same with blocks of
// 4 x 4 x 2 cells in (x, y, z) that run through all of t (k_bwd_block4), the
// operator's row shift included.  No floating-point atomics.
#include "arb_internal.h"

namespace {

// t[e] for a runtime e in 0..3 by selects (a dynamic index into a register
// array would place the array in scratch memory)
__device__ __forceinline__ double sel4(const double* t, int e) {
    return e == 0 ? t[0] : e == 1 ? t[1] : e == 2 ? t[2] : t[3];
}

// p(u), p'(u) and p''(u)/2 of c0 + c1 u + c2 u^2 + c3 u^3 (synthetic division).
__device__ __forceinline__ void h4dd(double c0, double c1, double c2, double c3, double u,
                                     double& p, double& d, double& hh) {
    p = c3;
    d = 0.0;
    hh = 0.0;
    hh = fma(hh, u, d); d = fma(d, u, p); p = fma(p, u, c2);
    hh = fma(hh, u, d); d = fma(d, u, p); p = fma(p, u, c1);
    hh = fma(hh, u, d); d = fma(d, u, p); p = fma(p, u, c0);
}

// Value, gradient and Hessian (cuboid units) of sum_i a_i u^ex v^ey w^ez by
// tensor Horner: rows along u (p, p', p''), then v, then w, keeping the
// derivative combinations of total order <= 2.
template <typename TC>
__device__ __forceinline__ void hess3(const TC* __restrict__ a, double u, double v, double w,
                                      double& val, double* g, double (*H)[3]) {
    double Q[4], Qv[4], Qvv[4], R[4], Rv[4], S[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        double P[4], Pu[4], Puu[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const TC* c = a + 16 * k + 4 * j;
            double hh;
            h4dd((double)c[0], (double)c[1], (double)c[2], (double)c[3], u, P[j], Pu[j], hh);
            Puu[j] = 2.0 * hh;
        }
        double hq;
        h4dd(P[0], P[1], P[2], P[3], v, Q[k], Qv[k], hq);
        Qvv[k] = 2.0 * hq;
        h4d<double>(Pu[0], Pu[1], Pu[2], Pu[3], v, R[k], Rv[k]);
        S[k] = h4<double>(Puu[0], Puu[1], Puu[2], Puu[3], v);
    }
    double hw;
    h4dd(Q[0], Q[1], Q[2], Q[3], w, val, g[2], hw);
    H[2][2] = 2.0 * hw;
    h4d<double>(R[0], R[1], R[2], R[3], w, g[0], H[0][2]);
    h4d<double>(Qv[0], Qv[1], Qv[2], Qv[3], w, g[1], H[1][2]);
    H[0][0] = h4<double>(S[0], S[1], S[2], S[3], w);
    H[1][1] = h4<double>(Qvv[0], Qvv[1], Qvv[2], Qvv[3], w);
    H[0][1] = h4<double>(Rv[0], Rv[1], Rv[2], Rv[3], w);
    H[1][0] = H[0][1];
    H[2][0] = H[0][2];
    H[2][1] = H[1][2];
}

// 4D: the 3D quantities of the four t-slices, combined along t.
template <typename TC>
__device__ __forceinline__ void hess4(const TC* __restrict__ a, double u, double v, double w,
                                      double t, double& val, double* g, double (*H)[4]) {
    double r[4], gs[3][4], hs[3][3][4];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        double gl[3], Hl[3][3];
        hess3<TC>(a + 64 * l, u, v, w, r[l], gl, Hl);
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            gs[x][l] = gl[x];
#pragma unroll
            for (int y = 0; y < 3; ++y) hs[x][y][l] = Hl[x][y];
        }
    }
    double ht;
    h4dd(r[0], r[1], r[2], r[3], t, val, g[3], ht);
    H[3][3] = 2.0 * ht;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        h4d<double>(gs[x][0], gs[x][1], gs[x][2], gs[x][3], t, g[x], H[x][3]);
        H[3][x] = H[x][3];
#pragma unroll
        for (int y = 0; y < 3; ++y)
            H[x][y] = h4<double>(hs[x][y][0], hs[x][y][1], hs[x][y][2], hs[x][y][3], t);
    }
}

// Cell key of each query for the node adjoint's grouping: its flat cell, or
// nc for rows outside the box (the group after the cells).
template <int D>
__global__ void __launch_bounds__(256)
k_bwd_keys(ArbGeom g, const double* __restrict__ q, int64_t n, int64_t ldq,
           int32_t* __restrict__ key) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double loc[D];
    bool oob;
    const int64_t flat = arb_reduce<D>(q + i * ldq, g, loc, &oob);
    key[i] = flat < g.nc ? (int32_t)flat : (int32_t)g.nc;
}

// Doubles of a 4D record: u, v, w, t, gv, gg / h (4), one of padding (16-byte
// loads).
constexpr int REC4 = 10;

// d/dq per query, and, for the node adjoint, the query's cell key and its
// record (3D: at row i; 4D: at the grouped position s).  Without perm,
// thread i takes query i: 3D reads a cell's 64 table coefficients as one
// contiguous 512-byte run, so query order costs nothing and the queries' own
// arrays are read and written in order.  With perm (the queries grouped by
// cell; 4D, whose 256 coefficients of a cell are 2 KB), thread s takes query
// perm[s], so neighbouring threads read the same cell's coefficients.
template <int D, typename TC>
__global__ void __launch_bounds__(256)
k_bwd_points(ArbGeom g, const TC* __restrict__ table, int32_t ninterp, int32_t kn,
             const double* __restrict__ q, int64_t n, int64_t ldq, const double* __restrict__ gv,
             const double* __restrict__ gg, double* __restrict__ dq,
             const int32_t* __restrict__ perm, int32_t* __restrict__ key,
             double* __restrict__ rec) {
    constexpr int K = 1 << (2 * D);
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int64_t i = perm ? (int64_t)perm[s] : s;
    if (i < 0 || i >= n) return;                    // unreachable: perm holds row indices
    double loc[D];
    bool oob;
    int64_t flat = arb_reduce<D>(q + i * ldq, g, loc, &oob);
    const bool ok = flat < g.nc;
    if (key) key[i] = ok ? (int32_t)flat : (int32_t)g.nc;  // rows outside: after the cells
    if (rec && ok) {
        // the node adjoint's per-query record: local coordinates, gv, gg / h
        if constexpr (D == 3) {
            double4* r4 = reinterpret_cast<double4*>(rec + i * 8);
            r4[0] = make_double4(loc[0], loc[1], loc[2], gv[i]);
            r4[1] = make_double4(gg[i * 3] / g.h[0], gg[i * 3 + 1] / g.h[1], gg[i * 3 + 2] / g.h[2], 0.0);
        } else {
            double2* r2 = reinterpret_cast<double2*>(rec + s * REC4);
            r2[0] = make_double2(loc[0], loc[1]);
            r2[1] = make_double2(loc[2], loc[3]);
            r2[2] = make_double2(gv[i], gg[i * 4] / g.h[0]);
            r2[3] = make_double2(gg[i * 4 + 1] / g.h[1], gg[i * 4 + 2] / g.h[2]);
            r2[4] = make_double2(gg[i * 4 + 3] / g.h[3], 0.0);
        }
    }
    if (!dq) return;
    if (!ok) {
#pragma unroll
        for (int x = 0; x < D; ++x) dq[i * D + x] = NAN;
        return;
    }
    double val, gr[D], H[D][D];
    const TC* a = table + (flat * ninterp + kn) * K;
    if constexpr (D == 3) hess3<TC>(a, loc[0], loc[1], loc[2], val, gr, H);
    else hess4<TC>(a, loc[0], loc[1], loc[2], loc[3], val, gr, H);
    const double v = gv[i];
#pragma unroll
    for (int x = 0; x < D; ++x) {
        double acc = v * (gr[x] / g.h[x]);
#pragma unroll
        for (int y = 0; y < D; ++y) acc += (H[x][y] / (g.h[x] * g.h[y])) * gg[i * D + y];
        dq[i * D + x] = acc;
    }
}

// 3D: a workgroup takes a block of BB^3 cells.  Four threads per cell form
// alpha_bar into LDS from the queries' records (u, v, w, gv,
// gg / h): thread g of a cell sums, over the cell's queries in index order,
// the entries ex + 4 ey + 16 ez with ex + 4 ey in 4g..4g+3,
//   gv u^ex v^ey w^ez + gk_u (u^ex)' v^ey w^ez + gk_v u^ex (v^ey)' w^ez
//                     + gk_w u^ex v^ey (w^ez)'      (gk = gg / h).
// A = M (x) M (x) M (z slowest; M the 4x4 map of arb_sep3.h), so the node
// adjoint of the block, A^T alpha_bar spread over the cells' neighbourhoods,
// is the transpose of the separable passes: z, then y, then x, each a gather
//   out(n) = sum over (c, o) with c + o = n of  sum_e M[e][o] in(c, e)
// over the cells c of the block and offsets o = 0..3.  The result is the
// block's node tile, (BB+3)^3 partial node gradients, written to
// tiles[block][node].  Every sum runs in a fixed order (no atomics).
__device__ __forceinline__ void pow3(double x, double* p, double* dp) {
    p[0] = 1.0; p[1] = x; p[2] = x * x; p[3] = p[2] * x;
    dp[0] = 0.0; dp[1] = 1.0; dp[2] = 2.0 * x; dp[3] = 3.0 * p[2];
}

// sum_e M[e][o] a_e (column o of M applied to a; M as in arb_sep3.h)
__device__ __forceinline__ double mcol(int o, double a0, double a1, double a2, double a3) {
    switch (o) {
        case 0: return fma(-0.5, a3, fma(-0.5, a1, a2));
        case 1: return fma(1.5, a3, fma(-2.5, a2, a0));
        case 2: return fma(-1.5, a3, fma(0.5, a1, 2.0 * a2));
        default: return 0.5 * (a3 - a2);
    }
}

constexpr int BB = 4;                              // block edge (cells)
constexpr int BN = BB + 3;                         // node tile edge
constexpr int BCELLS = BB * BB * BB;
constexpr int BTILE = BN * BN * BN;

// A cell holding more than C queries is summed in pieces: the
// queries at sorted positions [o C, (o + 1) C) of such a cell (C =
// BWD_CHUNK_OF, o C inside the cell) are summed by a chunk kernel into
// part[o], in index order, and the cell's own sum takes the queries before
// its first multiple of C in index order, then part[o] for each of its
// chunks in order: a fixed order, so the result still repeats bit for bit,
// and a cell of many queries (particles clustered in a few cells) is
// spread over many threads instead of four.
//
// A thread group adds a cell's queries one after another, about 2 us each (the
// chain perm -> record), and the partial sums about 1 us each, so the chunk
// balances the two; 1024 in both dimensions left clouds of particles waiting
// for a few cells.  Forward + backward of 1e6 queries in a cloud (ms, chunk
// 1024 / now): 3D mixed 25^3 nodes 3.9 / 1.4, 50^3 4.0 / 1.5, 96^3 0.87 / 0.88
// (with chunks of 128: 1.0, 1.0 and 1.14, its cells of some 150 queries then
// taking two kernels); 4D FP64 22 x 24 x 22 x 10 nodes 5.0 / 1.2.
template <int D>
constexpr int32_t BWD_CHUNK_OF = D == 3 ? 256 : 128;

// The chunk starting at sorted position o C, if it belongs to a cell of
// more than BWD_CHUNK_OF queries: [s0, s1) and that cell; q, ldq: the query
// positions (the cell of the query at o C, by the same reduction as the
// keys).
template <int D>
__device__ __forceinline__ bool bwd_chunk(const ArbGeom& g, const double* __restrict__ q,
                                          int64_t ldq, const int32_t* __restrict__ offs,
                                          const int32_t* __restrict__ perm, int64_t o,
                                          int32_t* s0, int32_t* s1) {
    const int64_t p0 = o * BWD_CHUNK_OF<D>;
    if (p0 >= offs[g.nc]) return false;              // the rows outside the box follow
    const int64_t i = perm[p0];
    double loc[D];
    bool oob;
    const int64_t c = arb_reduce<D>(q + i * ldq, g, loc, &oob);
    if (c < 0 || c >= g.nc) return false;            // cannot happen: p0 is a cell's row
    const int32_t e = offs[c + 1];
    if (e - offs[c] <= BWD_CHUNK_OF<D>) return false;      // summed whole by the cell kernel
    *s0 = (int32_t)p0;
    *s1 = p0 + BWD_CHUNK_OF<D> < e ? (int32_t)(p0 + BWD_CHUNK_OF<D>) : e;
    return true;
}

// 3D: thread gq (of four) of a cell: its 16 entries of alpha_bar, summed over
// the queries at sorted positions [s0, s1) in order, into acc[p][ez]
// (entries 4 gq + p + 16 ez).
__device__ __forceinline__ void abar_row3(const double4& r0, const double4& r1, int gq,
                                          double (*acc)[4]);

template <int NB>
__device__ __forceinline__ void abar_rows3(const double* __restrict__ rec,
                                           const int32_t* __restrict__ rperm, int32_t s0,
                                           int32_t s1, int gq, double (*acc)[4]) {
    // the record of sorted position s: rec[s] (written at the grouped
    // positions: a cell's records are consecutive) or rec[rperm[s]] (written
    // by row); NB (1 or 2) loaded together, then added in query order
    int32_t s = s0;
    if constexpr (NB == 2) {
        for (; s + 2 <= s1; s += 2) {
            const int64_t ra = rperm ? (int64_t)rperm[s] : s;
            const int64_t rb = rperm ? (int64_t)rperm[s + 1] : s + 1;
            const double4* r4a = reinterpret_cast<const double4*>(rec + ra * 8);
            const double4* r4b = reinterpret_cast<const double4*>(rec + rb * 8);
            const double4 a0 = r4a[0], a1 = r4a[1], b0 = r4b[0], b1 = r4b[1];
            abar_row3(a0, a1, gq, acc);
            abar_row3(b0, b1, gq, acc);
        }
    }
    for (; s < s1; ++s) {
        const int64_t ra = rperm ? (int64_t)rperm[s] : s;
        const double4* r4 = reinterpret_cast<const double4*>(rec + ra * 8);
        abar_row3(r4[0], r4[1], gq, acc);
    }
}

// One query's contribution (record r0 = u, v, w, gv; r1 = gg / h) to the 16
// entries of thread gq.
__device__ __forceinline__ void abar_row3(const double4& r0, const double4& r1, int gq,
                                          double (*acc)[4]) {
    {
        double pu[4], du[4], pv[4], dv[4], pw[4], dw[4];
        pow3(r0.x, pu, du);
        pow3(r0.y, pv, dv);
        pow3(r0.z, pw, dw);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int exy = 4 * gq + p, ex = exy & 3, ey = exy >> 2;
            const double a = sel4(pu, ex) * sel4(pv, ey);
            const double au = sel4(du, ex) * sel4(pv, ey);
            const double av = sel4(pu, ex) * sel4(dv, ey);
            const double base = fma(r1.y, av, fma(r1.x, au, r0.w * a));
            const double gwa = r1.z * a;
#pragma unroll
            for (int ez = 0; ez < 4; ++ez) acc[p][ez] += fma(gwa, dw[ez], base * pw[ez]);
        }
    }
}

// 3D chunk sums: four threads per chunk, part[o][entry] (64 entries).
__global__ void __launch_bounds__(256)
k_bwd_chunk3(ArbGeom g, const double* __restrict__ q, int64_t ldq, const double* __restrict__ rec,
             const int32_t* __restrict__ offs, const int32_t* __restrict__ perm,
             const int32_t* __restrict__ rperm, int64_t nchunk, double* __restrict__ part) {
    const int64_t o = (int64_t)blockIdx.x * 64 + (threadIdx.x >> 2);
    const int gq = threadIdx.x & 3;
    int32_t s0, s1;
    if (o >= nchunk || !bwd_chunk<3>(g, q, ldq, offs, perm, o, &s0, &s1)) return;
    double acc[4][4];
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int ez = 0; ez < 4; ++ez) acc[p][ez] = 0.0;
    abar_rows3<2>(rec, rperm, s0, s1, gq, acc);
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int ez = 0; ez < 4; ++ez) part[o * 64 + 4 * gq + p + 16 * ez] = acc[p][ez];
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5)))
k_bwd_block3(ArbGeom g, const double* __restrict__ rec, const int32_t* __restrict__ offs,
             const int32_t* __restrict__ rperm, int64_t nbx, int64_t nby,
             const double* __restrict__ part, double* __restrict__ tiles) {
    // the z pass's output, then the y pass's (20.6 KB in all)
    __shared__ double t2[BN][BB][BB][16];           // [z][cy][cx][ex + 4 ey]
    __shared__ double t1[BN][BN][BB][4];            // [z][y][cx][ex]
    for (int t = threadIdx.x; t < BN * BB * BB * 16; t += 256) (&t2[0][0][0][0])[t] = 0.0;
    const int64_t blk = blockIdx.x;
    const int64_t bx = blk % nbx, by = (blk / nbx) % nby, bz = blk / (nbx * nby);
    {
        const int cl = threadIdx.x >> 2, gq = threadIdx.x & 3;
        const int cx = cl & 3, cy = (cl >> 2) & 3, cz = cl >> 4;
        const int64_t x = bx * BB + cx, y = by * BB + cy, z = bz * BB + cz;
        double acc[4][4];                          // [pair][ez]: alpha_bar[4 gq + p + 16 ez]
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int ez = 0; ez < 4; ++ez) acc[p][ez] = 0.0;
        if (x < g.npos[0] && y < g.npos[1] && z < g.npos[2]) {
            const int64_t c = x + g.npos[0] * (y + g.npos[1] * z);
            const int32_t s0 = offs[c], s1 = offs[c + 1];
            if (s1 - s0 <= BWD_CHUNK_OF<3>) {
                abar_rows3<1>(rec, rperm, s0, s1, gq, acc);
            } else {
                // the queries before the cell's first chunk, then its chunks
                const int64_t ofirst = ((int64_t)s0 + BWD_CHUNK_OF<3> - 1) / BWD_CHUNK_OF<3>;
                const int32_t h1 = ofirst * BWD_CHUNK_OF<3> < s1 ? (int32_t)(ofirst * BWD_CHUNK_OF<3>) : s1;
                abar_rows3<1>(rec, rperm, s0, h1, gq, acc);
                // then the chunks' sums, in chunk order
                for (int64_t o = ofirst; o * BWD_CHUNK_OF<3> < s1; ++o) {
#pragma unroll
                    for (int p = 0; p < 4; ++p)
#pragma unroll
                        for (int ez = 0; ez < 4; ++ez)
                            acc[p][ez] += part[o * 64 + 4 * gq + p + 16 * ez];
                }
            }
        }
        // z: t2[z][cy][cx][exy] = sum_{cz + oz = z} sum_ez M[ez][oz] alpha_bar[cell][exy + 16 ez],
        // from the registers: one wave (one cz) at a time, cz descending, so
        // every entry adds its terms in ascending oz from 0.0
        __syncthreads();                           // t2 cleared
        for (int ph = BB - 1; ph >= 0; --ph) {
            if (cz == ph) {
#pragma unroll
                for (int p = 0; p < 4; ++p)
#pragma unroll
                    for (int oz = 0; oz < 4; ++oz)
                        t2[cz + oz][cy][cx][4 * gq + p] +=
                            mcol(oz, acc[p][0], acc[p][1], acc[p][2], acc[p][3]);
            }
            __syncthreads();
        }
    }
    // y: t1[z][y][cx][ex] = sum_{cy + oy = y} sum_ey M[ey][oy] t2[z][cy][cx][ex + 4 ey]
    for (int t = threadIdx.x; t < BN * BN * BB * 4; t += 256) {
        const int ex = t & 3, cx = (t >> 2) & 3, r = t >> 4, y = r % BN, z = r / BN;
        double sum = 0.0;
#pragma unroll
        for (int oy = 0; oy < 4; ++oy) {
            const int cy = y - oy;
            if (cy >= 0 && cy < BB) {
                const double* a = &t2[z][cy][cx][ex];
                sum += mcol(oy, a[0], a[4], a[8], a[12]);
            }
        }
        t1[z][y][cx][ex] = sum;
    }
    __syncthreads();
    // x: tile[z][y][x] = sum_{cx + ox = x} sum_ex M[ex][ox] t1[z][y][cx][ex]
    double* out = tiles + blk * BTILE;
    for (int t = threadIdx.x; t < BTILE; t += 256) {
        const int x = t % BN, r = t / BN, y = r % BN, z = r / BN;
        double sum = 0.0;
#pragma unroll
        for (int ox = 0; ox < 4; ++ox) {
            const int cx = x - ox;
            if (cx >= 0 && cx < BB) {
                const double* a = &t1[z][y][cx][0];
                sum += mcol(ox, a[0], a[1], a[2], a[3]);
            }
        }
        out[t] = sum;
    }
}

// Node gradient: the sum, over the blocks whose tile holds the node (at most
// two per axis), of the tile entries, blocks in ascending z, y, x order.
__global__ void __launch_bounds__(256)
k_bwd_nodes3(ArbGeom g, const double* __restrict__ tiles, int64_t nbx, int64_t nby, int64_t nbz,
             double* __restrict__ dval) {
    const int64_t nidx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (nidx >= g.nnodes) return;
    const int64_t i = nidx % g.n[0], j = (nidx / g.n[0]) % g.n[1], k = nidx / (g.n[0] * g.n[1]);
    // block b's tile holds nodes BB*b .. BB*b + BN - 1
    auto lo = [](int64_t v) { const int64_t b = v - (BN - 1); return b <= 0 ? (int64_t)0 : (b + BB - 1) / BB; };
    const int64_t x0 = lo(i), x1 = min(i / BB, nbx - 1);
    const int64_t y0 = lo(j), y1 = min(j / BB, nby - 1);
    const int64_t z0 = lo(k), z1 = min(k / BB, nbz - 1);
    double sum = 0.0;
    for (int64_t bz = z0; bz <= z1; ++bz)
        for (int64_t by = y0; by <= y1; ++by)
            for (int64_t bx = x0; bx <= x1; ++bx) {
                const int64_t blk = bx + nbx * (by + nby * bz);
                const int64_t t = (i - BB * bx) + BN * ((j - BB * by) + BN * (k - BB * bz));
                sum += tiles[blk * BTILE + t];
            }
    dval[nidx] = sum;
}

// 4D node adjoint.  alpha = (M (x) M (x) M (x) M) F + P c with alpha_85 = 0
// (arb_sep4.h): c_k = G(k-1) - G(k), G the xyzt central difference at the
// cell's corner nodes.  Its transpose, per cell:
//   alpha_bar_85 = 0;  c_bar = P^T alpha_bar;  G_bar(j) = c_bar_{j+1} - c_bar_j;
//   F_bar = (M (x) M (x) M (x) M)^T alpha_bar + the transposed differences of G_bar.
// The central difference at an end of the cell is the derivative of the
// cell's cubic there, a_1 at u = 0 and a_1 + 2 a_2 + 3 a_3 at u = 1, so the
// last term is (M (x) ..)^T of X (x) X (x) X (x) X G_bar with X = [[0,0], [1,1],
// [0,2], [0,3]] (power x end), and one transposed separable pass serves both.
//
// A workgroup takes a block of 4 x 4 x 2 cells in (x, y, z) and runs through
// all of t.  Eight threads per cell: thread gq holds, for the (ex, ey) pairs
// 2 gq and 2 gq + 1, the four ez and the four t planes that the cell touches,
//   ring[ot][pair][ez] = sum over queries of Q(ex, ey, ez) w_ot(t) + E w'_ot(t),
// w_ot the node weights along t (M applied to the powers of t, so the t pass
// is done query by query), Q = gv m + gk_u m_u + gk_v m_v + gk_w m_w and E = gk_t m
// for the monomial m = u^ex v^ey w^ez; and c_bar of the corners gq and gq + 8,
// from the Hermite end weights h_0 = t - 2t^2 + t^3, h_1 = t^3 - t^2 (the columns of
// P).  After cell layer ct, plane ct is complete: it goes through the
// transposed z, y and x passes to the block's 7 x 7 x 5 nodes of that plane,
// tiles[block][plane][node], and the ring moves on by one.  So a cell costs
// about 160 FP64 operations per query and thread, the passes run once per
// node plane instead of once per cell layer and power of t, and 9 doubles
// per cell go to memory.  On 48^3 x 16 nodes, 2e6 queries: 0.61 ms; A^T
// alpha_bar per cell (65536 products a cell, 256 doubles of it written and
// gathered) took 7.5 ms.  The node sums: 0.03 beside 0.62 ms.  It is bound by
// FP64 issue and the latency of offs -> record at two waves per SIMD (250
// VGPRs); sixteen threads per cell and 4 x 4 x 1 cells run four waves, but
// repeat more of each query's work: 0.69 ms.
constexpr int B4X = 4, B4Y = 4, B4Z = 2;
constexpr int N4X = B4X + 3, N4Y = B4Y + 3, N4Z = B4Z + 3;
constexpr int TILE4 = N4X * N4Y * N4Z;
// a thread's sums over a cell's queries: ring, c_bar (2), alpha_bar_85
constexpr int SUMS4 = 35;

struct Sums4 {
    double ring[4][2][4];
    double cb[2];
    double a85;
};

__device__ __forceinline__ void sums4_zero(Sums4& S) {
#pragma unroll
    for (int o = 0; o < 4; ++o)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) S.ring[o][p][e] = 0.0;
    S.cb[0] = S.cb[1] = S.a85 = 0.0;
}

struct Rec4 {
    double2 r[5];
};

__device__ __forceinline__ Rec4 load_rec4(const double* __restrict__ rec, int64_t s) {
    Rec4 x;
    const double2* r2 = reinterpret_cast<const double2*>(rec + s * REC4);
#pragma unroll
    for (int k = 0; k < 5; ++k) x.r[k] = r2[k];
    return x;
}

// Hermite end weight of end m and its derivative: x (c1 + c2 x + x^2) with
// (c1, c2) = (1, -2) or (0, -1)
__device__ __forceinline__ void hend(double x, int m, double& h, double& dh) {
    const double c1 = m ? 0.0 : 1.0, c2 = m ? -1.0 : -2.0;
    h = x * fma(x, x + c2, c1);
    dh = fma(x, fma(3.0, x, 2.0 * c2), c1);
}

// One query's contribution to the sums of thread gq of its cell.
__device__ __forceinline__ void sums4_row(const Rec4& x, int gq, Sums4& S) {
    const double u = x.r[0].x, v = x.r[0].y, w = x.r[1].x, t = x.r[1].y;
    const double gv = x.r[2].x, ku = x.r[2].y, kv = x.r[3].x, kw = x.r[3].y, kt = x.r[4].x;
    double wt[4], dwt[4];
    {
        const double t2 = t * t, t3 = t2 * t;
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            wt[o] = mcol(o, 1.0, t, t2, t3);
            dwt[o] = mcol(o, 0.0, 1.0, 2.0 * t, 3.0 * t2);
        }
    }
    const int exh = gq & 1, ey = gq >> 1;          // ex = 2 exh + p
    const double u2 = u * u, v2 = v * v, w2 = w * w;
    const double pv = ey == 0 ? 1.0 : ey == 1 ? v : ey == 2 ? v2 : v2 * v;
    const double dv = ey == 0 ? 0.0 : ey == 1 ? 1.0 : ey == 2 ? 2.0 * v : 3.0 * v2;
    const double pw[4] = {1.0, w, w2, w2 * w}, dw[4] = {0.0, 1.0, 2.0 * w, 3.0 * w2};
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const double pu = exh ? (p ? u2 * u : u2) : (p ? u : 1.0);
        const double du = exh ? (p ? 3.0 * u2 : 2.0 * u) : (p ? 1.0 : 0.0);
        const double a = pu * pv;
        const double base = fma(kv, pu * dv, fma(ku, du * pv, gv * a));
        const double wa = kw * a, ta = kt * a;
#pragma unroll
        for (int ez = 0; ez < 4; ++ez) {
            const double Q = fma(wa, dw[ez], base * pw[ez]), E = ta * pw[ez];
#pragma unroll
            for (int o = 0; o < 4; ++o)
                S.ring[o][p][ez] = fma(E, dwt[o], fma(Q, wt[o], S.ring[o][p][ez]));
        }
    }
    // c_bar of the corners gq (t end 0) and gq + 8 (t end 1)
    double hx, dx, hy, dy, hz, dz;
    hend(u, gq & 1, hx, dx);
    hend(v, (gq >> 1) & 1, hy, dy);
    hend(w, gq >> 2, hz, dz);
    const double hxy = hx * hy, m = hxy * hz;
    const double Qc = fma(kw, hxy * dz, fma(kv, hx * dy * hz, fma(ku, dx * hy * hz, gv * m)));
    const double Ec = kt * m;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        double ht, dt;
        hend(t, e, ht, dt);
        S.cb[e] = fma(Ec, dt, fma(Qc, ht, S.cb[e]));
    }
    // alpha_bar_85: the monomial u v w t
    const double uv = u * v, q85 = fma(kw, uv, fma(kv, u * w, fma(ku, v * w, gv * (uv * w))));
    S.a85 = fma(kt, uv * w, fma(q85, t, S.a85));
}

// The queries at sorted positions [s0, s1), in order.
__device__ __forceinline__ void sums4_rows(const double* __restrict__ rec, int32_t s0, int32_t s1,
                                           int gq, Sums4& S) {
    for (int32_t s = s0; s < s1; ++s) sums4_row(load_rec4(rec, s), gq, S);
}

// Chunk sums (cells of more than BWD_CHUNK_OF queries): eight threads per
// chunk, part[o][sum][gq].
__global__ void __launch_bounds__(256)
k_bwd_chunk4(ArbGeom g, const double* __restrict__ q, int64_t ldq, const double* __restrict__ rec,
             const int32_t* __restrict__ offs, const int32_t* __restrict__ perm, int64_t nchunk,
             double* __restrict__ part) {
    const int64_t o = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
    const int gq = threadIdx.x & 7;
    int32_t s0, s1;
    if (o >= nchunk || !bwd_chunk<4>(g, q, ldq, offs, perm, o, &s0, &s1)) return;
    Sums4 S;
    sums4_zero(S);
    sums4_rows(rec, s0, s1, gq, S);
    double* p = part + o * (8 * SUMS4) + gq;
#pragma unroll
    for (int i = 0; i < 32; ++i) p[8 * i] = S.ring[i >> 3][(i >> 2) & 1][i & 3];
    p[8 * 32] = S.cb[0];
    p[8 * 33] = S.cb[1];
    p[8 * 34] = S.a85;
}

__global__ void __launch_bounds__(256)
k_bwd_block4(ArbGeom g, const double* __restrict__ rec, const int32_t* __restrict__ offs,
             int64_t nbx, int64_t nby, const double* __restrict__ part,
             double* __restrict__ tiles) {
    // [z][cy][cx][ex + 4 ey] and [z][y][cx][ex]; a plane of t2 and a row of t1
    // padded so that the threads of the y and x passes spread over the banks
    constexpr int P2 = B4Y * B4X * 16 + 12, P1 = B4X * 4 + 2;
    __shared__ __align__(16) double t2[N4Z * P2];
    __shared__ __align__(16) double t1[N4Z * N4Y * P1];
    __shared__ __align__(16) double gb[B4X * B4Y * B4Z][16];    // G_bar per cell
    const int64_t blk = blockIdx.x;
    const int64_t bx = blk % nbx, by = (blk / nbx) % nby, bz = blk / (nbx * nby);
    const int cl = threadIdx.x >> 3, gq = threadIdx.x & 7;
    const int cx = cl & 3, cy = (cl >> 2) & 3, cz = cl >> 4;
    const int64_t x = bx * B4X + cx, y = by * B4Y + cy, z = bz * B4Z + cz;
    const bool in = x < g.npos[0] && y < g.npos[1] && z < g.npos[2];
    const int64_t c0 = x + g.npos[0] * (y + g.npos[1] * z);
    const int64_t layer = g.npos[0] * g.npos[1] * g.npos[2];
    const int32_t nct = (int32_t)g.npos[3], nt = (int32_t)g.n[3];
    double* out = tiles + blk * nt * TILE4;
    Sums4 S;
    sums4_zero(S);
    int idle = 4;                                    // layers since the last query
    // the bounds of the next layer's cell are loaded before this layer's sums
    int32_t n0 = 0, n1 = 0;
    auto fetch = [&](int32_t ct) {
        n0 = n1 = 0;
        if (in && ct < nct) {
            const int64_t c = c0 + layer * ct;
            n0 = offs[c];
            n1 = offs[c + 1];
        }
    };
    fetch(0);
    for (int32_t ct = 0; ct < nt; ++ct) {
        const int32_t s0 = n0, s1 = n1;
        fetch(ct + 1);
        idle = __syncthreads_or(s1 > s0) ? 0 : idle + 1;
        if (idle > 3) {                              // nothing in reach of this plane
            for (int t = threadIdx.x; t < TILE4; t += 256) out[(int64_t)ct * TILE4 + t] = 0.0;
            continue;
        }
        if (idle == 0) {
            S.cb[0] = S.cb[1] = S.a85 = 0.0;
            if (s1 - s0 <= BWD_CHUNK_OF<4>) {
                sums4_rows(rec, s0, s1, gq, S);
            } else {
                // the queries before the cell's first chunk, then its chunks
                const int64_t ofirst = ((int64_t)s0 + BWD_CHUNK_OF<4> - 1) / BWD_CHUNK_OF<4>;
                const int32_t h1 = ofirst * BWD_CHUNK_OF<4> < s1 ? (int32_t)(ofirst * BWD_CHUNK_OF<4>) : s1;
                sums4_rows(rec, s0, h1, gq, S);
                for (int64_t o = ofirst; o * BWD_CHUNK_OF<4> < s1; ++o) {
                    const double* p = part + o * (8 * SUMS4) + gq;
#pragma unroll
                    for (int i = 0; i < 32; ++i) S.ring[i >> 3][(i >> 2) & 1][i & 3] += p[8 * i];
                    S.cb[0] += p[8 * 32];
                    S.cb[1] += p[8 * 33];
                    S.a85 += p[8 * 34];
                }
            }
            // alpha_85 = 0: its part of the sums (M[1][ot] along t; P's column 0)
            if (gq == 2) {
                S.ring[0][1][1] += 0.5 * S.a85;
                S.ring[2][1][1] -= 0.5 * S.a85;
            }
            if (gq == 0) S.cb[0] -= S.a85;
            // G_bar(j) = c_bar_{j+1} - c_bar_j, corners j = gq and gq + 8
            const int lane = threadIdx.x & 63, nl = (lane & ~7) | ((gq + 1) & 7);
            const double n0 = __shfl(S.cb[0], nl), n1 = __shfl(S.cb[1], nl);
            gb[cl][gq] = (gq == 7 ? n1 : n0) - S.cb[0];
            gb[cl][gq + 8] = (gq == 7 ? 0.0 : n1) - S.cb[1];
            __syncthreads();
            // ring += X (x) X (x) X G_bar in (ex, ey, ez), the differences along t
            const int exh = gq & 1, ey = gq >> 1;
            if (ey) {
                const double ya = ey == 1 ? 1.0 : 0.0, yb = (double)ey;
#pragma unroll
                for (int mt = 0; mt < 2; ++mt) {
                    double r[2][2];                  // [mx][mz], summed over my
#pragma unroll
                    for (int mz = 0; mz < 2; ++mz)
#pragma unroll
                        for (int mx = 0; mx < 2; ++mx)
                            r[mx][mz] = fma(yb, gb[cl][mx + 2 + 4 * mz + 8 * mt],
                                            ya * gb[cl][mx + 4 * mz + 8 * mt]);
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const int ex = 2 * exh + p;
                        if (ex == 0) continue;
                        const double xa = ex == 1 ? 1.0 : 0.0, xb = (double)ex;
                        const double z0 = fma(xb, r[1][0], xa * r[0][0]);
                        const double z1 = fma(xb, r[1][1], xa * r[0][1]);
                        const double e[4] = {0.0, z0 + z1, 2.0 * z1, 3.0 * z1};
#pragma unroll
                        for (int ez = 1; ez < 4; ++ez) {
                            S.ring[mt][p][ez] -= 0.5 * e[ez];
                            S.ring[mt + 2][p][ez] += 0.5 * e[ez];
                        }
                    }
                }
            }
        }
        // plane ct.  z: t2[z][cy][cx][exy] = sum over cz + oz = z of
        // sum_ez M[ez][oz] ring[0][exy][ez], the lower cell layer first
#pragma unroll
        for (int ph = 0; ph < B4Z; ++ph) {
            if (cz == ph) {
#pragma unroll
                for (int oz = 0; oz < 4; ++oz) {
                    double2* o = reinterpret_cast<double2*>(t2 + (ph + oz) * P2 + (4 * cy + cx) * 16 + 2 * gq);
                    double2 b = make_double2(
                        mcol(oz, S.ring[0][0][0], S.ring[0][0][1], S.ring[0][0][2], S.ring[0][0][3]),
                        mcol(oz, S.ring[0][1][0], S.ring[0][1][1], S.ring[0][1][2], S.ring[0][1][3]));
                    if (ph > 0 && oz < 3) {
                        b.x += o->x;
                        b.y += o->y;
                    }
                    *o = b;
                }
            }
            __syncthreads();
        }
        // y: t1[z][y][cx][ex] = sum_{cy + oy = y} sum_ey M[ey][oy] t2[z][cy][cx][ex + 4 ey],
        // a thread per (z, cx, ex): its 16 values read once, 7 sums
        if (threadIdx.x < N4Z * B4X * 4) {
            const int ex = threadIdx.x & 3, tx = (threadIdx.x >> 2) & 3, zz = threadIdx.x >> 4;
            double sum[N4Y];
#pragma unroll
            for (int i = 0; i < N4Y; ++i) sum[i] = 0.0;
#pragma unroll
            for (int ty = 0; ty < B4Y; ++ty) {
                const double* a = t2 + zz * P2 + (4 * ty + tx) * 16 + ex;
                const double a0 = a[0], a1 = a[4], a2 = a[8], a3 = a[12];
#pragma unroll
                for (int oy = 0; oy < 4; ++oy) sum[ty + oy] += mcol(oy, a0, a1, a2, a3);
            }
#pragma unroll
            for (int i = 0; i < N4Y; ++i) t1[(zz * N4Y + i) * P1 + 4 * tx + ex] = sum[i];
        }
        __syncthreads();
        // x: the plane's nodes, sum_{cx + ox = x} sum_ex M[ex][ox] t1[z][y][cx][ex],
        // a thread per (z, y) row
        if (threadIdx.x < N4Z * N4Y) {
            const double* a = t1 + threadIdx.x * P1;
            double sum[N4X];
#pragma unroll
            for (int i = 0; i < N4X; ++i) sum[i] = 0.0;
#pragma unroll
            for (int tx = 0; tx < B4X; ++tx)
#pragma unroll
                for (int ox = 0; ox < 4; ++ox)
                    sum[tx + ox] += mcol(ox, a[4 * tx], a[4 * tx + 1], a[4 * tx + 2], a[4 * tx + 3]);
            double* o = out + (int64_t)ct * TILE4 + threadIdx.x * N4X;
#pragma unroll
            for (int i = 0; i < N4X; ++i) o[i] = sum[i];
        }
        // the ring moves on by one plane
#pragma unroll
        for (int o = 0; o < 4; ++o)
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int e = 0; e < 4; ++e) S.ring[o][p][e] = o < 3 ? S.ring[o + 1][p][e] : 0.0;
    }
}

// Node gradient: the sum, over the blocks whose tile holds the node (at most
// two in x and y, three in z), of the tile entries, blocks in ascending z, y,
// x order.
__global__ void __launch_bounds__(256)
k_bwd_nodes4(ArbGeom g, const double* __restrict__ tiles, int64_t nbx, int64_t nby, int64_t nbz,
             double* __restrict__ dval) {
    const int64_t nidx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (nidx >= g.nnodes) return;
    const int64_t i = nidx % g.n[0], j = (nidx / g.n[0]) % g.n[1];
    const int64_t r = nidx / (g.n[0] * g.n[1]), k = r % g.n[2], t = r / g.n[2];
    // the first block of edge b whose tile (b + 3 nodes) reaches node v
    auto lo = [](int64_t v, int b) { const int64_t w = v - (b + 2); return w <= 0 ? (int64_t)0 : (w + b - 1) / b; };
    const int64_t x0 = lo(i, B4X), x1 = min(i / B4X, nbx - 1);
    const int64_t y0 = lo(j, B4Y), y1 = min(j / B4Y, nby - 1);
    const int64_t z0 = lo(k, B4Z), z1 = min(k / B4Z, nbz - 1);
    double sum = 0.0;
    for (int64_t bz = z0; bz <= z1; ++bz)
        for (int64_t by = y0; by <= y1; ++by)
            for (int64_t bx = x0; bx <= x1; ++bx) {
                const int64_t blk = bx + nbx * (by + nby * bz);
                const int64_t e = (i - B4X * bx) + N4X * ((j - B4Y * by) + N4Y * (k - B4Z * bz));
                sum += tiles[(blk * g.n[3] + t) * TILE4 + e];
            }
    dval[nidx] = sum;
}

inline unsigned grid1(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

hipError_t arb_launch_bwd_keys(const ArbGeom& g, const double* q, int64_t n, int64_t ldq,
                               int32_t* key, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (g.ndim == 3)
        hipLaunchKernelGGL(k_bwd_keys<3>, dim3(grid1(n, 256)), dim3(256), 0, s, g, q, n, ldq, key);
    else
        hipLaunchKernelGGL(k_bwd_keys<4>, dim3(grid1(n, 256)), dim3(256), 0, s, g, q, n, ldq, key);
    return hipGetLastError();
}

hipError_t arb_launch_bwd_points(const ArbGeom& g, int32_t prec, const void* table,
                                 int32_t ninterp, int32_t kn, const double* q, int64_t n,
                                 int64_t ldq, const double* gv, const double* gg, double* dq,
                                 const int32_t* perm, int32_t* key, double* rec,
                                 hipStream_t s) {
    if (n <= 0) return hipSuccess;
    dim3 grid(grid1(n, 256)), block(256);
    if (g.ndim == 3) {
        if (prec == ARB_PREC_FP64)
            hipLaunchKernelGGL((k_bwd_points<3, double>), grid, block, 0, s, g, (const double*)table,
                               ninterp, kn, q, n, ldq, gv, gg, dq, perm, key, rec);
        else
            hipLaunchKernelGGL((k_bwd_points<3, float>), grid, block, 0, s, g, (const float*)table,
                               ninterp, kn, q, n, ldq, gv, gg, dq, perm, key, rec);
    } else {
        if (prec == ARB_PREC_FP64)
            hipLaunchKernelGGL((k_bwd_points<4, double>), grid, block, 0, s, g, (const double*)table,
                               ninterp, kn, q, n, ldq, gv, gg, dq, perm, key, rec);
        else
            hipLaunchKernelGGL((k_bwd_points<4, float>), grid, block, 0, s, g, (const float*)table,
                               ninterp, kn, q, n, ldq, gv, gg, dq, perm, key, rec);
    }
    return hipGetLastError();
}

// Blocks of the 3D node adjoint per axis, and the scratch it needs (doubles).
void arb_bwd_blocks3(const ArbGeom& g, int64_t* nb3) {
    for (int a = 0; a < 3; ++a) nb3[a] = (g.npos[a] + BB - 1) / BB;
}

int64_t arb_bwd_rec_elems(const ArbGeom& g) { return g.ndim == 3 ? 8 : REC4; }

void arb_bwd_blocks4(const ArbGeom& g, int64_t* nb4) {
    nb4[0] = (g.npos[0] + B4X - 1) / B4X;
    nb4[1] = (g.npos[1] + B4Y - 1) / B4Y;
    nb4[2] = (g.npos[2] + B4Z - 1) / B4Z;
}

int64_t arb_bwd_scratch(const ArbGeom& g) {
    int64_t nb[3];
    if (g.ndim == 3) {
        arb_bwd_blocks3(g, nb);
        return nb[0] * nb[1] * nb[2] * BTILE;
    }
    arb_bwd_blocks4(g, nb);
    return nb[0] * nb[1] * nb[2] * g.n[3] * TILE4;
}

static int64_t chunk_rows(const ArbGeom& g) {
    return g.ndim == 3 ? BWD_CHUNK_OF<3> : BWD_CHUNK_OF<4>;
}

int64_t arb_bwd_part_elems(const ArbGeom& g, int64_t n) {
    const int64_t nchunk = (n + chunk_rows(g) - 1) / chunk_rows(g);
    return (nchunk ? nchunk : 1) * (g.ndim == 3 ? 64 : 8 * SUMS4);
}

hipError_t arb_launch_bwd_cells(const ArbGeom& g, const double* q, int64_t ldq, const double* rec,
                                int32_t rec_grouped, const int32_t* offs, const int32_t* perm,
                                int64_t n, double* part, double* bbar, hipStream_t s) {
    const int32_t* rperm = rec_grouped ? nullptr : perm;
    const int64_t nchunk = (n + chunk_rows(g) - 1) / chunk_rows(g);
    int64_t nb[3];
    if (g.ndim == 3) {
        if (nchunk > 0)
            hipLaunchKernelGGL(k_bwd_chunk3, dim3(grid1(nchunk, 64)), dim3(256), 0, s, g, q, ldq,
                               rec, offs, perm, rperm, nchunk, part);
        arb_bwd_blocks3(g, nb);
        hipLaunchKernelGGL(k_bwd_block3, dim3((unsigned)(nb[0] * nb[1] * nb[2])), dim3(256), 0,
                           s, g, rec, offs, rperm, nb[0], nb[1], (const double*)part, bbar);
    } else {
        if (nchunk > 0)
            hipLaunchKernelGGL(k_bwd_chunk4, dim3(grid1(nchunk, 32)), dim3(256), 0, s, g, q, ldq,
                               rec, offs, perm, nchunk, part);
        arb_bwd_blocks4(g, nb);
        hipLaunchKernelGGL(k_bwd_block4, dim3((unsigned)(nb[0] * nb[1] * nb[2])), dim3(256), 0,
                           s, g, rec, offs, nb[0], nb[1], (const double*)part, bbar);
    }
    return hipGetLastError();
}

hipError_t arb_launch_bwd_nodes(const ArbGeom& g, const double* bbar, double* dval, hipStream_t s) {
    dim3 grid(grid1(g.nnodes, 256)), block(256);
    int64_t nb[3];
    if (g.ndim == 3) {
        arb_bwd_blocks3(g, nb);
        hipLaunchKernelGGL(k_bwd_nodes3, grid, block, 0, s, g, bbar, nb[0], nb[1], nb[2], dval);
    } else {
        arb_bwd_blocks4(g, nb);
        hipLaunchKernelGGL(k_bwd_nodes4, grid, block, 0, s, g, bbar, nb[0], nb[1], nb[2], dval);
    }
    return hipGetLastError();
}
