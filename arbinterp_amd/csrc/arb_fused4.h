// Quadcubic coefficients of a block of 4 x 4 x 2 cells in (x, y, z) at one
// t, formed in LDS from node values, for the 4D query that evaluates without
// the coefficient table (k_query.hip).  The operations of the table build
// (k_coef.hip, arb_sep4.h) in its order, so the coefficients are the table's
// bits.
//
// A row takes four lanes, one per power et of t.  passes() leaves in LDS, for
// every et, the 16 (ex, ey) values of each (cell column, node plane) after
// the t, x and y passes, and the row-shift correction folded over x, y and t;
// a lane forms the z pass and the rest of the correction in registers, four
// coefficients (ez) of one (ex, ey) at a time (coef), straight into Horner's
// rule of its t slice.  The lanes of a quad then exchange their slices'
// results (quad_all) and finish along t.  So 256 coefficients per cell are
// neither written nor read: the table is 2 KB a cell and interpolant, the
// node values 8 bytes.
//
// A workgroup runs through layers of t of one (x, y, z) block, a node plane
// ahead: a step needs one new plane of 7 x 7 x 5 nodes, and the loads of the
// next step's plane and rows are in flight during this one's passes and
// evaluation (with one layer per workgroup the wait for them was most of its
// time).  78 KB of LDS: two workgroups of 256 threads per CU.  The block is a
// full workgroup's work at the densities queries come in (1.7 rows per cell:
// 54 of its 64 rows), and one layer of t at a time keeps t2 at 46 KB.
#pragma once
#include "arb_sep4.h"

namespace arbf4 {

constexpr int BX = 4, BY = 4, BZ = 2, TH = 256;
constexpr int NX = BX + 3, NY = BY + 3, NZ = BZ + 3, NT3 = NX * NY * NZ, NT4 = 4 * NT3;
constexpr int GX = BX + 1, GY = BY + 1, GZ = BZ + 1, NG = GX * GY * GZ;
constexpr int NC = BX * BY * BZ;
constexpr int ROWS = TH / 4;                        // rows evaluated at a time
constexpr int SEG = 64;                             // layers of a workgroup at most
// doubles per (cell column, node plane) of t2: 16 values, padded so that
// neighbouring columns start in different banks; and the powers of t apart
constexpr int CS = 18, PL = BX * BY * CS, ETS = NZ * PL + 8;

struct Smem {
    double t2[4 * ETS];                             // [et][z][cy][cx][4 ey + ex]
    double2 cs[NC * 27];                            // [cell][et - 1][ey - 1][ex - 1]: S(mz = 0, 1)
    double nodes[4 * NT3];                          // plane t in slot t & 3: [z][y][x]
    double pw[4 * NT3];                             // the powers of t: [et][z][y][x]
    double gc[2 * NG];                              // xyzt differences, corner plane t in t & 1
    int2 rows[SEG];                                 // the layers' sorted positions
    unsigned char bad[NC];                          // cells with a non-finite stencil
};

// The block's node column of this thread (tid < NT3: one (x, y, z)), four
// planes of t from the current layer's first on.
struct Column {
    int64_t src;                                    // its first plane's node
    bool in;
    double v[4], next;
    unsigned nf;                                    // non-finite among v, newest lowest
};

__device__ __forceinline__ void column_origin(const ArbGeom& g, const int64_t* c0, Column& C) {
    const int e = threadIdx.x, x = e % NX, y = (e / NX) % NY, z = e / (NX * NY);
    const int64_t nx = c0[0] + x, ny = c0[1] + y, nz = c0[2] + z;
    // nodes past the grid read as 0 (only cells outside the grid use them);
    // the loads are unconditional (index 0 when unused)
    C.in = e < NT3 && nx < g.n[0] && ny < g.n[1] && nz < g.n[2];
    C.src = C.in ? nx + g.nstride[1] * ny + g.nstride[2] * nz : 0;
}

__device__ __forceinline__ double column_load(const double* __restrict__ F, const ArbGeom& g,
                                              const Column& C, int64_t plane) {
    return F[C.src + (C.in ? g.nstride[3] * plane : 0)];
}

// The planes t .. t + 3 before the first step.
__device__ __forceinline__ void column_start(const double* __restrict__ F, const ArbGeom& g,
                                             int64_t t, Column& C, Smem& S) {
#pragma unroll
    for (int j = 0; j < 4; ++j) C.v[j] = column_load(F, g, C, t + j);
    C.nf = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (!C.in) C.v[j] = 0.0;
        C.nf = 2 * C.nf + (isfinite(C.v[j]) ? 0 : 1);
        if (threadIdx.x < NT3) S.nodes[((t + j) & 3) * NT3 + threadIdx.x] = C.v[j];
    }
}

// On to layer t: its last plane, t + 3, is C.next.
__device__ __forceinline__ void column_step(int64_t t, Column& C, Smem& S) {
#pragma unroll
    for (int j = 0; j < 3; ++j) C.v[j] = C.v[j + 1];
    C.v[3] = C.in ? C.next : 0.0;
    C.nf = (2 * C.nf + (isfinite(C.v[3]) ? 0 : 1)) & 15;
    if (threadIdx.x < NT3) S.nodes[((t + 3) & 3) * NT3 + threadIdx.x] = C.v[3];
}

// The passes of layer t.  Block-wide: a barrier behind column_start /
// column_step comes before passes_t (the powers of t and the xyzt
// differences; half: gc holds the corner plane t + 1 already), one before
// passes_xy, one after it.
__device__ __forceinline__ void passes_t(int64_t t, const Column& C, bool half, bool anybad, Smem& S) {
    const int tid = threadIdx.x;
    if (anybad && tid < NC) {
        const int cx = tid % BX, cy = (tid / BX) % BY, cz = tid / (BX * BY);
        bool bad = false;
#pragma unroll 1
        for (int r = 0; r < 64; ++r)
            for (int x = 0; x < 4; ++x)
                bad |= !isfinite(S.nodes[(((r >> 4) * NZ + cz + ((r >> 2) & 3)) * NY + cy + (r & 3)) * NX +
                                         cx + x]);
        S.bad[tid] = bad ? 1 : 0;
    }
    if (tid < NT3) {
        double c[4];
        arbs3::cub4(C.v[0], C.v[1], C.v[2], C.v[3], c);
#pragma unroll
        for (int e = 0; e < 4; ++e) S.pw[tid + e * NT3] = c[e];
    }
    // xyzt differences of corner planes t + 1 and t + 2, from the last thread
    // on: arbs4::corner_diff's terms in its order
    for (int i = TH - 1 - tid + (half ? NG : 0); i < 2 * NG; i += TH) {
        const int gt = i >= NG ? 1 : 0, r = i - gt * NG;
        const int gx = r % GX, gy = (r / GX) % GY, gz = r / (GX * GY);
        const int64_t p = t + 1 + gt;
        const double* at = S.nodes + ((gz + 1) * NY + gy + 1) * NX + gx + 1;
        double acc = 0.0;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int off = ((m & 1) ? 1 : -1) + ((m & 2) ? NX : -NX) + ((m & 4) ? NX * NY : -NX * NY);
            const double v = at[(int)((m & 8 ? p + 1 : p - 1) & 3) * NT3 + off];
            acc += (__builtin_popcount(~m & 15) & 1) ? -v : v;
        }
        S.gc[(int)(p & 1) * NG + r] = acc * 0.0625;
    }
}

// The x and y passes and the correction's sums over x, y and t.
__device__ __forceinline__ void passes_xy(int64_t t, Smem& S) {
    const int tid = threadIdx.x;
    // x and y passes of one (power of t, cell column, node plane) per item; a
    // row's x pass is formed again for the up to four columns in y that use
    // it, which saves an LDS round trip and a barrier
    for (int i = tid; i < BX * BY * NZ * 4; i += TH) {
        const int x = i % BX, y = (i / BX) % BY, r = i / (BX * BY), z = r % NZ, et = r / NZ;
        double cxp[4][4];                           // [oy][ex]
#pragma unroll
        for (int oy = 0; oy < 4; ++oy) {
            const double* nd = S.pw + et * NT3 + (z * NY + y + oy) * NX + x;
            arbs3::cub4(nd[0], nd[1], nd[2], nd[3], cxp[oy]);
        }
        double* out = S.t2 + et * ETS + z * PL + (y * BX + x) * CS;
#pragma unroll
        for (int h = 0; h < 4; h += 2) {
            double ca[4], cb[4];
            arbs3::cub4(cxp[0][h], cxp[1][h], cxp[2][h], cxp[3][h], ca);
            arbs3::cub4(cxp[0][h + 1], cxp[1][h + 1], cxp[2][h + 1], cxp[3][h + 1], cb);
#pragma unroll
            for (int ey = 0; ey < 4; ++ey)
                *reinterpret_cast<double2*>(out + 4 * ey + h) = make_double2(ca[ey], cb[ey]);
        }
    }
    // the correction of arbs4::shift_rows up to its sums S over x, y and t,
    // one (cell, ex) per thread
    const int i = TH - 1 - tid;
    if (i < NC * 3) {
        const int cell = i % NC, ex = 1 + i / NC;
        const int cx = cell % BX, cy = (cell / BX) % BY, cz = cell / (BX * BY);
        auto G = [&](int c) {
            return S.gc[(int)((t + 1 + ((c >> 3) & 1)) & 1) * NG +
                        ((cz + ((c >> 2) & 1)) * GY + cy + ((c >> 1) & 1)) * GX + cx + (c & 1)];
        };
        const double hx0 = arbs4::hd(ex, 0), hx1 = arbs4::hd(ex, 1);
        double X[8];                                // [my + 2 mz + 4 mt]
        double prev = 0.0;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const double g0 = G(2 * m), g1 = G(2 * m + 1);
            X[m] = fma(hx1, g0 - g1, hx0 * (prev - g0));
            prev = g1;
        }
#pragma unroll
        for (int ey = 1; ey < 4; ++ey) {
            double Y[4];                            // [mz + 2 mt]
#pragma unroll
            for (int m = 0; m < 4; ++m)
                Y[m] = fma(arbs4::hd(ey, 1), X[2 * m + 1], arbs4::hd(ey, 0) * X[2 * m]);
#pragma unroll
            for (int et = 1; et < 4; ++et) {
                const double h0 = arbs4::hd(et, 0), h1 = arbs4::hd(et, 1);
                S.cs[cell * 27 + (et - 1) * 9 + (ey - 1) * 3 + ex - 1] =
                    make_double2(fma(h1, Y[2], h0 * Y[0]), fma(h1, Y[3], h0 * Y[1]));
            }
        }
    }
}

// The four coefficients (ez) of every ex, for one ey, of power et of t in
// local cell lc (cx + BX (cy + BY cz)); al[ex][ez].
template <typename T>
__device__ __forceinline__ void coef(const Smem& S, int lc, int et, int ey, T (*al)[4]) {
    const double* col = S.t2 + et * ETS + (lc / (BX * BY)) * PL + (lc % (BX * BY)) * CS;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        double2 f[4];
#pragma unroll
        for (int z = 0; z < 4; ++z)
            f[z] = *reinterpret_cast<const double2*>(col + z * PL + 4 * ey + 2 * h);
        double c[2][4];
        arbs3::cub4(f[0].x, f[1].x, f[2].x, f[3].x, c[0]);
        arbs3::cub4(f[0].y, f[1].y, f[2].y, f[3].y, c[1]);
        if (ey > 0 && et > 0) {
            const double2* cs = S.cs + lc * 27 + (et - 1) * 9 + (ey - 1) * 3;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const int ex = 2 * h + p;
                if (ex == 0) continue;
                const double2 s = cs[ex - 1];
#pragma unroll
                for (int ez = 1; ez < 4; ++ez)
                    c[p][ez] += fma(arbs4::hd(ez, 1), s.y, arbs4::hd(ez, 0) * s.x);
                if (ex == 1 && ey == 1 && et == 1) c[p][1] = 0.0;   // row 85
            }
        }
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int ez = 0; ez < 4; ++ez) al[2 * h + p][ez] = (T)c[p][ez];
    }
}

// x of lane L of the calling lane's quad.
template <int L>
__device__ __forceinline__ float quad_lane(float x) {
    const int v = __float_as_int(x);
    return __int_as_float(__builtin_amdgcn_update_dpp(v, v, L * 0x55, 0xf, 0xf, true));
}
template <int L>
__device__ __forceinline__ int quad_lane(int v) {
    return __builtin_amdgcn_update_dpp(v, v, L * 0x55, 0xf, 0xf, true);
}
template <int L>
__device__ __forceinline__ double quad_lane(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, L * 0x55, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(lo, lo, L * 0x55, 0xf, 0xf, true));
}
// x of the four lanes of the quad (every lane of it must call).
template <typename T>
__device__ __forceinline__ void quad_all(T x, T* r) {
    r[0] = quad_lane<0>(x);
    r[1] = quad_lane<1>(x);
    r[2] = quad_lane<2>(x);
    r[3] = quad_lane<3>(x);
}

// a[e] for a runtime e in 0..3 by selects
template <typename T>
__device__ __forceinline__ T pick(int e, T a0, T a1, T a2, T a3) {
    return e < 2 ? (e == 0 ? a0 : a1) : (e == 2 ? a2 : a3);
}

// The lane's axis (et) of a row: the reduction of arb_reduce_axes, one axis per
// lane of the quad.
struct Axis {
    double lo, h, rh;
};

__device__ __forceinline__ Axis lane_axis(const ArbGeom& g, int et) {
    Axis A;
    A.lo = pick(et, g.lo[0], g.lo[1], g.lo[2], g.lo[3]);
    A.h = pick(et, g.h[0], g.h[1], g.h[2], g.h[3]);
    A.rh = pick(et, g.rh[0], g.rh[1], g.rh[2], g.rh[3]);
    return A;
}

// Local coordinate (of the lane's axis) and local cell of the quad's row in
// the block of cells at (c0, c1, c2) and layer t; x: the lane's coordinate.
// False for a row that is not in it.  row: whether the quad has one.  One
// without takes IntMin, not x, which then is another row's and may lie
// anywhere: nothing below may run on it.
//
// A row of the block is inside the box and its flat index below nc < 2^32.
// Its index along an axis can still reach past the axis: a coordinate at
// IntMax, or any beyond the cells that an axis whose first spacing is its
// smallest counts.  Only then the flat index is decoded (bucket_of, in 32
// bits), three divisions however far past it lies.
__device__ __forceinline__ bool place_row(bool row, double x, const Axis& A, const ArbGeom& g,
                                          int c0, int c1, int c2, int t, double* loc, int* lc) {
    const double a = row ? x - A.lo : 0.0;
    double iu = a * A.rh;                           // arb_div_h
    iu = fma(fma(-iu, A.h, a), A.rh, iu);
    iu = fma(fma(-iu, A.h, a), A.rh, iu);
    if (A.rh == 0.0) iu = a / A.h;
    const double fl = floor(iu);
    *loc = iu - fl;
    int q[4];
    quad_all((int)(uint32_t)fl, q);
    const uint32_t n0 = (uint32_t)g.npos[0], n1 = (uint32_t)g.npos[1], n2 = (uint32_t)g.npos[2];
    uint32_t i[4] = {(uint32_t)q[0], (uint32_t)q[1], (uint32_t)q[2], (uint32_t)q[3]};
    if (i[0] >= n0 || i[1] >= n1 || i[2] >= n2) {
        uint32_t rem = i[0] + n0 * (i[1] + n1 * (i[2] + n2 * i[3]));
        i[0] = rem % n0;
        rem /= n0;
        i[1] = rem % n1;
        rem /= n1;
        i[2] = rem % n2;
        i[3] = rem / n2;
    }
    const uint32_t l0 = i[0] - (uint32_t)c0, l1 = i[1] - (uint32_t)c1, l2 = i[2] - (uint32_t)c2;
    *lc = (int)(l0 + BX * (l1 + BY * l2));
    return l0 < (uint32_t)BX && l1 < (uint32_t)BY && l2 < (uint32_t)BZ && i[3] == (uint32_t)t;
}

}  // namespace arbf4
