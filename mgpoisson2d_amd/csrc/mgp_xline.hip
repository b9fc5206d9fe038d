// mgp_xline.hip -- x-line relaxation of the resident fast solver on gfx950.
//
// A sweep of one row colour solves, for every row j of the colour,
//     T_j delta = f - L e     (row j),   e(:, j) += delta
// where L is the reference 9-point operator with homogeneous BCs (ghosts
// eliminated) and T_j its tridiagonal part along the row: the coefficients
// of e(i-1,j), e(i,j), e(i+1,j) in (L e)(i,j).
//
// Interior cells evaluate L and T from the face metrics already loaded for
// the residual (cell_lap_interior's stencil, differentiated by hand).  Ring
// cells (i = 0, nx-1 or j = 0, ny-1), whose stencils carry the boundary
// extrapolations and the Dirichlet ghost rule, use an explicit coefficient
// table probed once per level with unit impulses (k_ring_coef).
//
// One workgroup (64 to 1024 threads) per row:
//  1. coalesced pass: each thread evaluates d = f - L e and the row
//     coefficients for cells i = tid + NT u (groups of loads issued up front);
//  2. the values go through LDS into contiguous chunks of C or C+1 cells
//     per thread (padded stride C+1: no bank conflicts);
//  3. partition method in registers: each chunk is eliminated to one row in
//     the chunks' last unknowns;
//  4. that system is solved by the first wave: one row per lane (after an
//     elimination of NT / 64 chunks per lane) by parallel cyclic reduction
//     with cross-lane shuffles;
//  5. back substitution in registers, transpose back, coalesced e update.
// Rows are mapped to workgroups so that the rows an XCD processes are
// contiguous (workgroups are dealt to the 8 XCDs round robin): neighbouring
// rows share their halo rows through that XCD's L2.
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "mgp_batch.h"
#include "mgp_host.h"
#include "mgp_kernels.h"
#include "mgp_stencil.h"

namespace mgp {

namespace {

// Threads per row of the line solve: 256; in the batched launches (many
// rows) 64 for rows of at most 512 cells and 128 up to 1024 cells, so that
// a CU holds more rows at once (a short row then occupies one or two waves).
constexpr int XL_THREADS = 256;
constexpr int XL_SHORT = 64;
constexpr int XL_SHORT_MAX_NX = 512;
constexpr int XL_MID = 128;
constexpr int XL_MID_MAX_NX = 1024;
// FP32 rows of 4112 .. 8207 cells: 512 threads, chunks of 16 (139 KB of LDS),
// so the mixed-precision cycle solves rows of 8192 cells whole.
constexpr int XL_WIDE = 512;
// The single-problem solver's launches of few rows (up to two per CU: every
// coarse level) take as long as one row solve, so they use more threads per
// row than the fine levels' launches, whose many rows fill the CUs: rows of
// 129 .. 512 cells 256 threads instead of one wave (512^2 FP64 37.5 -> 31.1 ms;
// at 128 cells and below one wave is as fast or faster), FP32 rows of 1025 ..
// 2048 cells 512 threads (1500 x 800: 18.7 -> 16.9 ms; FP64 rows of that length
// and rows of 513 .. 1024 cells were slower by 7 and 12 %).
constexpr unsigned XL_FEW_ROWS = 512;
constexpr int XL_SHORT_FEW_MAX_NX = 128;
constexpr int XL_LONG_MIN_NX = 1024, XL_LONG_MAX_NX = 2048;
constexpr int XL_WIDEST = 1024;  // FP32 rows past 4111 cells, few of them
constexpr int RING_PLANES = 9;

// Impulse whose ghosts follow the homogeneous fill of the MG levels
// (Dirichlet order 3 / LAH negate; Neumann sides contribute no ghost).
struct ImpulseFilled {
    int ci, cj;
    Grid g;
    int t[4], m[4];
    __device__ double v(int i, int j) const { return (i == ci && j == cj) ? 1.0 : 0.0; }
    __device__ static double dg(int type, int mode, double p0, double p1, double p2) {
        if (type != BC_DIRI) return 0.0;
        if (mode == MODE_LAH) return -p0;
        return -3.0 * p0 + p1 - (1.0 / 5.0) * p2;
    }
    __device__ double operator()(int i, int j) const {
        const int nx = g.nx, ny = g.ny;
        const bool xin = i >= 0 && i < nx, yin = j >= 0 && j < ny;
        if (xin && yin) return v(i, j);
        if (!xin && !yin) return 0.0;
        if (i < 0) return dg(t[XLO], m[XLO], v(0, j), v(1, j), v(2, j));
        if (i >= nx) return dg(t[XHI], m[XHI], v(nx - 1, j), v(nx - 2, j), v(nx - 3, j));
        if (j < 0) return dg(t[YLO], m[YLO], v(i, 0), v(i, 1), v(i, 2));
        return dg(t[YHI], m[YHI], v(i, ny - 1), v(i, ny - 2), v(i, ny - 3));
    }
};

__host__ __device__ inline int ring_count(int nx, int ny) { return 2 * nx + 2 * (ny - 2); }

// Every ring-cell stencil lies in a 3x3 window of valid cells: the window
// reaches inward (two cells) across each boundary side the cell touches and
// one cell either way along it.  Window origin (w0, v0) of cell (i, j):
//   w0 = 0 on column 0, -2 on column nx-1, else -1   (likewise v0 for rows).
// Ring cell index r: rows j = 0 (r = i) and ny-1 (r = nx + i), then columns
// i = 0 (r = 2 nx + j - 1) and nx-1 (r = 2 nx + ny - 2 + j - 1), 1 <= j <= ny-2.
// Table plane q = 3 a + b holds the coefficient of e(i + w0 + b, j + v0 + a).
__device__ __forceinline__ int window_origin(int i, int n) { return i == 0 ? 0 : (i == n - 1 ? -2 : -1); }

__device__ inline void ring_cell(int nx, int ny, int r, int &i, int &j) {
    if (r < 2 * nx) {
        const bool top = r >= nx;
        i = top ? r - nx : r;
        j = top ? ny - 1 : 0;
    } else {
        const int rr = r - 2 * nx;
        const bool right = rr >= ny - 2;
        i = right ? nx - 1 : 0;
        j = (right ? rr - (ny - 2) : rr) + 1;
    }
}

__device__ __forceinline__ int ring_index(int nx, int ny, int i, int j) {
    if (j == 0) return i;
    if (j == ny - 1) return nx + i;
    return 2 * nx + (i == 0 ? 0 : ny - 2) + (j - 1);
}

// (L e)(i, j) at a ring cell from the table.  All nine table entries and
// field values are loaded before any is used (one memory round trip).
// far: where the window's row two rows in is read from (cell i at
// [OFFX + i]; rows 0 and ny-1 in the line relaxation), null for the field.
template <typename T>
__device__ __forceinline__ T ring_lap(gconst<T> *e, gconst<T> *K, int nring, const Grid &g, int i, int j,
                                      gconst<T> *far = nullptr) {
    const int w0 = window_origin(i, g.nx), v0 = window_origin(j, g.ny);
    const int r = ring_index(g.nx, g.ny, i, j);
    gconst<T> *row[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) row[a] = e + ix(g.pitch, -OFFX, j + v0 + a);
    if (far && j == 0) row[2] = far;
    if (far && j == g.ny - 1) row[0] = far;
    T kv[9], ev[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        kv[q] = K[(size_t)q * nring + r];
        ev[q] = row[q / 3][OFFX + i + w0 + q % 3];
    }
    T lap = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q) lap += kv[q] * ev[q];
    return lap;
}

// Coefficients of e(i-1, j), e(i, j), e(i+1, j) at a ring cell (0 where the
// neighbour is outside the window, i.e. not a valid cell).
template <typename T>
__device__ __forceinline__ void ring_row_coef(gconst<T> *K, int nring, const Grid &g, int i, int j, T &a, T &b,
                                              T &c) {
    const int w0 = window_origin(i, g.nx), v0 = window_origin(j, g.ny);
    const int r = ring_index(g.nx, g.ny, i, j);
    const int base = 3 * (-v0);  // window row of j itself
    a = w0 <= -1 ? K[(size_t)(base + (-1 - w0)) * nring + r] : T(0);
    b = K[(size_t)(base + (0 - w0)) * nring + r];
    c = w0 + 2 >= 1 ? K[(size_t)(base + (1 - w0)) * nring + r] : T(0);
}

// K[q * nring + r]: coefficient of e(i + w0 + q%3, j + v0 + q/3) in the
// homogeneous L at ring cell r (impulse response with the ghost rule).
__global__ void __launch_bounds__(256) k_ring_coef(double *K, Grid g, Geo geo, Bc bc) {
    const int nring = ring_count(g.nx, g.ny);
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= RING_PLANES * nring) return;
    const int q = id / nring, r = id % nring;
    int i, j;
    ring_cell(g.nx, g.ny, r, i, j);
    ImpulseFilled imp;
    imp.g = g;
    for (int k = 0; k < 4; ++k) {
        imp.t[k] = bc.type[k];
        imp.m[k] = bc.mode[k];
    }
    imp.ci = i + window_origin(i, g.nx) + q % 3;
    imp.cj = j + window_origin(j, g.ny) + q / 3;
    K[id] = cell_lap(imp, g, geo, bc, 1, i, j);
}

// Position of cell i in the chunk layout: the first rem chunks hold C+1
// cells, the others C; chunk t starts at LDS slot t*(C+1).
template <int C>
__device__ __forceinline__ int chunk_pos(int i, int rem) {
    const int big = rem * (C + 1);
    if (i < big) return i;
    const int k = i - big;
    return big + (k / C) * (C + 1) + k % C;
}

// Row j of the workgroup's launch.  XCD-aware: XCD x (= blockIdx % 8) takes a
// contiguous block of q8 or q8+1 slots.
__device__ __forceinline__ int launch_slot() {
    const int nb = gridDim.x, b = blockIdx.x, x = b & 7;
    const int q8 = nb >> 3, r8 = nb & 7;
    return x * q8 + (x < r8 ? x : r8) + (b >> 3);
}

// LDS elements of a row of NT full chunks (xline_lds_bytes_for).
__host__ __device__ constexpr int row_lds_elems(int C, int NT) {
    return 4 * NT * (C + 1) > NT * (C + 1) + 8 * NT ? 4 * NT * (C + 1) : NT * (C + 1) + 8 * NT;
}

template <typename T>
struct RowCtx {
    int nx, ny, P, nt, rem, nring;
    int i0, nxg;  // the cells solved: i0 .. i0+nx-1 of a row of nxg cells (a whole row: 0, nx)
    T idx, idy, idx2, idy2, ixy4;
};

// The inverse spacings are formed in FP64 and rounded once to T.
template <typename T>
__device__ __forceinline__ RowCtx<T> row_ctx(const Grid &g, int nt, int C) {
    RowCtx<T> r;
    r.nx = g.nx;
    r.i0 = 0;
    r.nxg = g.nx;
    r.ny = g.ny;
    r.P = g.pitch;
    r.nt = nt;
    r.rem = g.nx - nt * C;
    r.nring = ring_count(g.nx, g.ny);
    const double idx = 1.0 / g.dx, idy = 1.0 / g.dy;
    r.idx = (T)idx;
    r.idy = (T)idy;
    r.idx2 = (T)(idx * idx);
    r.idy2 = (T)(idy * idy);
    r.ixy4 = (T)(0.25 * idx * idy);
    return r;
}

// Buffer-addressed reads of a field of a level: one 32-bit byte offset per
// cell in a vector register, the row offsets (multiples of the pitch) in
// scalar registers and the column neighbours in the instruction's immediate
// offset.  Flat loads need a 64-bit address per array and neighbour: in the
// batched mid-row kernel 350 of its 2700 vector instructions were 64-bit
// address arithmetic.  A buffer of 2^31 - 1 bytes from the start of the
// row above the one solved: the reads span three rows, so none is clipped.
template <typename T>
struct Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ explicit Buf(const T *p)
        : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(p), 0, 0x7fffffff, 0x00020000)) {}
    __device__ __forceinline__ T operator()(int vo, int so) const {
        if constexpr (sizeof(T) == 4)
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0));
        else
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0));
    }
};

// Coalesced pass over row j: for cells i = tid + NT u, the residual
// d = f - L e and the row coefficients a, b, c, written into the chunk layout
// (Ld, La, Lb, Lc).  Interior cells use the metric stencil, ring cells the
// table.  Lanes past the row end evaluate the last cell and store into the
// chunk layout's last slot, which no chunk uses (the last chunk has C cells):
// the loop stays branch-free.
//
// RG cells' loads are issued together before their stencils are evaluated,
// so RG memory round trips overlap instead of following one another (one
// cell at a time, a coarse-level row pass took 5.4 us of a 10.6 us row
// solve).  The batched kernels take the RG of batch_rg: no more than fits
// their VGPR budget, since they rely on many workgroups per CU.
template <int C, int NT, bool SEG = false, int RG = 1, typename T, typename GM>
__device__ __forceinline__ void row_pass(const RowCtx<T> &X, const T *e_, const T *f_, const T *K_, const Grid &g,
                                         const GM &geo_, int j, const T *far, int tid, T *Ld, T *La, T *Lb, T *Lc,
                                         T (&ev)[C + 1]) {
    constexpr int U = C + 1;
    gconst<T> *e = gptr(e_), *f = gptr(f_), *K = gptr(K_);
    // SEG: the cells solved may be a segment of the row (xline_rows); whole
    // rows compile without the segment terms
    const int nx = X.nx, ny = X.ny, P = X.P, i0 = SEG ? X.i0 : 0, nxg = SEG ? X.nxg : X.nx;
    const T fourth = T(0.25);
    const int dump = X.nt * (C + 1) - 1;
    // A segment of a longer row is solved as a line of its own: its couplings
    // to the cells beyond its ends (in the neighbouring segments) stay in the
    // residual and leave its tridiagonal system (a = 0 at its first cell,
    // c = 0 at its last), as in block Gauss-Seidel over the segments.
    const bool cut_w = SEG && i0 > 0, cut_e = SEG && i0 + nx < nxg;
    if (j != 0 && j != ny - 1) {
        // the buffers start at cell (-1, j-1) of each array (j is the same
        // for the whole workgroup), so the offsets are small and never
        // negative whatever the array's size
        const size_t r0 = ix(P, 0, j - 1) - 1;
        const Buf<T> bE(e_ + r0), bJxx(geo_.Jxx + r0), bJxy(geo_.Jxy + r0), bJyy(geo_.Jyy + r0),
            bJyx(geo_.Jyx + r0), bF(f_ + r0);
        struct CellIn {
            T p, pe, pw, pn, ps, ene, enw, ese, esw, Jxx_e, Jxx_w, Jxy_e, Jxy_w, Jyy_n, Jyy_s, Jyx_n, Jyx_s, fv;
        };
#pragma unroll
        for (int u0 = 0; u0 < U; u0 += RG) {
            CellIn in[RG];
#pragma unroll
            for (int r = 0; r < RG; ++r) {
                const int u = u0 + r;
                if (u >= U) break;
                const int iraw = tid + NT * u;
                const int il = iraw < nx ? iraw : nx - 1;
                const size_t c = ix(P, i0 + il, j);
                // interior stencil; for i = 0, nx-1 the reads stay inside the
                // padded level and the values are replaced below
                // bytes from cell (i-1, j-1) (i elements past the buffer's
                // start); rows j and j+1 one and two pitches on
                constexpr int ES = (int)sizeof(T);
                const int vo = (int)((c - P - 1 - r0) * ES), s1 = P * ES, s2 = 2 * P * ES;
                in[r].esw = bE(vo, 0);
                in[r].ps = bE(vo + ES, 0);
                in[r].ese = bE(vo + 2 * ES, 0);
                in[r].pw = bE(vo, s1);
                in[r].p = bE(vo + ES, s1);
                in[r].pe = bE(vo + 2 * ES, s1);
                in[r].enw = bE(vo, s2);
                in[r].pn = bE(vo + ES, s2);
                in[r].ene = bE(vo + 2 * ES, s2);
                in[r].Jxx_w = bJxx(vo + ES, s1);
                in[r].Jxx_e = bJxx(vo + 2 * ES, s1);
                in[r].Jxy_w = bJxy(vo + ES, s1);
                in[r].Jxy_e = bJxy(vo + 2 * ES, s1);
                in[r].Jyy_s = bJyy(vo + ES, s1);
                in[r].Jyy_n = bJyy(vo + ES, s2);
                in[r].Jyx_s = bJyx(vo + ES, s1);
                in[r].Jyx_n = bJyx(vo + ES, s2);
                in[r].fv = bF(vo + ES, s1);
            }
#pragma unroll
            for (int r = 0; r < RG; ++r) {
                const int u = u0 + r;
                if (u >= U) break;
                const int iraw = tid + NT * u;
                const int il = iraw < nx ? iraw : nx - 1;
                const CellIn &v = in[r];
                const T xfe = v.Jxx_e * (v.pe - v.p) * X.idx + v.Jxy_e * fourth * (v.ene - v.ese + v.pn - v.ps) * X.idy;
                const T xfw = v.Jxx_w * (v.p - v.pw) * X.idx + v.Jxy_w * fourth * (v.pn - v.ps + v.enw - v.esw) * X.idy;
                const T yfn = v.Jyy_n * (v.pn - v.p) * X.idy + v.Jyx_n * fourth * (v.ene - v.enw + v.pe - v.pw) * X.idx;
                const T yfs = v.Jyy_s * (v.p - v.ps) * X.idy + v.Jyx_s * fourth * (v.pe - v.pw + v.ese - v.esw) * X.idx;
                ev[u] = v.p;
                const int o = iraw < nx ? chunk_pos<C>(il, X.rem) : dump;
                Ld[o] = v.fv - ((xfe - xfw) * X.idx + (yfn - yfs) * X.idy);
                La[o] = cut_w && il == 0 ? T(0) : v.Jxx_w * X.idx2 - (v.Jyx_n - v.Jyx_s) * X.ixy4;
                Lb[o] = -(v.Jxx_e + v.Jxx_w) * X.idx2 - (v.Jyy_n + v.Jyy_s) * X.idy2;
                Lc[o] = cut_e && il == nx - 1 ? T(0) : v.Jxx_e * X.idx2 + (v.Jyx_n - v.Jyx_s) * X.ixy4;
            }
        }
        // the two ring cells of the row (i = 0, nxg-1), where they lie in
        // the cells solved: explicit stencil table
        for (int side = 0; side < 2; ++side) {
            const int iend = side ? nxg - 1 : 0, il = iend - i0;
            if (il < 0 || il >= nx || il % NT != tid) continue;
            const int o = chunk_pos<C>(il, X.rem);
            Ld[o] = f[ix(P, iend, j)] - ring_lap(e, K, X.nring, g, iend, j);
            ring_row_coef(K, X.nring, g, iend, j, La[o], Lb[o], Lc[o]);
        }
    } else {
        // boundary row: every cell from the table
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int iraw = tid + NT * u;
            const int il = iraw < nx ? iraw : nx - 1;
            const int i = i0 + il;
            ev[u] = e[ix(P, i, j)];
            const T fv = f[ix(P, i, j)];
            const T lap = ring_lap(e, K, X.nring, g, i, j, gptr(far));
            T a, b, c;
            ring_row_coef(K, X.nring, g, i, j, a, b, c);
            const int o = iraw < nx ? chunk_pos<C>(il, X.rem) : dump;
            Ld[o] = fv - lap;
            La[o] = cut_w && il == 0 ? T(0) : a;
            Lb[o] = b;
            Lc[o] = cut_e && il == nx - 1 ? T(0) : c;
        }
    }
}

// Coalesced update e(:, j) += x, x in the chunk layout.  The row pass's values
// ev serve where registers hold them across the solve (one memory round trip
// less); the 17-cell chunks and the segmented kernels would spill them.
template <int C, bool SEG>
constexpr bool keep_values() {
    return C < 16 && !SEG;
}

template <int C, int NT, bool SEG = false, typename T>
__device__ __forceinline__ void row_update_add(const RowCtx<T> &X, T *e_, int j, int tid, const T *Lx,
                                               const T (&ev)[C + 1]) {
    __attribute__((address_space(1))) T *e = (__attribute__((address_space(1))) T *)e_;
#pragma unroll
    for (int u = 0; u < C + 1; ++u) {
        const int i = tid + NT * u;
        if (i >= X.nx) continue;
        const size_t c = ix(X.P, (SEG ? X.i0 : 0) + i, j);
        e[c] = (keep_values<C, SEG>() ? ev[u] : e[c]) + Lx[chunk_pos<C>(i, X.rem)];
    }
}

// Reciprocals of the line solves: v_rcp_f64 (measured error up to 4.4e-8)
// refined by two Newton steps, which leaves 1.1e-16, an ulp (2e-15 after
// one).  Each is used for several products, so an error in it would act as
// a perturbation of the row's diagonal, times the row system's condition.
__device__ __forceinline__ double rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
    return __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
}
// FP32: v_rcp_f32 alone (about 1 ulp).
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }

template <typename T>
struct Row4 {
    T a, b, c, d;
};

// ---------------------------------------------------------------------------
// The row system is solved by partition.  A chunk of consecutive rows is
// eliminated to one row in the last unknowns of the chunks (its own, the
// previous and the next chunk's): a forward sweep leaves the chunk's last row
// in terms of the previous chunk's last unknown, its own and the next chunk's
// first, and the back substitution gives every other unknown of the chunk,
// the first included, as a linear form G + H x_prev + M x_last.  Each row
// costs one reciprocal.  What bounds a row is this serial chain and the row
// pass before it; keeping both ends of each chunk as unknowns took two sweeps,
// three reciprocals a row and a system of twice the size (single FP64 solves:
// 64^2 13.54 -> 10.56 ms, 512^2 52.4 -> 43.4, 2048^2 134.7 -> 116.0).
// ---------------------------------------------------------------------------
// Rows a x(k-1) + b x(k) + c x(k+1) = d, k = 0 .. len-1 (len = N or N-1 >= 2).
// On return (a, b, c, d) at row len-1 are the last row's coefficients of
// x_prev, x_last and the next chunk's first unknown, and its right-hand side;
// at the rows before, (d, a, c) hold the forms (G, H, M).
template <int N, bool SHORT, typename T>
__device__ __forceinline__ void eliminate(T (&a)[N], T (&b)[N], T (&c)[N], T (&d)[N], int len, Row4<T> &last) {
    T ib[N];
    ib[0] = rcp(b[0]);
#pragma unroll
    for (int k = 1; k < N; ++k)
        if (!SHORT || k < N - 1 || len == N) {
            const T r = a[k] * ib[k - 1];
            a[k] = -r * a[k - 1];
            b[k] = b[k] - r * c[k - 1];
            d[k] = d[k] - r * d[k - 1];
            ib[k] = rcp(b[k]);
        }
    const bool full = !SHORT || len == N;
    last = Row4<T>{full ? a[N - 1] : a[N - 2], full ? b[N - 1] : b[N - 2], full ? c[N - 1] : c[N - 2],
                   full ? d[N - 1] : d[N - 2]};
    T G = 0, H = 0, M = 1;
#pragma unroll
    for (int k = N - 2; k >= 0; --k)
        if (!SHORT || k < N - 2 || len == N) {
            G = (d[k] - c[k] * G) * ib[k];
            H = (-a[k] - c[k] * H) * ib[k];
            M = (-c[k] * M) * ib[k];
            d[k] = G;
            a[k] = H;
            c[k] = M;
        }
}

// The last row with the next chunk's first unknown g + h x_last + m x_next put in.
template <typename T>
__device__ __forceinline__ Row4<T> join(const Row4<T> &r, T g, T h, T m) {
    return Row4<T>{r.a, r.b + r.c * h, r.c * m, r.d - r.c * g};
}

// Solves the 64-row tridiagonal system of one row per lane by parallel cyclic
// reduction on rows scaled to a unit diagonal (one reciprocal and six
// shuffles a step); n: rows that are not identity rows.  A lane whose
// neighbour is missing has a (or c) = 0, so what it is handed does not count.
template <typename T>
__device__ __forceinline__ T wave_pcr(const Row4<T> &r, int n) {
    const T i0 = rcp(r.b);
    T a = r.a * i0, c = r.c * i0, d = r.d * i0;
    for (int st = 1; st < n; st *= 2) {
        const T am = __shfl_up(a, st), cm = __shfl_up(c, st), dm = __shfl_up(d, st);
        const T ap = __shfl_down(a, st), cp = __shfl_down(c, st), dp = __shfl_down(d, st);
        const T q = rcp(T(1) - a * cm - c * ap);
        d = (d - a * dm - c * dp) * q;
        a = -a * am * q;
        c = -c * cp * q;
    }
    return d;
}

// Interface solve of a row of more than one wave (NT chunks, one per thread),
// by the first wave: lane l takes the L = NT / 64 chunks L l .. L l + L - 1,
// eliminates their rows to one, and the 64 lane rows go through wave_pcr.
// I: 7 arrays of NT values in LDS (the chunk's last row a, b, c, d and the form
// G, H, M of its first unknown), chunk t at (t % L) * 64 + t / L, so that a
// lane's reads are free of bank conflicts; X receives the chunks' last
// unknowns in order.
template <int NT>
__device__ __forceinline__ int iface_pos(int t) {
    constexpr int L = NT / 64;
    return (t % L) * 64 + t / L;
}

template <int NT, typename T>
__device__ __forceinline__ void interface_solve(const T *I, T *X, int nt, int l) {
    constexpr int L = NT / 64;
    T a[L], b[L], c[L], d[L], g[L], h[L], m[L];
#pragma unroll
    for (int k = 0; k < L; ++k) {
        const int q = k * 64 + l;
        a[k] = I[q];
        b[k] = I[NT + q];
        c[k] = I[2 * NT + q];
        d[k] = I[3 * NT + q];
        g[k] = I[4 * NT + q];
        h[k] = I[5 * NT + q];
        m[k] = I[6 * NT + q];
    }
    const T gn = __shfl_down(g[0], 1), hn = __shfl_down(h[0], 1), mn = __shfl_down(m[0], 1);
#pragma unroll
    for (int k = 0; k < L; ++k) {
        const bool end = k == L - 1;
        const Row4<T> r = join(Row4<T>{a[k], b[k], c[k], d[k]}, end ? gn : g[(k + 1) % L], end ? hn : h[(k + 1) % L],
                               end ? mn : m[(k + 1) % L]);
        b[k] = r.b;
        c[k] = r.c;
        d[k] = r.d;
    }
    Row4<T> last;
    eliminate<L, false>(a, b, c, d, L, last);
    const T gs = __shfl_down(d[0], 1), hs = __shfl_down(a[0], 1), ms = __shfl_down(c[0], 1);
    const T xe = wave_pcr(join(last, gs, hs, ms), (nt + L - 1) / L);
    const T xp = __shfl_up(xe, 1);
#pragma unroll
    for (int k = 0; k < L - 1; ++k) X[L * l + k] = d[k] + a[k] * xp + c[k] * xe;
    X[L * l + L - 1] = xe;
}

// ---------------------------------------------------------------------------
// On-the-fly solve of one row: coefficients from the metrics, elimination,
// interface solve and back substitution per call.
// LDS: 4 nt (C+1) elements, or nt (C+1) + 8 NT (rows of more than one wave).
// ---------------------------------------------------------------------------
// Barrier of a row's NT threads.  ALONE: they are the workgroup; else the
// workgroup holds 256 / NT rows of the same NT, which pass the barriers
// together (waves that have ended do not count), a row of one wave by itself.
template <int NT, bool ALONE>
__device__ __forceinline__ void row_sync() {
    if (!ALONE && NT == 64) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

template <int C, int NT, bool SEG = false, int RG = 1, bool ALONE = true, typename T, typename GM>
__device__ __forceinline__ void xline_row(const RowCtx<T> &X, T *__restrict__ e, const T *__restrict__ f, const T *__restrict__ K,
                          const Grid &g, const GM &geo, int j, const T *far, int tid, T *lds) {
    constexpr int CP = C + 1;
    const int nt = X.nt;
    const int NT1 = nt * CP;
    T *Ld = lds, *Lb = lds + NT1, *La = lds + 2 * NT1, *Lc = lds + 3 * NT1;
    T ev[CP];
    row_pass<C, NT, SEG, RG>(X, e, f, K, g, geo, j, far, tid, Ld, La, Lb, Lc, ev);
    row_sync<NT, ALONE>();

    // each thread takes its chunk into registers
    T ca[CP], cb[CP], cc[CP], cd[CP];
    const int len = tid < nt ? C + (tid < X.rem ? 1 : 0) : 0;
#pragma unroll
    for (int k = 0; k < CP; ++k)
        if (k < len) {
            cd[k] = Ld[tid * CP + k];
            cb[k] = Lb[tid * CP + k];
            ca[k] = La[tid * CP + k];
            cc[k] = Lc[tid * CP + k];
        }
    row_sync<NT, ALONE>();

    // chunks past the row's end are identity rows
    Row4<T> last{0, 1, 0, 0};
    T g0 = 0, h0 = 0, m0 = 0;
    if (tid < nt) {
        eliminate<CP, true>(ca, cb, cc, cd, len, last);
        g0 = cd[0];
        h0 = ca[0];
        m0 = cc[0];
    }
    T xe, xp;
    if (NT == 64) {
        const T gn = __shfl_down(g0, 1), hn = __shfl_down(h0, 1), mn = __shfl_down(m0, 1);
        xe = wave_pcr(join(last, gn, hn, mn), nt);
        xp = __shfl_up(xe, 1);
    } else {
        // staged once through LDS, solved by wave 0, read back once: two barriers
        T *I = lds + NT1, *IX = I + 7 * NT;
        const int q = iface_pos<NT>(tid);
        I[q] = last.a;
        I[NT + q] = last.b;
        I[2 * NT + q] = last.c;
        I[3 * NT + q] = last.d;
        I[4 * NT + q] = g0;
        I[5 * NT + q] = h0;
        I[6 * NT + q] = m0;
        row_sync<NT, ALONE>();
        if (tid < 64) interface_solve<NT>(I, IX, nt, tid);
        row_sync<NT, ALONE>();
        xe = IX[tid];
        xp = tid ? IX[tid - 1] : T(0);
    }

    // back substitution, then the coalesced update
    if (tid < nt) {
        const bool longc = len == CP;
#pragma unroll
        for (int k = 0; k <= C - 1; ++k)
            if (k <= len - 2) lds[tid * CP + k] = cd[k] + ca[k] * xp + cc[k] * xe;
        lds[tid * CP + (longc ? C : C - 1)] = xe;
    }
    row_sync<NT, ALONE>();
    row_update_add<C, NT, SEG>(X, e, j, tid, lds, ev);
}

// Row `row` of e into `to` (XlFar).
template <int NT, typename T>
__device__ __forceinline__ void save_row(T *to, const T *e, const Grid &g, int row, int tid) {
    for (int i = tid; i < g.nx; i += NT) to[OFFX + i] = e[ix(g.pitch, i, row)];
}

// Rows j = row0 + slot*rowstep, one workgroup each; the workgroups past the
// rows save the far rows of the next launch.
//
// Rows longer than one workgroup's line solve are cut into segments of
// seglen cells, each solved as a line (row_pass).  A launch relaxes segments
// seg0, seg0 + segstep, .. of its rows, nsegl of them per row: launch slot s
// takes row slot s / nsegl, segment seg0 + segstep (s % nsegl).  With
// segstep 2 the even segments of a colour run in one launch and the odd ones
// in the next, so no workgroup reads a cell that another one of the same
// launch writes: a segment's residual reaches one cell beyond each end, into
// a segment of the other parity.  A whole row: seglen = nx, nsegl = 1.
template <int C, int NT, bool SEG, int RG = 3, typename T, typename GM>
__device__ __forceinline__ void xline_rows(T *__restrict__ e, const T *__restrict__ f, const T *__restrict__ K,
                                           const Grid &g, const GM &geo, int row0, int rowstep, int nrows, int nt,
                                           const XlFar<T> &far, int seglen, int seg0, int segstep, int nsegl) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    T *lds = reinterpret_cast<T *>(lds_bytes);
    RowCtx<T> X = row_ctx<T>(g, nt, C);
    int slot = launch_slot();
    if (slot >= nrows * nsegl) {
        const bool first = slot == nrows * nsegl && far.save[0] >= 0;
        save_row<NT>(first ? far.to[0] : far.to[1], e, g, first ? far.save[0] : far.save[1],
                     (int)threadIdx.x);
        return;
    }
    if (SEG) {
        X.nx = seglen;
        X.rem = seglen - nt * C;
        X.i0 = (seg0 + segstep * (slot % nsegl)) * seglen;
        slot /= nsegl;
    }
    const int j = row0 + slot * rowstep;
    xline_row<C, NT, SEG, RG>(X, e, f, K, g, geo, j, j == 0 ? far.lo : far.hi, (int)threadIdx.x, lds);
}

// Waves per SIMD of the fine-level kernel: the LDS of one workgroup at
// C = 8 (73.7 KB in FP64, 36.9 KB in FP32) allows two workgroups per CU in
// FP64 and four in FP32, and the register budget is set to match.
template <typename T>
constexpr int xl_waves() {
    return sizeof(T) == 8 ? 2 : 3;
}

// Rows up to 2055 cells: the fine levels are bandwidth-bound and need the
// other workgroups of the CU to cover the elimination and interface phases
// of each one.
template <int C, bool SEG, typename T, typename GM>
__global__ void __launch_bounds__(XL_THREADS) __attribute__((amdgpu_waves_per_eu(xl_waves<T>(), xl_waves<T>())))
k_xline(T *__restrict__ e, const T *__restrict__ f, const T *__restrict__ K, Grid g, GM geo, int row0, int rowstep,
        int nrows, int nt, XlFar<T> far, int seglen, int seg0, int segstep, int nsegl) {
    xline_rows<C, XL_THREADS, SEG>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl);
}

// Rows one 64-thread wave takes: at most 512 cells, or 128 in launches of few
// rows (XL_SHORT_FEW_MAX_NX).
template <int C, bool SEG, typename T, typename GM>
__global__ void __launch_bounds__(XL_SHORT) __attribute__((amdgpu_waves_per_eu(2)))
k_xline_short(T *__restrict__ e, const T *__restrict__ f, const T *__restrict__ K, Grid g, GM geo, int row0,
              int rowstep, int nrows, int nt, XlFar<T> far, int seglen, int seg0, int segstep, int nsegl) {
    xline_rows<C, XL_SHORT, SEG>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl);
}

// FP32 rows past 4111 cells, and rows of 1025 .. 2048 in launches of few rows.
template <int C, int NT, typename T, typename GM>
__global__ void __launch_bounds__(NT) k_xline_wide(T *__restrict__ e, const T *__restrict__ f,
                                                        const T *__restrict__ K, Grid g, GM geo, int row0,
                                                        int rowstep, int nrows, int nt, XlFar<T> far, int seglen,
                                                        int seg0, int segstep, int nsegl) {
    xline_rows<C, NT, false>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl);
}

// Longer rows (C = 16): one workgroup per CU in FP64 (139 KB of LDS), all registers.
template <int C, bool SEG, typename T, typename GM>
__global__ void __launch_bounds__(XL_THREADS) k_xline_long(T *__restrict__ e, const T *__restrict__ f,
                                                           const T *__restrict__ K, Grid g, GM geo, int row0,
                                                           int rowstep, int nrows, int nt, XlFar<T> far,
                                                           int seglen, int seg0, int segstep, int nsegl) {
    xline_rows<C, XL_THREADS, SEG>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl);
}

// Preconditioner residual restricted 1x2 in y, with the coarse correction
// cleared:  rc(i, J) = (r(i, 2J) + r(i, 2J+1)) / 2,  r = f - L e  (interior
// stencil from the metrics, ring cells from the table),  ec(i, J) = 0, with
// its far rows farc (XlFar: lo, then hi one pitch on).  Over the tile of
// 64 x 4 R N coarse cells from (i0, J0) by a workgroup of 256 threads: a wave
// takes N times R coarse rows of the interior columns, 2 R fine rows at a
// stretch (lap_rows), then the coarse cells of one side of the ring.  Bound by
// memory on the fine levels: 56 bytes a fine cell, 40 us on the finest level of
// 2048 x 2048 (235 MB).  Of one level a launch, R = 1, the mean over that
// grid's nine levels is 11.9 us (16.1 with the ring's cells among the others; R
// = 2 the same, and 5.6 against 4.8 on the levels of 512 x 512).  Batched, R = 2
// and N = 2, means over the levels and a whole solve with its finished problems
// masked: 7.4 us (13.3) for 24 odd FP64 problems, 19.1 (25.5) for 256 FP32 ones;
// R = 1 takes 7.8 and 19.9, R = 4 7.3 and 18.8 with 190 registers.  The finest
// level of all 256 takes 126 us.
template <int R, int N, typename T, typename G>
__device__ __forceinline__ void restrict_tile(T *rc, T *ec, T *farc, const T *e, const T *f, const T *K,
                                              const Grid &gf, const Grid &gc, const G &geo, int off, int i0, int J0) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, P = gf.pitch;
    const T idx = (T)(1.0 / gf.dx), idy = (T)(1.0 / gf.dy);
    const auto put = [&](int i, int J, T s) {
        const size_t c = ix(gc.pitch, i, J);
        rc[c] = s;
        ec[c] = 0;
        if (J < 2) farc[J * gc.pitch + OFFX + i] = 0;
    };
    int i = i0 + lane;
    if (i > 0 && i < gf.nx - 1) {
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const int J = J0 + (wave * N + n) * R, j = off + 2 * J;
            if (J + R <= gc.ny && j > 0 && j + 2 * R - 1 < gf.ny - 1) {
                const size_t c = ix(P, i, j);
                T v[2 * R], rhs[2 * R];
#pragma unroll
                for (int r = 0; r < 2 * R; ++r) rhs[r] = gptr(f)[c + r * P];
                lap_rows<2 * R>(e, geo, P, c, idx, idy, v);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    T s = 0;
                    s = s + T(0.5) * (rhs[2 * r] - v[2 * r]);
                    put(i, J + r, s + T(0.5) * (rhs[2 * r + 1] - v[2 * r + 1]));
                }
            } else if (R > 1) {
                for (int r = 0; r < R; ++r) {
                    const int jr = j + 2 * r;
                    if (J + r >= gc.ny || jr <= 0 || jr + 1 >= gf.ny - 1) continue;
                    const size_t c = ix(P, i, jr);
                    T v[2], s = 0;
                    lap_rows<2>(e, geo, P, c, idx, idy, v);
                    s = s + T(0.5) * (gptr(f)[c] - v[0]);
                    put(i, J + r, s + T(0.5) * (gptr(f)[c + P] - v[1]));
                }
            }
        }
    }
    // Coarse cells with a fine cell on the ring: rows 0 and gc.ny - 1 where
    // they cover the fine grid's first and last row, and the end columns.
    const bool lo = off == 0, hi = off + 2 * gc.ny == gf.ny;
    int J;
    if (wave < 2) {
        J = wave == 0 ? 0 : gc.ny - 1;
        i = i0 + lane;
        if (i >= gc.nx || J < J0 || J >= J0 + 4 * R * N || !(wave == 0 ? lo : hi)) return;
        if (wave == 1 && lo && J == 0) return;
    } else {
        J = J0 + lane;
        i = wave == 2 ? 0 : gc.nx - 1;
        if (lane >= 4 * R * N || J >= gc.ny || i < i0 || i >= i0 + 64) return;
        if ((lo && J == 0) || (hi && J == gc.ny - 1)) return;
    }
    const int nring = ring_count(gf.nx, gf.ny);
    T s = 0;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int j = off + 2 * J + b;
        const size_t c = ix(P, i, j);
        T v[1];
        if (i == 0 || i == gf.nx - 1 || j == 0 || j == gf.ny - 1) v[0] = ring_lap(gptr(e), gptr(K), nring, gf, i, j);
        else lap_rows<1>(e, geo, P, c, idx, idy, v);
        s = s + T(0.5) * (f[c] - v[0]);
    }
    put(i, J, s);
}

template <typename T, typename G>
__global__ void __launch_bounds__(256) k_residual_restrict_y(T *rc, T *ec, T *farc, const T *e, const T *f,
                                                             const T *K, Grid gf, Grid gc, G geo, int off) {
    restrict_tile<1, 1>(rc, ec, farc, e, f, K, gf, gc, geo, off, blockIdx.x * 64, blockIdx.y * 4);
}

// ---------------------------------------------------------------------------
// Batched forms: the workgroup's task or tile names the level (and through
// it the problem); workgroups of inactive problems return at once.
// ---------------------------------------------------------------------------
// The level's fields of the cycle's element type.
__device__ __forceinline__ void level_fields(const BLev *L, int sel, double *&e, const double *&f, const double *&K,
                                             double *&far, Geo &geo) {
    far = L->far;
    e = L->e[sel];
    f = L->f[sel];
    K = L->K;
    geo = L->geo;
}
__device__ __forceinline__ void level_fields(const BLev *L, int, float *&e, const float *&f, const float *&K,
                                             float *&far, GeoF &geo) {
    far = L->far32;
    e = L->e32;
    f = L->f32;
    K = L->K32;
    geo = L->geo32;
}

// Cells whose loads the batched kernels' row pass issues together: as many
// as fit without costing a wave per SIMD (FP32: 2 of the 3 cells of a chunk
// of 2, 3 of 5, 2 of 9; the C = 4 kernel keeps 4 waves with 119 VGPRs, the
// others their 87 and 154-159).  The batched mix's finest FP32 launch set
// went from 0.70 to 0.67 ms, bit-identical.  FP64: 2 cells for every chunk
// length (126, 152, 228 and 240 VGPRs: 4, 3, 2 and 2 waves, as with one).
template <int C, typename T>
constexpr int batch_rg() {
    return sizeof(T) == 8 ? 2 : (C == 4 ? 3 : 2);
}

template <int C, int NT, bool ALONE, typename T>
__device__ __forceinline__ void xline_task(const XlTask &t, const BLev *levs, const int *active, int sel, int k, int tid,
                                           T *lds) {
    const BLev *L = levs + t.lev;
    if (!active[L->prob] || (k >= 0 && k >= L->sweeps)) return;
    const Grid g = L->g;
    T *e, *far;
    const T *f, *K;
    typename std::conditional<sizeof(T) == 8, Geo, GeoF>::type geo;
    level_fields(L, sel, e, f, K, far, geo);
    if (t.save) {
        save_row<NT>(far + t.side * g.pitch, (const T *)e, g, t.row, tid);
        return;
    }
    const RowCtx<T> X = row_ctx<T>(g, L->nt, C);
    xline_row<C, NT, false, batch_rg<C, T>(), ALONE>(X, e, f, K, g, geo, t.row, t.row == 0 ? far : far + g.pitch, tid,
                                                     lds);
}

template <int C, int NT, typename T>
__device__ __forceinline__ void xline_alone(const XlTask *tasks, const BLev *levs, const int *active, int sel, int k) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    xline_task<C, NT, true, T>(tasks[launch_slot()], levs, active, sel, k, (int)threadIdx.x,
                               reinterpret_cast<T *>(lds_bytes));
}

template <int C, typename T>
__global__ void __launch_bounds__(XL_THREADS) __attribute__((amdgpu_waves_per_eu(xl_waves<T>(), xl_waves<T>())))
k_xline_batch(const XlTask *tasks, const BLev *levs, const int *active, int sel, int k) {
    xline_alone<C, XL_THREADS, T>(tasks, levs, active, sel, k);
}

template <int C, typename T>
__global__ void __launch_bounds__(XL_THREADS) k_xline_batch_long(const XlTask *tasks, const BLev *levs,
                                                                 const int *active, int sel, int k) {
    xline_alone<C, XL_THREADS, T>(tasks, levs, active, sel, k);
}

// Short rows (nx <= 512): one wave per row.
template <int C, typename T>
__global__ void __launch_bounds__(XL_SHORT) __attribute__((amdgpu_waves_per_eu(2)))
k_xline_batch_short(const XlTask *tasks, const BLev *levs, const int *active, int sel, int k) {
    xline_alone<C, XL_SHORT, T>(tasks, levs, active, sel, k);
}

// Rows of 513..1024 cells: two waves per row.
template <int C, typename T>
__global__ void __launch_bounds__(XL_MID) __attribute__((amdgpu_waves_per_eu(2)))
k_xline_batch_mid(const XlTask *tasks, const BLev *levs, const int *active, int sel, int k) {
    xline_alone<C, XL_MID, T>(tasks, levs, active, sel, k);
}

// Rows of every width in one launch: a workgroup of 256 threads takes 4, 2 or
// 1 rows of one class (XlBlock).  A phase's classes cover different problems,
// and on the coarse levels each class's launch would cost one row solve (or,
// side by side on several streams, a fork and a join) for a handful of rows.
template <int C, int NT, typename T>
__device__ __forceinline__ void xline_block(const XlBlock &b, const XlTask *tasks, const BLev *levs, const int *active,
                                            int sel, int k, T *lds) {
    const int sub = (int)threadIdx.x / NT, tid = (int)threadIdx.x % NT;
    if (sub >= b.count) return;
    xline_task<C, NT, NT == XL_THREADS, T>(tasks[b.first + sub], levs, active, sel, k, tid, lds + sub * row_lds_elems(C, NT));
}

// The classes of the batched line kernels.
#define MGP_XL_CLASSES(X)                                                                        \
    X(2, XL_SHORT) X(4, XL_SHORT) X(8, XL_SHORT) X(2, XL_MID) X(4, XL_MID) X(8, XL_MID)          \
    X(2, XL_THREADS) X(4, XL_THREADS) X(8, XL_THREADS) X(16, XL_THREADS)

template <typename T>
__global__ void __launch_bounds__(XL_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
k_xline_mixed(const XlBlock *blocks, const XlTask *tasks, const BLev *levs, const int *active, int sel, int k) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    T *lds = reinterpret_cast<T *>(lds_bytes);
    const XlBlock b = blocks[launch_slot()];
    switch (b.cls) {
#define MGP_XL_CASE(C, NT) \
    case xl_class(C, NT): xline_block<C, NT, T>(b, tasks, levs, active, sel, k, lds); break;
        MGP_XL_CLASSES(MGP_XL_CASE)
#undef MGP_XL_CASE
    }
}

template <typename T>
__global__ void __launch_bounds__(256) k_restrict_batch(const BTile *tiles, const BLev *levs, const int *active,
                                                        int sel) {
    const BTile t = tiles[blockIdx.x];
    const BLev *F = levs + t.item, *Cl = levs + t.item + 1;
    if (!active[F->prob]) return;
    T *fe, *ce, *cf, *far, *cfar;
    const T *ff, *K, *cff, *cK;
    typename std::conditional<sizeof(T) == 8, Geo, GeoF>::type geo, cgeo;
    level_fields(F, sel, fe, ff, K, far, geo);
    level_fields(Cl, 0, ce, cff, cK, cfar, cgeo);
    cf = const_cast<T *>(cff);
    restrict_tile<2, BT_ROWS / 8>(cf, ce, cfar, (const T *)fe, ff, K, F->g, Cl->g, geo, F->off, t.tx * 64, t.ty * BT_ROWS);
}

template <typename T>
__global__ void __launch_bounds__(256) k_prolong_batch(const BTile *tiles, const BLev *levs, const int *active,
                                                       int sel) {
    const BTile t = tiles[blockIdx.x];
    const BLev *F = levs + t.item, *Cl = levs + t.item + 1;
    if (!active[F->prob]) return;
    const int i = t.tx * 64 + (threadIdx.x & 63);
    const Grid gf = F->g, gc = Cl->g;
    if (i >= gf.nx) return;
    T *fe, *ce, *far, *cfar;
    const T *ff, *K, *cf, *cK;
    typename std::conditional<sizeof(T) == 8, Geo, GeoF>::type geo, cgeo;
    level_fields(F, sel, fe, ff, K, far, geo);
    level_fields(Cl, 0, ce, cf, cK, cfar, cgeo);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int j = t.ty * BT_ROWS + (threadIdx.x >> 6) + 4 * r;
        if (j < gf.ny) prolong_y_cell(fe, (const T *)ce, far, gf, gc, (T)F->slo, (T)F->shi, i, j, F->off);
    }
}

// Chunk length for a row of nx cells: the smallest C in {2, 4, 8, 16} with
// floor(nx / C) <= 256 chunks.  nx >= C*C then holds, so the remainder is
// spread one cell per chunk (chunks of C or C+1 cells).
int xline_chunk(int nx, int nt_max = XL_THREADS) {
    for (int C = 2; C <= 16; C *= 2)
        if (nx / C <= nt_max) return C;
    return 0;
}

}  // namespace

int ring_table_elems(const Grid &g) { return RING_PLANES * ring_count(g.nx, g.ny); }

void launch_ring_coef(hipStream_t s, double *K, const Grid &g, const Geo &geo, const Bc &bc) {
    const int n = ring_table_elems(g);
    k_ring_coef<<<(n + 255) / 256, 256, 0, s>>>(K, g, geo, bc);
}

size_t xline_lds_bytes(int nx, size_t elem) { return xline_lds_bytes_for(nx, xline_chunk(nx), elem, XL_THREADS); }

size_t xline_lds_bytes_for(int nx, int C, size_t elem, int threads) {
    if (C == 0) return (size_t)-1;
    const size_t nt = (size_t)(nx / C);
    // chunk staging (4 arrays), or one chunk array plus the interface rows and unknowns
    const size_t tr = 4 * nt * (C + 1), iface = nt * (C + 1) + (threads > 64 ? 8 * (size_t)threads : 0);
    return (tr > iface ? tr : iface) * elem;
}

bool xline_batch_class(int C, int threads) {
    switch (xl_class(C, threads)) {
#define MGP_XL_CASE(c, nt) case xl_class(c, nt):
        MGP_XL_CLASSES(MGP_XL_CASE)
#undef MGP_XL_CASE
        return true;
    default: return false;
    }
}

int xline_block_rows(int threads) { return XL_THREADS / threads; }

size_t xline_block_lds(int C, int threads, size_t elem) {
    return (size_t)xline_block_rows(threads) * row_lds_elems(C, threads) * elem;
}

bool xline_supported(int nx) { return xline_segments(nx, sizeof(double)) != 0; }

bool xline_single_line(int nx) { return nx >= 4 && xline_chunk(nx) != 0; }

bool xline_whole(int nx, size_t elem) { return xline_segments(nx, elem) == 1; }

int xline_segments(int nx, size_t elem) {
    if (nx < 4) return 0;
    if (xline_chunk(nx) != 0) return 1;
    if (elem == sizeof(float) && xline_chunk(nx, XL_WIDE) == 16) return 1;
    for (int n = 2; n <= 64; n *= 2)
        if (nx % n == 0 && nx / n >= 4 && xline_chunk(nx / n) != 0) return n;
    return 0;
}

int xline_batch_chunk(int nx, int threads, size_t elem) {
    if (nx < 4 || (threads != XL_SHORT && threads != XL_MID && threads != XL_THREADS)) return 0;
    const int C = xline_chunk(nx, threads);
    if (C == 0 || (C == 16 && threads != XL_THREADS)) return 0;
    return xline_lds_bytes_for(nx, C, elem, threads) <= 160 * 1024 ? C : 0;
}

void xline_batch_shape(int nx, int &C, int &threads) {
    threads = nx <= XL_SHORT_MAX_NX ? XL_SHORT : (nx <= XL_MID_MAX_NX ? XL_MID : XL_THREADS);
    C = xline_chunk(nx, threads);
}

template <typename T, typename G>
static void residual_restrict_y(hipStream_t s, T *rc, T *ec, T *farc, const T *e, const T *f, const T *K,
                                const Grid &gf, const Grid &gc, const G &geo, int off) {
    const dim3 grid((unsigned)((gc.nx + 63) / 64), (unsigned)((gc.ny + 3) / 4));
    k_residual_restrict_y<<<grid, 256, 0, s>>>(rc, ec, farc, e, f, K, gf, gc, geo, off);
}

void launch_residual_restrict_y(hipStream_t s, double *rc, double *ec, double *farc, const double *e, const double *f,
                                const double *K, const Grid &gf, const Grid &gc, const Geo &geo, int off) {
    residual_restrict_y(s, rc, ec, farc, e, f, K, gf, gc, geo, off);
}

void launch_residual_restrict_y(hipStream_t s, float *rc, float *ec, float *farc, const float *e, const float *f, const float *K,
                                const Grid &gf, const Grid &gc, const GeoF &geo, int off) {
    residual_restrict_y(s, rc, ec, farc, e, f, K, gf, gc, geo, off);
}

// One launch of the line kernel for rows (SEG = false) or segments of seglen cells.
template <bool SEG, typename T, typename G>
static void xline_launch(hipStream_t s, T *e, const T *f, const T *K, const Grid &g, const G &geo, int row0,
                         int rowstep, int nrows, const XlFar<T> &far, int seglen, int seg0, int segstep, int nsegl,
                         unsigned grid) {
    const bool few = grid <= XL_FEW_ROWS;
    if (sizeof(T) == 4 && !SEG && (xline_chunk(seglen) == 0 || (few && seglen > XL_LONG_MIN_NX && seglen <= XL_LONG_MAX_NX))) {
        if constexpr (sizeof(T) == 4 && !SEG) {
            // few rows: the widest form; rows past 4111 cells always (xline_segments)
            if (xline_chunk(seglen) != 0) {
                const size_t lds = xline_lds_bytes_for(seglen, 4, sizeof(T), XL_WIDE);
                k_xline_wide<4, XL_WIDE><<<grid, XL_WIDE, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, seglen / 4, far, seglen, seg0, segstep, nsegl);
            } else if (few && xline_chunk(seglen, XL_WIDEST) == 8) {
                const size_t lds = xline_lds_bytes_for(seglen, 8, sizeof(T), XL_WIDEST);
                k_xline_wide<8, XL_WIDEST><<<grid, XL_WIDEST, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, seglen / 8, far, seglen, seg0, segstep, nsegl);
            } else {
                const size_t lds = xline_lds_bytes_for(seglen, 16, sizeof(T), XL_WIDE);
                k_xline_wide<16, XL_WIDE><<<grid, XL_WIDE, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, seglen / 16, far, seglen, seg0, segstep, nsegl);
            }
        }
    } else if (seglen <= (few ? XL_SHORT_FEW_MAX_NX : XL_SHORT_MAX_NX)) {
        const int C = xline_chunk(seglen, XL_SHORT), nt = seglen / C;
        const size_t lds = xline_lds_bytes_for(seglen, C, sizeof(T), XL_SHORT);
        switch (C) {
            case 2: k_xline_short<2, SEG><<<grid, XL_SHORT, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl); break;
            case 4: k_xline_short<4, SEG><<<grid, XL_SHORT, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl); break;
            default: k_xline_short<8, SEG><<<grid, XL_SHORT, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl); break;
        }
    } else {
        const int C = xline_chunk(seglen);
        const size_t lds = xline_lds_bytes(seglen, sizeof(T));
        if (lds > 160 * 1024) {
            g_last_error = "k_xline: row length not supported";
            throw Failure(MGP_ERR_UNSUPPORTED);
        }
        const int nt = seglen / C;
        switch (C) {
            case 2: k_xline<2, SEG><<<grid, XL_THREADS, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl); break;
            case 4: k_xline<4, SEG><<<grid, XL_THREADS, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl); break;
            case 8: k_xline<8, SEG><<<grid, XL_THREADS, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl); break;
            default: k_xline_long<16, SEG><<<grid, XL_THREADS, lds, s>>>(e, f, K, g, geo, row0, rowstep, nrows, nt, far, seglen, seg0, segstep, nsegl); break;
        }
    }
}

template <typename T, typename G>
static void xline(hipStream_t s, T *e, const T *f, const T *K, const Grid &g, const G &geo, int row0, int rowstep,
                  int nrows, const XlFar<T> &far, int part = -1) {
    if (nrows <= 0) return;
    const int nseg = xline_segments(g.nx, sizeof(T));
    if (nseg == 0) {
        g_last_error = "k_xline: row length not supported";
        throw Failure(MGP_ERR_UNSUPPORTED);
    }
    const int seglen = g.nx / nseg;
    // whole rows in one launch; segmented rows: the even segments, then the odd ones
    const int nlaunch = nseg == 1 ? 1 : 2, segstep = nseg == 1 ? 1 : 2, nsegl = nseg == 1 ? 1 : nseg / 2;
    const unsigned grid = (unsigned)(nrows * nsegl + (far.save[0] >= 0) + (far.save[1] >= 0));
    for (int seg0 = 0; seg0 < nlaunch; ++seg0) {
        if (part >= 0 && seg0 != part) continue;
        if (nseg > 1) xline_launch<true>(s, e, f, K, g, geo, row0, rowstep, nrows, far, seglen, seg0, segstep, nsegl, grid);
        else xline_launch<false>(s, e, f, K, g, geo, row0, rowstep, nrows, far, seglen, seg0, segstep, nsegl, grid);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) {
            g_last_error = std::string("k_xline launch: ") + hipGetErrorString(err);
            throw Failure(MGP_ERR_HIP);
        }
    }
}

void launch_xline(hipStream_t s, double *e, const double *f, const double *K, const Grid &g, const Geo &geo,
                  int row0, int rowstep, int nrows, const XlFar<double> &far, int part) {
    xline(s, e, f, K, g, geo, row0, rowstep, nrows, far, part);
}

template <typename T>
static void xline_batch(hipStream_t s, const XlTask *tasks, int ntasks, const BLev *levs, const int *active, int sel,
                        int C, int threads, size_t lds, int k) {
    if (threads == XL_SHORT) {
        switch (C) {
            case 2: k_xline_batch_short<2, T><<<ntasks, XL_SHORT, lds, s>>>(tasks, levs, active, sel, k); break;
            case 4: k_xline_batch_short<4, T><<<ntasks, XL_SHORT, lds, s>>>(tasks, levs, active, sel, k); break;
            case 8: k_xline_batch_short<8, T><<<ntasks, XL_SHORT, lds, s>>>(tasks, levs, active, sel, k); break;
            default:
                g_last_error = "k_xline_batch_short: chunk length must be 2, 4 or 8";
                throw Failure(MGP_ERR_ARG);
        }
    } else if (threads == XL_MID) {
        switch (C) {
            case 2: k_xline_batch_mid<2, T><<<ntasks, XL_MID, lds, s>>>(tasks, levs, active, sel, k); break;
            case 4: k_xline_batch_mid<4, T><<<ntasks, XL_MID, lds, s>>>(tasks, levs, active, sel, k); break;
            case 8: k_xline_batch_mid<8, T><<<ntasks, XL_MID, lds, s>>>(tasks, levs, active, sel, k); break;
            default:
                g_last_error = "k_xline_batch_mid: chunk length must be 2, 4 or 8";
                throw Failure(MGP_ERR_ARG);
        }
    } else switch (C) {
        case 2: k_xline_batch<2, T><<<ntasks, XL_THREADS, lds, s>>>(tasks, levs, active, sel, k); break;
        case 4: k_xline_batch<4, T><<<ntasks, XL_THREADS, lds, s>>>(tasks, levs, active, sel, k); break;
        case 8: k_xline_batch<8, T><<<ntasks, XL_THREADS, lds, s>>>(tasks, levs, active, sel, k); break;
        case 16: k_xline_batch_long<16, T><<<ntasks, XL_THREADS, lds, s>>>(tasks, levs, active, sel, k); break;
        default:
            g_last_error = "k_xline_batch: chunk length must be 2, 4, 8 or 16";
            throw Failure(MGP_ERR_ARG);
    }
}

void launch_xline_batch(hipStream_t s, const XlTask *tasks, int ntasks, const BLev *levs, const int *active, int sel,
                        int C, int threads, size_t lds, int k, bool fp32) {
    if (ntasks <= 0) return;
    if (fp32) xline_batch<float>(s, tasks, ntasks, levs, active, sel, C, threads, lds, k);
    else xline_batch<double>(s, tasks, ntasks, levs, active, sel, C, threads, lds, k);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        g_last_error = std::string("k_xline_batch launch: ") + hipGetErrorString(err);
        throw Failure(MGP_ERR_HIP);
    }
}

void launch_xline(hipStream_t s, float *e, const float *f, const float *K, const Grid &g, const GeoF &geo, int row0,
                  int rowstep, int nrows, const XlFar<float> &far) {
    xline(s, e, f, K, g, geo, row0, rowstep, nrows, far);
}

void launch_xline_mixed(hipStream_t s, const XlBlock *blocks, int nblocks, const XlTask *tasks, const BLev *levs,
                        const int *active, int sel, size_t lds, int k, bool fp32) {
    if (nblocks <= 0) return;
    if (fp32) k_xline_mixed<float><<<nblocks, XL_THREADS, lds, s>>>(blocks, tasks, levs, active, sel, k);
    else k_xline_mixed<double><<<nblocks, XL_THREADS, lds, s>>>(blocks, tasks, levs, active, sel, k);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        g_last_error = std::string("k_xline_mixed launch: ") + hipGetErrorString(err);
        throw Failure(MGP_ERR_HIP);
    }
}

void launch_restrict_batch(hipStream_t s, const BTile *tiles, int ntiles, const BLev *levs, const int *active,
                           int sel, bool fp32) {
    if (ntiles <= 0) return;
    if (fp32) k_restrict_batch<float><<<ntiles, 256, 0, s>>>(tiles, levs, active, sel);
    else k_restrict_batch<double><<<ntiles, 256, 0, s>>>(tiles, levs, active, sel);
}

void launch_prolong_batch(hipStream_t s, const BTile *tiles, int ntiles, const BLev *levs, const int *active,
                          int sel, bool fp32) {
    if (ntiles <= 0) return;
    if (fp32) k_prolong_batch<float><<<ntiles, 256, 0, s>>>(tiles, levs, active, sel);
    else k_prolong_batch<double><<<ntiles, 256, 0, s>>>(tiles, levs, active, sel);
}

}  // namespace mgp
