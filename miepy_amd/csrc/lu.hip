// Dense LU with partial pivoting: the `exact` method of solve_linear_system.
//
// Replaces interaction_matrix.partialPivLu().solve(p_src)
// (cpp/src/interactions.cpp:356-357, and :338-339 on the preconditioned path).
// Right-looking blocked LU with panels of kNb = 32 columns:
//
//   for each panel [k0, k0 + 32):
//     the panel in strips of 16 to 4 columns: one workgroup holds a strip's
//       rows in registers and factors it column by column (pivot p = the
//       first row i >= j of largest |A[i][j]|, partial pivoting as Eigen's
//       PartialPivLU; the modulus is compared squared), then swaps and solves
//       the strip's rows of the panel columns to its right; a second launch
//       updates the rows below in those columns;
//     the panel's 32 row swaps applied to all other columns at once, and for
//       the columns to the right U12 = L11^-1 A12 in the same pass;
//     A22 -= L21 U12 on the FP64 matrix cores (v_mfma_f64_16x16x4f64),
//     64 x 64 complex tiles, K = 32 complex = 64 real positions.
//
// L (unit diagonal) and U overwrite A; the row swaps, in order, become one
// permutation at the end of the factorization.  The solve gathers b through
// that permutation and runs blocked forward and back substitution (a
// one-wave solve of each 64 x 64 diagonal block, then a block-column
// update of the rows below / above).  Everything is FP64.
//
// A panel column costs 2-4 us in a strip (33 us per 8 columns of 2500 rows,
// 38 us per 16 columns of 500), where two launches per column took 11 us.
// exact solve of n = 2910: 38.9 ms with those, 17.3 ms now.

#include <algorithm>
#include <climits>
#include <cstdio>
#include <vector>

#include "common.hpp"


namespace {

constexpr int kNb = 32;         // panel width = K of the trailing update
constexpr int kT = 256;         // threads per workgroup
constexpr int kMaxParts = 240;  // workgroups of the pivot searches (partial maxima)
constexpr int kTile = 64;       // trailing-update tile (complex rows and columns)

size_t al256(size_t b) { return (b + 255) & ~size_t(255); }

struct LuWs {
    int* piv;     // [n] pivot row of each column
    int* perm;    // [n] row permutation: (P b)[k] = b[perm[k]]
    double* pval; // [kMaxParts] partial maxima of |A[i][j]|^2
    int* pidx;    // [kMaxParts] their rows
    int* info;    // 0, or 1 + the first column without a nonzero pivot
};

size_t ws_bytes(int n) {
    return 2 * al256(sizeof(int) * (size_t)n) + al256(sizeof(double) * kMaxParts) + al256(sizeof(int) * kMaxParts) +
           256;
}

LuWs ws_view(void* w, int n) {
    char* p = (char*)w;
    LuWs v;
    v.piv = (int*)p; p += al256(sizeof(int) * (size_t)n);
    v.perm = (int*)p; p += al256(sizeof(int) * (size_t)n);
    v.pval = (double*)p; p += al256(sizeof(double) * kMaxParts);
    v.pidx = (int*)p; p += al256(sizeof(int) * kMaxParts);
    v.info = (int*)p;
    return v;
}

// (value, row) with the larger value winning and the lower row on ties: the
// first maximum, as a sequential scan finds it.
__device__ inline void better(double& v, int& i, double v2, int i2) {
    if (v2 > v || (v2 == v && i2 < i)) {
        v = v2;
        i = i2;
    }
}

// Block-wide reduction of (v, i) to thread 0 (all threads must call).
__device__ inline void block_best(double& v, int& i) {
    __shared__ double sv[kT / 64];
    __shared__ int si[kT / 64];
    for (int off = 32; off > 0; off >>= 1) {
        const double v2 = __shfl_xor(v, off);
        const int i2 = __shfl_xor(i, off);
        better(v, i, v2, i2);
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) {
        sv[w] = v;
        si[w] = i;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 1; k < kT / 64; k++) better(v, i, sv[k], si[k]);
    __syncthreads();
}

__global__ __launch_bounds__(kT) void k_lu_add_identity(double2* __restrict__ A, int n) {
    const int i = blockIdx.x * kT + threadIdx.x;
    if (i < n) A[(size_t)i * n + i].x += 1.0;
}

// Partial maxima of |A[i][j]|^2 over rows i >= j (the first column of a panel).
__global__ __launch_bounds__(kT) void k_lu_pivot_search(const double2* __restrict__ A, int n, int j,
                                                        double* __restrict__ pval, int* __restrict__ pidx) {
    double v = -1.0;
    int idx = INT_MAX;
    for (int i = j + blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) {
        const double2 a = A[(size_t)i * n + j];
        better(v, idx, a.x * a.x + a.y * a.y, i);
    }
    block_best(v, idx);
    if (threadIdx.x == 0) {
        pval[blockIdx.x] = v;
        pidx[blockIdx.x] = idx;
    }
}

// Reduce the partial maxima to column j's pivot row p (every workgroup
// redundantly), record it, and swap the whole rows j and p.  A column
// without a nonzero (finite) pivot records info and keeps p = j.
__global__ __launch_bounds__(kT) void k_lu_swap(double2* __restrict__ A, int n, int j, const double* __restrict__ pval,
                                                const int* __restrict__ pidx, int nparts, int* __restrict__ piv,
                                                int* __restrict__ info) {
    __shared__ int sp;
    double v = -1.0;
    int idx = INT_MAX;
    if ((int)threadIdx.x < nparts) {
        v = pval[threadIdx.x];
        idx = pidx[threadIdx.x];
    }
    block_best(v, idx);
    if (threadIdx.x == 0) {
        const bool ok = v > 0.0 && v <= 1.7976931348623157e308 && idx < n;
        sp = ok ? idx : j;
        if (blockIdx.x == 0) {
            piv[j] = sp;
            if (!ok && *info == 0) *info = j + 1;
        }
    }
    __syncthreads();
    const int p = sp;
    if (p == j) return;
    double2* rj = A + (size_t)j * n;
    double2* rp = A + (size_t)p * n;
    for (int c = blockIdx.x * kT + threadIdx.x; c < n; c += gridDim.x * kT) {
        const double2 t = rj[c];
        rj[c] = rp[c];
        rp[c] = t;
    }
}

// Column j of the panel [.., k_end): A[i][j] /= A[j][j] for i > j, then
// A[i][c] -= A[i][j] A[j][c] for the panel columns j < c < k_end, and the
// partial maxima of the updated column j + 1 (when it is in the panel).
__global__ __launch_bounds__(kT) void k_lu_panel(double2* __restrict__ A, int n, int j, int k_end,
                                                 double* __restrict__ pval, int* __restrict__ pidx) {
    __shared__ double2 urow[kNb];
    __shared__ double2 dpiv;
    const int w = k_end - j - 1;  // 0 .. kNb - 1
    if ((int)threadIdx.x < w) urow[threadIdx.x] = A[(size_t)j * n + j + 1 + threadIdx.x];
    if (threadIdx.x == 0) dpiv = A[(size_t)j * n + j];
    __syncthreads();
    const double2 d = dpiv;
    double v = -1.0;
    int idx = INT_MAX;
    for (int i = j + 1 + blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) {
        double2* row = A + (size_t)i * n;
        const double2 l = cdiv(row[j], d);
        row[j] = l;
        for (int c = 0; c < w; c++) row[j + 1 + c] = csub(row[j + 1 + c], cmul(l, urow[c]));
        if (w > 0) {
            const double2 a = row[j + 1];
            better(v, idx, a.x * a.x + a.y * a.y, i);
        }
    }
    if (w > 0) {
        block_best(v, idx);
        if (threadIdx.x == 0) {
            pval[blockIdx.x] = v;
            pidx[blockIdx.x] = idx;
        }
    }
}

// by value: a conditional on two array entries would select their addresses and put the arrays into scratch
__device__ __forceinline__ double2 csel(bool c, double2 x, double2 y) {
    return make_double2(c ? x.x : y.x, c ? x.y : y.y);
}

// a / b from inv, a reciprocal of b good to a few units in the last place: the
// product alone carries the reciprocal's rounding into every entry, one step on
// the remainder a - q b takes it out (diagonally dominant n = 20: error of the
// solution 2.14e-16 and 2.04e-16, 2.02e-16 with a division per entry).
__device__ __forceinline__ double2 cquot(double2 a, double2 b, double2 inv) {
    double2 q = cmul(a, inv);
    const double rx = fma(q.y, b.y, fma(-q.x, b.x, a.x)), ry = fma(-q.y, b.x, fma(-q.x, b.y, a.y));
    q.x = fma(-ry, inv.y, fma(rx, inv.x, q.x));
    q.y = fma(ry, inv.x, fma(rx, inv.y, q.y));
    return q;
}

constexpr int kStripT = 512;  // threads of the strip kernel: 256 registers each

// Rows a thread holds at a strip width (4 registers per entry, about 200 in all).
constexpr int strip_rows(int w) { return w == 16 ? 2 : w == 8 ? 5 : 10; }

// Widest strip whose rows fit the registers of one workgroup; 0: none (the
// column-by-column path).  Wider strips save launches and in-panel updates.
int strip_width(int rows) {
    for (int w = 16; w >= 4; w /= 2)
        if (rows <= kStripT * strip_rows(w)) return w;
    return 0;
}

// Largest unsigned value of the wave's lanes, or of its first 8 lanes
// (valid in every lane): row shifts and row broadcasts, one instruction per
// step where a cross-lane permute takes over 100 cycles.
template <int CTRL, int MASK>
__device__ __forceinline__ unsigned max_step(unsigned v) {
    return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, MASK, 0xf, false));
}
__device__ __forceinline__ unsigned wave_max(unsigned v) {
    v = max_step<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
    v = max_step<0x112, 0xf>(v);
    v = max_step<0x114, 0xf>(v);
    v = max_step<0x118, 0xf>(v);
    v = max_step<0x142, 0xa>(v);  // row_bcast:15, 31
    v = max_step<0x143, 0xc>(v);
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ unsigned first8_max(unsigned v) {
    v = max_step<0x111, 0xf>(v);
    v = max_step<0x112, 0xf>(v);
    v = max_step<0x114, 0xf>(v);
    return (unsigned)__builtin_amdgcn_readlane((int)v, 7);
}

// The lane (of the wave, or of its first 8) whose modulus is largest, the
// lowest row among equals: non-negative doubles order as their bits, so the
// high words, the low words and the complemented rows are reduced in turn.
// Returns the winner's row; hi and lo become its modulus.
template <bool FIRST8>
__device__ __forceinline__ int best_row(unsigned& hi, unsigned& lo, int row) {
    auto red = [](unsigned v) { return FIRST8 ? first8_max(v) : wave_max(v); };
    const unsigned h = red(hi);
    const unsigned l = red(hi == h ? lo : 0u);
    const unsigned r = red(hi == h && lo == l ? ~(unsigned)row : 0u);
    hi = h;
    lo = l;
    return (int)~r;
}

// Columns [j0, j0 + W) of the panel that ends at k_end, rows [j0, n): thread
// t holds the rows j0 + t + 512 i.  Per column every wave finds its first row
// of largest modulus and puts that row into LDS (the wave that holds row j
// puts that one there too); after one barrier every wave picks the best of the
// 8, and each thread exchanges, scales by 1 / pivot and updates its rows in
// registers.  The column at hand is always a[.][0]: the entries rotate by one
// after each column, so that one loop body serves all of them.  One workgroup:
// the columns are a serial chain of reductions, which workgroups on several
// CUs would have to carry through memory.  At the end the strip's swaps are
// applied to the panel's other columns, and its unit triangle to the rows
// [j0, j0 + W) of those to the right.
template <int W, int RPT>
__global__ __launch_bounds__(kStripT) void k_lu_strip(double2* __restrict__ A, int n, int k0, int j0,
                                                      int k_end, int* __restrict__ piv, int* __restrict__ info) {
    constexpr int NW = kStripT / 64;
    __shared__ unsigned shi[2][NW], slo[2][NW];
    __shared__ int srow[2][NW];
    __shared__ double2 cand[2][NW][W], jrow[2][W];
    __shared__ double2 L[W][W + 1];
    __shared__ int sp[W];
    __shared__ double2 stage[kStripT * (W + 1)];  // 512 rows between the runs read from A and a thread's own
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    double2 a[RPT][W];
    // A is read and written in runs of a strip's row (W consecutive lanes); 64 rows at a time, a row per
    // lane, cost 64 lines per access and half of the kernel's time.
    const int rr = t / W, rc = t % W;  // access k covers row 512 i + 512 / W k + rr, column rc
    constexpr int RK = kStripT / W;
#pragma unroll
    for (int i = 0; i < RPT; i++)
#pragma unroll
        for (int k = 0; k < W; k++) {
            const int r = j0 + kStripT * i + RK * k + rr;
            a[i][k] = r < n ? A[(size_t)r * n + j0 + rc] : make_double2(0.0, 0.0);
        }
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < W; k++) stage[(RK * k + rr) * (W + 1) + rc] = a[i][k];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < W; c++) a[i][c] = stage[t * (W + 1) + c];
    }
#pragma unroll 1
    for (int jj = 0; jj < W; jj++) {
        const int j = j0 + jj, buf = jj & 1;  // a[.][c] is column (jj + c) % W of the strip
        double v = 0.0;  // a NaN is never a pivot
        int idx = INT_MAX;
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            const int r = j0 + t + kStripT * i;
            const double m2 = a[i][0].x * a[i][0].x + a[i][0].y * a[i][0].y;
            if (r >= j && r < n && m2 > v) {
                v = m2;
                idx = r;
            }
        }
        unsigned hi = (unsigned)__double2hiint(v), lo = (unsigned)__double2loint(v);
        const int wbest = best_row<false>(hi, lo, idx);
        if (lane == 0) {
            shi[buf][wv] = hi;
            slo[buf][wv] = lo;
            srow[buf][wv] = wbest;
        }
        if (idx == wbest && idx != INT_MAX) {
#pragma unroll
            for (int i = 0; i < RPT; i++)
                if (j0 + t + kStripT * i == idx)
#pragma unroll
                    for (int c = 0; c < W; c++) cand[buf][wv][c] = a[i][c];
        }
        if (t == jj) {
#pragma unroll
            for (int c = 0; c < W; c++) jrow[buf][c] = a[0][c];
        }
        __syncthreads();
        const int k = lane & (NW - 1);
        unsigned bh = shi[buf][k], bl = slo[buf][k];
        const int brow = srow[buf][k];
        const int best = best_row<true>(bh, bl, brow);
        const double pv = __hiloint2double((int)bh, (int)bl);  // |pivot|^2
        const bool ok = pv > 0.0 && pv <= 1.7976931348623157e308;
        const int p = ok ? best : j;  // a column without a nonzero (finite) pivot keeps p = j
        const double2* prow = ok ? cand[buf][((p - j0) % kStripT) / 64] : jrow[buf];
        if (t == jj) {
            sp[jj] = p;
            piv[j] = p;
            if (!ok && *info == 0) *info = j + 1;
        }
        const double2 pj = prow[0];
        // 1 / pivot from one reciprocal of |pivot|^2 where that is far from the ends of the range
        double2 inv;
        if (pv > 1e-280 && pv < 1e280) {
            double rc = __builtin_amdgcn_rcp(pv);
            rc = fma(fma(-pv, rc, 1.0), rc, rc);
            rc = fma(fma(-pv, rc, 1.0), rc, rc);
            inv = make_double2(pj.x * rc, -pj.y * rc);
        } else {
            inv = cdiv(make_double2(1.0, 0.0), pj);
        }
        if (p != j) {
#pragma unroll
            for (int i = 0; i < RPT; i++)
                if (j0 + t + kStripT * i == p)
#pragma unroll
                    for (int c = 0; c < W; c++) a[i][c] = jrow[buf][c];
            if (t == jj) {
#pragma unroll
                for (int c = 0; c < W; c++) a[0][c] = prow[c];
            }
        }
        double2 l[RPT], done[RPT];
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            // More rows per thread: the remainder step would cost 1.3 % of a solve (n = 2910), whose error the
            // longer sums decide (3.7e-15 and 3.8e-15 without and with it).
            l[i] = W == 16 ? cquot(a[i][0], pj, inv) : cmul(a[i][0], inv);
            done[i] = csel(i > 0 || t > jj, l[i], a[i][0]);  // rows up to j are final
        }
#pragma unroll
        for (int c = 1; c < W; c++) {
            if (c < W - jj) {  // not factored yet
                const double2 u = prow[c];
#pragma unroll
                for (int i = 0; i < RPT; i++) {
                    const double2 x = csub(a[i][c], cmul(l[i], u));
                    a[i][c] = csel(i > 0 || t > jj, x, a[i][c]);
                }
            }
#pragma unroll
            for (int i = 0; i < RPT; i++) a[i][c - 1] = a[i][c];
        }
#pragma unroll
        for (int i = 0; i < RPT; i++) a[i][W - 1] = done[i];
    }
    if (t < W) {
#pragma unroll
        for (int c = 0; c < W; c++) L[t][c] = a[0][c];
    }
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        __syncthreads();
#pragma unroll
        for (int c = 0; c < W; c++) stage[t * (W + 1) + c] = a[i][c];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < W; k++) {
            const int r = j0 + kStripT * i + RK * k + rr;
            if (r < n) A[(size_t)r * n + j0 + rc] = stage[(RK * k + rr) * (W + 1) + rc];
        }
    }
    const int left = j0 - k0, rest = k_end - k0 - W;  // the panel's columns left of the strip, and both sides
    // their rows: [0, W) the strip's, [W, 2 W) the pivots'
    auto top = (double2(*)[kNb - W + 1])stage;
    auto col = [&](int c) { return c < left ? k0 + c : c + k0 + W; };
    __syncthreads();  // sp of the last column is set, stage is read
    for (int u = t; u < 2 * W * rest; u += kStripT) {
        const int q = u / rest, c = u - q * rest;
        top[q][c] = A[(size_t)(q < W ? j0 + q : sp[q - W]) * n + col(c)];
    }
    __syncthreads();
    // one thread per column: the swaps in order (a pivot row inside the strip is
    // its top row, a repeated one its first copy), then the unit triangle
    if (t < rest) {
        int slot[W];
#pragma unroll
        for (int k = 0; k < W; k++) {
            int s = sp[k] < j0 + W ? sp[k] - j0 : W + k;
#pragma unroll
            for (int e = W - 1; e >= 0; e--)
                if (e < k && s >= W && sp[e] == sp[k]) s = W + e;
            slot[k] = s;
            const double2 x = top[k][t], y = top[s][t];
            top[k][t] = y;
            top[s][t] = x;
        }
        if (t >= left) {
#pragma unroll
            for (int r = 1; r < W; r++) {
                double2 x = top[r][t];
#pragma unroll
                for (int q = 0; q < r; q++) x = csub(x, cmul(L[r][q], top[q][t]));
                top[r][t] = x;
            }
        }
#pragma unroll
        for (int k = 0; k < W; k++) {
            A[(size_t)(j0 + k) * n + col(t)] = top[k][t];
            if (slot[k] >= W) A[(size_t)sp[k] * n + col(t)] = top[slot[k]][t];
        }
    }
}

// A[i][c] -= sum_q L[i][j0 + q] U[j0 + q][c] for the rows i >= j0 + W and the
// panel columns [j0 + W, k_end): four threads per row, each every fourth column.
template <int W>
__global__ __launch_bounds__(kT) void k_lu_strip_update(double2* __restrict__ A, int n, int j0, int k_end) {
    __shared__ double2 U[W][kNb];
    const int c0 = j0 + W, rest = k_end - c0;
    for (int u = threadIdx.x; u < W * rest; u += kT) {
        const int q = u / rest, c = u - q * rest;
        U[q][c] = A[(size_t)(j0 + q) * n + c0 + c];
    }
    __syncthreads();
    const int i = c0 + blockIdx.x * (kT / 4) + (threadIdx.x >> 2);
    if (i >= n) return;
    double2* row = A + (size_t)i * n;
    double2 l[W];
#pragma unroll
    for (int q = 0; q < W; q++) l[q] = row[j0 + q];
    for (int c = threadIdx.x & 3; c < rest; c += 4) {
        double2 x = row[c0 + c];
#pragma unroll
        for (int q = 0; q < W; q++) x = csub(x, cmul(l[q], U[q][c]));
        row[c0 + c] = x;
    }
}

// The panel's row swaps applied to the columns outside it, 64 columns per
// workgroup: the panel's 32 rows and its pivot rows are read once and written
// once where the swaps take them (each of the up to 64 rows is followed
// through the 32 swaps by one lane).  Right of the panel the 32 rows become
// U12 = L11^-1 A12 on the way, four lanes per column: a solved entry goes to
// the other three by a quad permute, each then updates its 8 rows.
constexpr int kSwapCols = 64;

// lane Q's value to its quad
template <int Q>
__device__ __forceinline__ double quad_bcast(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x55 * Q, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x55 * Q, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double2 quad_bcast(double2 v, int q) {
    switch (q) {
        case 0: return make_double2(quad_bcast<0>(v.x), quad_bcast<0>(v.y));
        case 1: return make_double2(quad_bcast<1>(v.x), quad_bcast<1>(v.y));
        case 2: return make_double2(quad_bcast<2>(v.x), quad_bcast<2>(v.y));
        default: return make_double2(quad_bcast<3>(v.x), quad_bcast<3>(v.y));
    }
}

__global__ __launch_bounds__(kT) void k_lu_swap_trsm(double2* __restrict__ A, int n, int k0,
                                                     const int* __restrict__ piv) {
    __shared__ double2 X[2 * kNb][kSwapCols + 1];
    __shared__ double2 L[kNb][kNb + 1];
    __shared__ int row[2 * kNb], dst[2 * kNb], from[kNb];
    const int t = threadIdx.x;
    // column block b: the columns left of the panel, then those right of it
    const int left = (k0 + kSwapCols - 1) / kSwapCols, b = blockIdx.x;
    const bool right = b >= left;
    const int c0 = right ? k0 + kNb + (b - left) * kSwapCols : b * kSwapCols;
    const int cols = min(kSwapCols, (right ? n : k0) - c0);
    if (t < 2 * kNb) {
        // slot s < 32: row k0 + s; slot 32 + k: the row of pivot k if it lies below the panel and
        // no earlier pivot is the same row, else unused (-1).  pos: where the slot's data ends.
        int mine = k0 + t;
        if (t >= kNb) {
            mine = piv[k0 + t - kNb];
            if (mine < k0 + kNb) mine = -1;
        }
        int pos = mine;
#pragma unroll
        for (int k = 0; k < kNb; k++) {
            const int p = piv[k0 + k];
            if (t > kNb + k && mine == p) mine = -1;
            if (pos == k0 + k) pos = p;
            else if (pos == p) pos = k0 + k;
        }
        row[t] = mine;
        dst[t] = pos;
        if (mine >= 0 && pos < k0 + kNb) from[pos - k0] = t;
    }
    if (right)
        for (int u = t; u < kNb * kNb; u += kT) L[u / kNb][u % kNb] = A[(size_t)(k0 + u / kNb) * n + k0 + u % kNb];
    __syncthreads();
    const int cc = t & (kSwapCols - 1), q0 = t / kSwapCols;  // one column, every fourth slot
    if (cc < cols) {
        constexpr int kLoads = 2 * kNb * kSwapCols / kT;
        double2 v[kLoads];  // an unused slot reads row 0: every load is issued before the first is waited for
#pragma unroll
        for (int e = 0; e < kLoads; e++)
            v[e] = A[(size_t)max(row[q0 + e * (kT / kSwapCols)], 0) * n + c0 + cc];
#pragma unroll
        for (int e = 0; e < kLoads; e++) X[q0 + e * (kT / kSwapCols)][cc] = v[e];
    }
    __syncthreads();
    if (cc < cols)
        for (int q = q0; q < 2 * kNb; q += kT / kSwapCols)
            if (row[q] >= 0 && dst[q] != row[q] && (!right || dst[q] >= k0 + kNb))
                A[(size_t)dst[q] * n + c0 + cc] = X[q][cc];
    if (!right) return;
    const int h = t & 3, ct = t >> 2;  // lane h of column ct holds the rows 4 e + h
    double2 x[kNb / 4];
#pragma unroll
    for (int e = 0; e < kNb / 4; e++) x[e] = X[from[4 * e + h]][ct];
#pragma unroll
    for (int q = 0; q < kNb - 1; q++) {
        const double2 xq = quad_bcast(x[q / 4], q & 3);
#pragma unroll
        for (int e = q / 4; e < kNb / 4; e++) {
            const double2 d = cmul(L[4 * e + h][q], xq);
            if (4 * e + h > q) x[e] = csub(x[e], d);
        }
    }
    __syncthreads();  // every column has read X
#pragma unroll
    for (int e = 0; e < kNb / 4; e++) X[4 * e + h][ct] = x[e];
    __syncthreads();
    if (cc < cols)
        for (int r = q0; r < kNb; r += kT / kSwapCols) A[(size_t)(k0 + r) * n + c0 + cc] = X[r][cc];
}

// U12 = L11^-1 A12: rows [k0, k0 + kNb), columns [k0 + kNb, n) (after whole-row
// swaps of the column-by-column path).
__global__ __launch_bounds__(kT) void k_lu_trsm(double2* __restrict__ A, int n, int k0) {
    __shared__ double2 L[kNb][kNb + 1];
    for (int u = threadIdx.x; u < kNb * kNb; u += kT) {
        const int r = u / kNb, q = u - r * kNb;
        L[r][q] = A[(size_t)(k0 + r) * n + k0 + q];
    }
    __syncthreads();
    const int c = k0 + kNb + blockIdx.x * kT + threadIdx.x;
    if (c >= n) return;
    double2 x[kNb];
#pragma unroll
    for (int r = 0; r < kNb; r++) x[r] = A[(size_t)(k0 + r) * n + c];
#pragma unroll
    for (int r = 1; r < kNb; r++) {
        double2 s = x[r];
#pragma unroll
        for (int q = 0; q < r; q++) s = csub(s, cmul(L[r][q], x[q]));
        x[r] = s;
    }
#pragma unroll
    for (int r = 1; r < kNb; r++) A[(size_t)(k0 + r) * n + c] = x[r];
}

typedef double d4v __attribute__((ext_vector_type(4)));

// B operand of the complex product as a real one: K position 2q + odd holds
// Re (odd = 0) or Im (odd = 1) of L[.][q]; real output column 2c + part is
// Re (part 0) or Im (part 1) of the product, so B'[2q][2c] = Re U, B'[2q+1][2c]
// = -Im U, B'[2q][2c+1] = Im U, B'[2q+1][2c+1] = Re U.
__device__ inline double bprime(double2 u, int odd, int part) {
    return odd ? (part ? u.x : -u.y) : (part ? u.y : u.x);
}

// A22 -= L21 U12 for rows and columns >= k0 + kNb: one workgroup per 64 x 64
// complex tile, each wave 16 rows x 64 complex columns (8 MFMA tiles of 16
// real columns), K = 64 real positions in 16 steps.  The MFMA operand and
// result layouts: A[row = lane & 15][k = lane >> 4], B[k = lane >> 4][col =
// lane & 15], D[row = 4 q + (lane >> 4)][col = lane & 15] for q = 0..3.
__global__ __launch_bounds__(kT) void k_lu_gemm(double2* __restrict__ A, int n, int k0) {
    __shared__ double2 Ls[kTile][kNb + 1];
    __shared__ double2 Us[kNb][kTile + 1];
    const int r0 = k0 + kNb;
    const int tr = r0 + blockIdx.y * kTile, tc = r0 + blockIdx.x * kTile;
    for (int u = threadIdx.x; u < kTile * kNb; u += kT) {
        const int r = u / kNb, q = u - r * kNb;
        const int i = tr + r;
        Ls[r][q] = i < n ? A[(size_t)i * n + k0 + q] : make_double2(0.0, 0.0);
    }
    for (int u = threadIdx.x; u < kNb * kTile; u += kT) {
        const int q = u / kTile, cc = u - q * kTile;
        const int c = tc + cc;
        Us[q][cc] = c < n ? A[(size_t)(k0 + q) * n + c] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int g = lane >> 4, col = lane & 15, part = col & 1;
    double* Ad = (double*)A;
    d4v acc[8];
#pragma unroll
    for (int t = 0; t < 8; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int i = tr + w * 16 + 4 * q + g, c = tc + t * 8 + (col >> 1);
            acc[t][q] = (i < n && c < n) ? Ad[2 * ((size_t)i * n + c) + part] : 0.0;
        }
    const int odd = g & 1;
#pragma unroll
    for (int s = 0; s < 2 * kNb / 4; s++) {
        const int q = 2 * s + (g >> 1);
        const double2 lv = Ls[w * 16 + col][q];
        const double a = odd ? -lv.y : -lv.x;
#pragma unroll
        for (int t = 0; t < 8; t++)
            acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bprime(Us[q][t * 8 + (col >> 1)], odd, part), acc[t], 0,
                                                          0, 0);
    }
#pragma unroll
    for (int t = 0; t < 8; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int i = tr + w * 16 + 4 * q + g, c = tc + t * 8 + (col >> 1);
            if (i < n && c < n) Ad[2 * ((size_t)i * n + c) + part] = acc[t][q];
        }
}

// x[s][k] = b[s][perm[k]]
__global__ __launch_bounds__(kT) void k_lu_permute(const double2* __restrict__ b, double2* __restrict__ x,
                                                   const int* __restrict__ perm, int n) {
    const int k = blockIdx.x * kT + threadIdx.x;
    const size_t o = (size_t)blockIdx.y * n;
    if (k < n) x[o + k] = b[o + perm[k]];
}

// Diagonal block [b0, b0 + nb) of L (unit lower, LOWER) or U (upper, with its
// diagonal): one wave per right-hand side (grid.x), lane q holds unknown q.  A
// solved unknown is broadcast and every lane adds its term: a step is a
// broadcast and one multiply-add, where a wave-wide sum per row took 0.5 us.
// The terms are summed apart from y and taken off once: off y one by one, each
// rounds at the size of y (diagonally dominant n = 33: error of the solution
// 3.5e-16, 2.6e-16 so).
__device__ __forceinline__ double lane_value(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
constexpr int kSb = 64;  // unknowns per diagonal block of the substitutions
template <bool LOWER>
__global__ __launch_bounds__(kT) void k_lu_diag_solve(const double2* __restrict__ LU, int n, int b0, int nb,
                                                      double2* __restrict__ x) {
    __shared__ double2 B[kSb][kSb + 1];
    const int q = threadIdx.x & (kSb - 1);
#pragma unroll
    for (int k = 0; k < kSb; k += kT / kSb) {
        const int r = k + threadIdx.x / kSb;
        if (r < nb && q < nb) B[r][q] = LU[(size_t)(b0 + r) * n + b0 + q];
    }
    __syncthreads();
    if (threadIdx.x >= kSb) return;
    double2* xs = x + (size_t)blockIdx.x * n + b0;
    double2 y = q < nb ? xs[q] : make_double2(0.0, 0.0);
    const double2 inv = !LOWER && q < nb ? cdiv(make_double2(1.0, 0.0), B[q][q]) : make_double2(1.0, 0.0);
    double2 t = make_double2(0.0, 0.0);  // this unknown's sum of solved terms
    for (int k = 0; k < nb; k++) {
        const int r = LOWER ? k : nb - 1 - k;
        const double2 b = B[q][r];
        double2 v = csub(y, t);
        if (!LOWER) v = cquot(v, b, inv);
        const double2 s = make_double2(lane_value(v.x, r), lane_value(v.y, r));
        if (q == r) y = v;
        if (q < nb && (LOWER ? q > r : q < r)) cfma(t, b, s);
    }
    if (q < nb) xs[q] = y;
}

// x[s][i] -= sum_q LU[i][b0 + q] x[s][b0 + q] for the rows i in [i0, i1)
// (below the block for L, above it for U): four threads per row, each every
// fourth column (64-byte runs of the row), for up to kUpdS right-hand sides
// (grid.y groups), so that a row of LU is read once per group.
constexpr int kUpdS = 4;
__global__ __launch_bounds__(kT) void k_lu_block_update(const double2* __restrict__ LU, int n, int S, int b0, int nb,
                                                        int i0, int i1, double2* __restrict__ x) {
    __shared__ double2 xb[kUpdS][kSb];
    const int s0 = blockIdx.y * kUpdS, ns = min(kUpdS, S - s0);
    for (int u = threadIdx.x; u < kUpdS * kSb; u += kT) {
        const int s = u / kSb, q = u % kSb;
        xb[s][q] = s < ns && q < nb ? x[(size_t)(s0 + s) * n + b0 + q] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    const int i = i0 + blockIdx.x * (kT / 4) + (threadIdx.x >> 2), part = threadIdx.x & 3;
    const double2* row = LU + (size_t)min(i, i1 - 1) * n + b0;
    double2 acc[kUpdS];
#pragma unroll
    for (int s = 0; s < kUpdS; s++) acc[s] = make_double2(0.0, 0.0);
#pragma unroll
    for (int k = 0; k < kSb / 4; k++) {
        const int q = 4 * k + part;
        const double2 l = q < nb ? row[q] : make_double2(0.0, 0.0);
#pragma unroll
        for (int s = 0; s < kUpdS; s++) cfma(acc[s], l, xb[s][q]);
    }
#pragma unroll
    for (int s = 0; s < kUpdS; s++) {
#pragma unroll
        for (int off = 1; off < 4; off <<= 1) {
            acc[s].x += __shfl_xor(acc[s].x, off);
            acc[s].y += __shfl_xor(acc[s].y, off);
        }
        if (s == part && s < ns && i < i1) {
            double2* o = x + (size_t)(s0 + s) * n + i;
            *o = csub(*o, acc[s]);
        }
    }
}

int parts_for(int rows) {
    int g = (rows + kT - 1) / kT;
    return g < 1 ? 1 : (g > kMaxParts ? kMaxParts : g);
}

// One panel column by column with whole-row swaps: two launches per column.
void factor_columns(double2* A, int n, int k0, int k_end, const LuWs& W, int swap_grid, hipStream_t st) {
    int nparts = parts_for(n - k0);
    hipLaunchKernelGGL(k_lu_pivot_search, dim3(nparts), dim3(kT), 0, st, (const double2*)A, n, k0, W.pval, W.pidx);
    for (int j = k0; j < k_end; j++) {
        hipLaunchKernelGGL(k_lu_swap, dim3(swap_grid), dim3(kT), 0, st, A, n, j, (const double*)W.pval,
                           (const int*)W.pidx, nparts, W.piv, W.info);
        const int g = parts_for(n - j - 1);
        hipLaunchKernelGGL(k_lu_panel, dim3(g), dim3(kT), 0, st, A, n, j, k_end, W.pval, W.pidx);
        nparts = g;  // the partial maxima of column j + 1 (when j + 1 < k_end)
    }
}

// One strip of w columns and the update of the panel's columns right of it.
template <int W, int RPT>
void launch_strip(double2* A, int n, int k0, int j0, const LuWs& ws, hipStream_t st) {
    const int k_end = k0 + kNb;
    hipLaunchKernelGGL((k_lu_strip<W, RPT>), dim3(1), dim3(kStripT), 0, st, A, n, k0, j0, k_end, ws.piv, ws.info);
    if (j0 + W < k_end)
        hipLaunchKernelGGL((k_lu_strip_update<W>), dim3((n - j0 - W + kT / 4 - 1) / (kT / 4)), dim3(kT), 0, st, A, n,
                           j0, k_end);
}

void factor_strips(double2* A, int n, int k0, int w, const LuWs& ws, hipStream_t st) {
    for (int j0 = k0; j0 < k0 + kNb; j0 += w) {
        const int rpt = (n - j0 + kStripT - 1) / kStripT;  // rows per thread
        if (w == 16 && rpt <= 1) launch_strip<16, 1>(A, n, k0, j0, ws, st);
        else if (w == 16) launch_strip<16, 2>(A, n, k0, j0, ws, st);
        else if (w == 8 && rpt <= 3) launch_strip<8, 3>(A, n, k0, j0, ws, st);
        else if (w == 8) launch_strip<8, 5>(A, n, k0, j0, ws, st);
        else if (rpt <= 7) launch_strip<4, 7>(A, n, k0, j0, ws, st);
        else launch_strip<4, 10>(A, n, k0, j0, ws, st);
    }
}

int lu_factor(int n, double2* A, int add_identity, void* workspace, int* info_out, hipStream_t st) {
    const LuWs W = ws_view(workspace, n);
    MPA_HIP_CHECK(hipMemsetAsync(W.info, 0, sizeof(int), st));
    if (add_identity) hipLaunchKernelGGL(k_lu_add_identity, dim3((n + kT - 1) / kT), dim3(kT), 0, st, A, n);
    const int swap_grid = std::min(64, (n + kT - 1) / kT);
    for (int k0 = 0; k0 < n; k0 += kNb) {
        const int k_end = std::min(n, k0 + kNb);
        const int tiles = (n - k_end + kTile - 1) / kTile;
        const int w = strip_width(n - k0);
        // A last panel of fewer than 32 columns, or rows past the registers of a workgroup: column by column.
        if (w == 0 || k_end - k0 < kNb) {
            factor_columns(A, n, k0, k_end, W, swap_grid, st);
            if (k_end < n)
                hipLaunchKernelGGL(k_lu_trsm, dim3((n - k_end + kT - 1) / kT), dim3(kT), 0, st, A, n, k0);
        } else {
            factor_strips(A, n, k0, w, W, st);
            const int cols = (k0 + kSwapCols - 1) / kSwapCols + (n - k_end + kSwapCols - 1) / kSwapCols;
            if (cols)
                hipLaunchKernelGGL(k_lu_swap_trsm, dim3(cols), dim3(kT), 0, st, A, n, k0, (const int*)W.piv);
        }
        if (tiles > 0) hipLaunchKernelGGL(k_lu_gemm, dim3(tiles, tiles), dim3(kT), 0, st, A, n, k0);
        MPA_LAUNCH_CHECK();
    }
    // the swaps, in order, as one permutation of the right-hand side's rows
    std::vector<int> piv(n), perm(n);
    int info = 0;
    MPA_HIP_CHECK(hipMemcpyAsync(piv.data(), W.piv, sizeof(int) * n, hipMemcpyDeviceToHost, st));
    MPA_HIP_CHECK(hipMemcpyAsync(&info, W.info, sizeof(int), hipMemcpyDeviceToHost, st));
    MPA_HIP_CHECK(hipStreamSynchronize(st));
    for (int k = 0; k < n; k++) perm[k] = k;
    for (int j = 0; j < n; j++) std::swap(perm[j], perm[piv[j]]);
    MPA_HIP_CHECK(hipMemcpyAsync(W.perm, perm.data(), sizeof(int) * n, hipMemcpyHostToDevice, st));
    MPA_HIP_CHECK(hipStreamSynchronize(st));
    if (info_out) *info_out = info;
    if (info) {
        char msg[96];
        std::snprintf(msg, sizeof msg, "lu_factor: singular matrix (no nonzero pivot in column %d)", info - 1);
        mpa_set_error(msg);
        return MPA_BREAKDOWN;
    }
    return MPA_OK;
}

int lu_solve(int n, int S, const double2* LU, void* workspace, const double2* b, double2* x, hipStream_t st) {
    const LuWs W = ws_view(workspace, n);
    hipLaunchKernelGGL(k_lu_permute, dim3((n + kT - 1) / kT, S), dim3(kT), 0, st, b, x, (const int*)W.perm, n);
    const unsigned groups = (S + kUpdS - 1) / kUpdS;
    constexpr int rows = kT / 4;
    for (int b0 = 0; b0 < n; b0 += kSb) {  // L y = P b
        const int nb = std::min(kSb, n - b0), i0 = b0 + nb;
        hipLaunchKernelGGL(k_lu_diag_solve<true>, dim3(S), dim3(kT), 0, st, LU, n, b0, nb, x);
        if (i0 < n)
            hipLaunchKernelGGL(k_lu_block_update, dim3((n - i0 + rows - 1) / rows, groups), dim3(kT), 0, st, LU, n, S,
                               b0, nb, i0, n, x);
    }
    for (int b0 = ((n - 1) / kSb) * kSb; b0 >= 0; b0 -= kSb) {  // U x = y
        const int nb = std::min(kSb, n - b0);
        hipLaunchKernelGGL(k_lu_diag_solve<false>, dim3(S), dim3(kT), 0, st, LU, n, b0, nb, x);
        if (b0 > 0)
            hipLaunchKernelGGL(k_lu_block_update, dim3((b0 + rows - 1) / rows, groups), dim3(kT), 0, st, LU, n, S, b0,
                               nb, 0, b0, x);
    }
    MPA_LAUNCH_CHECK();
    return MPA_OK;
}

}  // namespace

extern "C" {

size_t mpa_lu_workspace_bytes(int n) { return n < 1 ? 0 : ws_bytes(n); }

int mpa_lu_factor(int n, void* A, int add_identity, void* workspace, int* info_out, void* stream) {
    if (n < 1 || !A || !workspace) {
        mpa_set_error("lu_factor: bad argument");
        return MPA_ERR_ARG;
    }
    return lu_factor(n, (double2*)A, add_identity, workspace, info_out, (hipStream_t)stream);
}

int mpa_lu_solve(int n, int nrhs, const void* LU, void* workspace, const void* b, void* x, void* stream) {
    if (n < 1 || nrhs < 1 || nrhs > 65535 || !LU || !workspace || !b || !x || b == x) {
        mpa_set_error("lu_solve: bad argument (b and x must be distinct buffers)");
        return MPA_ERR_ARG;
    }
    return lu_solve(n, nrhs, (const double2*)LU, workspace, (const double2*)b, (double2*)x, (hipStream_t)stream);
}

}  // extern "C"
