// Dense complex matvec / multi-RHS product: kernels, tile variants, the
// autotuner and the C ABI.  Replaces the OpenMP row-block GEMV of
// cpp/src/interactions.cpp:62-95 (and the products inside Eigen's BiCGSTAB).
//
// The system matrix is read from HBM once per pass in 16-byte loads.  It is not
// reused within a call, so these are nontemporal and leave the caches to x,
// but for matrix-core tiles over rows that are no whole 128-byte lines
// (gemm_rows).  Vector-ALU tiles (one pass): each wave of a workgroup owns R
// consecutive rows of one system and runs along the full rows with U chunks
// per lane in flight; the x chunk loaded for a column is reused for the R rows
// and for up to SG right-hand sides held in registers.  Matrix-core tiles: 8
// right-hand sides per pass up to 8 of them, 16 beyond.  Jobs whose system has converged for all right-hand sides return before
// touching the matrix.

#include <vector>

#include "gemv.hpp"

namespace mpa {
namespace {

typedef double dvec2 __attribute__((ext_vector_type(2)));
typedef float fvec4 __attribute__((ext_vector_type(4)));

template <typename T> struct Chunk;
template <> struct Chunk<double> {
    using v = dvec2;
    static constexpr int C = 1;  // complex entries per 16-byte chunk
};
template <> struct Chunk<float> {
    using v = fvec4;
    static constexpr int C = 2;
};

__device__ inline void chunk_fma(double& ar, double& ai, dvec2 a, dvec2 x) {
    ar = fma(a.x, x.x, ar);
    ar = fma(-a.y, x.y, ar);
    ai = fma(a.x, x.y, ai);
    ai = fma(a.y, x.x, ai);
}
__device__ inline void chunk_fma(float& ar, float& ai, fvec4 a, fvec4 x) {
    ar = fmaf(a.x, x.x, ar);
    ar = fmaf(-a.y, x.y, ar);
    ai = fmaf(a.x, x.y, ai);
    ai = fmaf(a.y, x.x, ai);
    ar = fmaf(a.z, x.z, ar);
    ar = fmaf(-a.w, x.w, ar);
    ai = fmaf(a.z, x.w, ai);
    ai = fmaf(a.w, x.z, ai);
}

__device__ inline bool all_done(const SysDev& d) {
    const Scal* scal = glob(d.scal);
    for (int s = 0; s < d.S; s++)
        if (!scal[s].done) return false;
    return true;
}

// One workgroup's share of a matvec job: its four waves own R rows each from
// row `first` on, up to row `end`; SG right-hand sides per pass, U chunks in
// flight.  A row's sum is taken in the same order whatever R, SG and U are,
// so a launch may pick its tile freely.
template <typename T, int R, int SG, int U>
__device__ inline void gemv_rows(const MvDev& J, int first, int end) {
    using V = typename Chunk<T>::v;
    constexpr int C = Chunk<T>::C;
    const int n = J.n;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int row0 = first + w * R;
    end = min(end, n);
    if (row0 >= end) return;
    const int nv = n / C;  // 16-byte chunks per row (n is even)
    const T* A = glob((const T*)J.A);
    const V* Ar[R];
#pragma unroll
    for (int r = 0; r < R; r++) Ar[r] = (const V*)(A + (size_t)2 * n * min(row0 + r, end - 1));
    for (int s0 = 0; s0 < J.S; s0 += SG) {
        T ar[R][SG], ai[R][SG];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int s = 0; s < SG; s++) ar[r][s] = ai[r][s] = 0;
        const V* xs[SG];
#pragma unroll
        for (int s = 0; s < SG; s++) xs[s] = (const V*)(glob((const T*)J.x) + (size_t)2 * n * min(s0 + s, J.S - 1));
        int c = lane;
        for (; c + 64 * (U - 1) < nv; c += 64 * U) {
            V xv[SG][U];
#pragma unroll
            for (int s = 0; s < SG; s++)
#pragma unroll
                for (int u = 0; u < U; u++) xv[s][u] = xs[s][c + 64 * u];
            V av[R][U];
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int u = 0; u < U; u++) av[r][u] = __builtin_nontemporal_load(Ar[r] + c + 64 * u);
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int s = 0; s < SG; s++)
#pragma unroll
                    for (int u = 0; u < U; u++) chunk_fma(ar[r][s], ai[r][s], av[r][u], xv[s][u]);
        }
        for (; c < nv; c += 64) {
            V xv[SG];
#pragma unroll
            for (int s = 0; s < SG; s++) xv[s] = xs[s][c];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const V a = __builtin_nontemporal_load(Ar[r] + c);
#pragma unroll
                for (int s = 0; s < SG; s++) chunk_fma(ar[r][s], ai[r][s], a, xv[s]);
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int s = 0; s < SG; s++) {
                T re = ar[r][s], im = ai[r][s];
                for (int off = 32; off > 0; off >>= 1) {
                    re += __shfl_xor(re, off);
                    im += __shfl_xor(im, off);
                }
                const int row = row0 + r;
                if (lane == 0 && row < end && s0 + s < J.S) {
                    const size_t o = (size_t)(s0 + s) * n + row;
                    cplx_t<T> yv = cmake<T>(re, im);
                    if (J.add_identity) yv = cadd(yv, glob((const cplx_t<T>*)J.x)[o]);
                    glob((cplx_t<T>*)J.y)[o] = yv;
                }
            }
    }
}

// ---- multi-RHS products on the matrix cores ------------------------------------
//
// Y = (I +) A X as a real GEMM: a complex row of A is the real row (Re a_0,
// Im a_0, Re a_1, ...), and right-hand side s contributes two real columns
// (one per output part),
//   X'[2j][(s,re)] = Re x_j,  X'[2j][(s,im)] = Im x_j,
//   X'[2j+1][(s,re)] = -Im x_j, X'[2j+1][(s,im)] = Re x_j,
// so that Y_re = sum Re a Re x - Im a Im x and Y_im = sum Re a Im x + Im a Re x.
// Eight right-hand sides fill the 16 real columns of one MFMA tile
// (v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64).
//
// A workgroup owns 16 rows and its W waves split the columns of those rows
// (wave w takes the K steps w, w + W, ...), so that also a matrix of a few
// thousand rows gives every CU several independent streams.  A wave moves a K
// step of its 16 rows and of the right-hand sides from global memory into
// registers in runs of 64 Q bytes per row, one step ahead, and through its own
// part of LDS into the MFMA operand layout; nothing is shared between waves,
// so the loop has no barriers.  At the end the waves' tiles are added in LDS.
// Rows of an LDS buffer are padded by 16 bytes: the 16 rows of
// one operand read then cover all banks.
//   A operand: lane l holds row l % 16 and, per 16-byte read, 4 consecutive
//     reals of c64 (2 complex) or 2 of c128 (1 complex) at the K offset of
//     its group g = l / 16; its components feed 4 or 2 MFMAs, each with the
//     X' operand of the same K position (col l % 16: s = col / 2, part = col % 2).
//   D[i]: row 4 g + i (f32) or 4 i + g (f64), column l % 16.

typedef double d4v __attribute__((ext_vector_type(4)));

constexpr int kGemmS8 = 8;  // right-hand sides per 16-column tile
constexpr int kGemmW = 8;   // waves per workgroup (the column split)
constexpr int kGemmQ = 4;   // 64-byte groups of a row per K step

template <typename T> struct MfmaTile;
template <> struct MfmaTile<float> {
    using acc = fvec4;
    static constexpr int C = 2;  // complex entries per 16-byte load
    static constexpr int K = 4;  // MFMAs per 16-byte load of A
    __device__ static int row(int g, int i) { return 4 * g + i; }
    // the K MFMAs of one 16-byte load of A times X', number e into chain (c0 + e) % NC
    template <int NC>
    __device__ static void fma(acc (&d)[NC], int c0, fvec4 a, fvec4 x, int part) {
        const float b[K] = {part ? x.y : x.x, part ? x.x : -x.y, part ? x.w : x.z, part ? x.z : -x.w};
#pragma unroll
        for (int e = 0; e < K; e++) {
            acc& s = d[(c0 + e) % NC];
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], s, 0, 0, 0);
        }
    }
};
template <> struct MfmaTile<double> {
    using acc = d4v;
    static constexpr int C = 1;
    static constexpr int K = 2;
    __device__ static int row(int g, int i) { return 4 * i + g; }
    template <int NC>
    __device__ static void fma(acc (&d)[NC], int c0, dvec2 a, dvec2 x, int part) {
        const double b[K] = {part ? x.y : x.x, part ? x.x : -x.y};
#pragma unroll
        for (int e = 0; e < K; e++) {
            acc& s = d[(c0 + e) % NC];
            s = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], b[e], s, 0, 0, 0);
        }
    }
};

// Orders a wave's own LDS writes and reads by different lanes.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// 16-byte chunks of LDS a wave needs: 16 rows of A and 8 NT of X, 4 Q chunks
// and one of padding each.
constexpr int gemm_wave_chunks(int RT, int NT) { return (16 * RT + 8 * NT) * (4 * kGemmQ + 1); }

// Accumulators per tile.  An MFMA rounds once per product, so one accumulator
// per wave adds n / 4 products one after the other.  With one column tile every
// MFMA of a K step has its own: n / 64 (c64) or n / 32 (c128) products and a
// tree, which is the rounding of the vector tiles' 64 lane sums.  Error of 3
// sources against 64 bits (c64; c128 against 80), one accumulator and now:
// n = 330 1.8e-7 and 8.6e-8 (vector tile 9.0e-8), 9990 9.0e-7 and 2.4e-7
// (3.2e-7); c128 330 3.1e-16 and 1.7e-16 (1.7e-16), 9990 1.6e-15 and 6.2e-16
// (6.2e-16).
template <typename T, int NT>
constexpr int gemm_chains() {
    return NT == 1 ? kGemmQ * MfmaTile<T>::K : 1;
}

// The right-hand sides [s0, s0 + 8 NT) of rows [r0, r0 + 16 RT).
template <typename T, int RT, int NT, bool STREAM>
__device__ __forceinline__ void gemm_pass(const MvDev& J, int r0, int s0, typename Chunk<T>::v* lds) {
    using V = typename Chunk<T>::v;
    using M = MfmaTile<T>;
    constexpr int W = kGemmW, Q = kGemmQ, C = M::C, CH = 4 * Q, RS = CH + 1;  // chunks per row and K step; padded row in LDS
    constexpr int LA = RT * Q, LX = NT * Q / 2;            // loads per lane: 16 (or 8 NT) rows x CH chunks / 64
    const int n = J.n;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, col = lane & 15, part = col & 1;
    V* la = lds + w * gemm_wave_chunks(RT, NT);
    V* lx = la + 16 * RT * RS;
    // lane's chunk of load k: id = 64 k + lane, row id / CH, chunk id % CH, as a byte offset from the pass's
    // first row and source, whose addresses stay in scalar registers
    const char* A0 = (const char*)(glob((const cplx_t<T>*)J.A) + (size_t)n * r0);
    const char* x0 = (const char*)(glob((const cplx_t<T>*)J.x) + (size_t)n * s0);
    constexpr unsigned ES = sizeof(cplx_t<T>);
    unsigned oa[LA], ox[LX];
    const int ch = lane % CH;
#pragma unroll
    for (int k = 0; k < LA; k++) oa[k] = (unsigned)min((64 * k + lane) / CH, n - 1 - r0) * n * ES + 16 * ch;
#pragma unroll
    for (int k = 0; k < LX; k++) ox[k] = (unsigned)min((64 * k + lane) / CH, J.S - 1 - s0) * n * ES + 16 * ch;
    constexpr int NC = gemm_chains<T, NT>();
    typename M::acc acc[RT][NT][NC];
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int u = 0; u < NT; u++)
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[t][u][c][i] = 0;
    const int nv = n / C;  // 16-byte chunks per row (n is even)
    const int steps = (nv + CH - 1) / CH;
    V a[LA], x[LX];
    auto load = [&](int kb) {
        const bool in = kb * CH + ch < nv;
        // Opaque, or the compiler keeps a 64-bit pointer per load: 30 registers more, which leave one
        // workgroup per CU (30 systems of n = 640, c64, 8 sources: 184 us per iteration, 169 with two).
        unsigned step = kb * (16 * CH);
        asm volatile("" : "+s"(step));
#pragma unroll
        for (int k = 0; k < LA; k++) {
            const V* p = (const V*)(A0 + (size_t)(oa[k] + step));
            a[k] = !in ? V(0) : STREAM ? __builtin_nontemporal_load(p) : *p;
        }
#pragma unroll
        for (int k = 0; k < LX; k++) x[k] = in ? *(const V*)(x0 + (size_t)(ox[k] + step)) : V(0);
    };
    if (w < steps) load(w);
    for (int kb = w; kb < steps; kb += W) {
#pragma unroll
        for (int k = 0; k < LA; k++) la[(64 * k + lane) / CH * RS + ch] = a[k];
#pragma unroll
        for (int k = 0; k < LX; k++) lx[(64 * k + lane) / CH * RS + ch] = x[k];
        wave_fence();
        if (kb + W < steps) load(kb + W);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            V av[RT];
#pragma unroll
            for (int t = 0; t < RT; t++) av[t] = la[(16 * t + col) * RS + 4 * q + g];
#pragma unroll
            for (int u = 0; u < NT; u++) {
                const V xv = lx[(8 * u + (col >> 1)) * RS + 4 * q + g];
#pragma unroll
                for (int t = 0; t < RT; t++) M::fma(acc[t][u], q * M::K, av[t], xv, part);
            }
        }
        wave_fence();  // the next step's writes stay behind these reads
    }
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int u = 0; u < NT; u++)
#pragma unroll
            for (int h = NC / 2; h > 0; h /= 2)
#pragma unroll
                for (int c = 0; c < h; c++) acc[t][u][c] += acc[t][u][c + h];
    // the waves' tiles, added as a tree (over the operand buffers)
    constexpr int TILE = RT * NT * 256;
    T* red = (T*)lds;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int u = 0; u < NT; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) red[w * TILE + ((t * NT + u) * 4 + i) * 64 + lane] = acc[t][u][0][i];
    __syncthreads();
    for (int e = tid; e < TILE; e += 64 * W) {
        T p[W];
#pragma unroll
        for (int k = 0; k < W; k++) p[k] = red[k * TILE + e];
#pragma unroll
        for (int h = W / 2; h > 0; h /= 2)
#pragma unroll
            for (int k = 0; k < h; k++) p[k] += p[k + h];
        T v = p[0];
        const int l = e & 63, i = (e >> 6) & 3, tu = e >> 8, t = tu / NT, u = tu - t * NT;
        const int r = r0 + 16 * t + M::row(l >> 4, i), s = s0 + 8 * u + ((l & 15) >> 1);
        if (r < n && s < J.S) {
            const size_t o = 2 * ((size_t)s * n + r) + (l & 1);
            if (J.add_identity) v += glob((const T*)J.x)[o];
            glob((T*)J.y)[o] = v;
        }
    }
    __syncthreads();  // before the next pass overwrites the sums
}

// All right-hand sides in passes of 8 NT (A streamed once per pass).
template <typename T, int RT, int NT>
__device__ __forceinline__ void gemm_rows(const MvDev& J, int first) {
    constexpr int ops = kGemmW * gemm_wave_chunks(RT, NT);                         // operand buffers
    constexpr int sums = kGemmW * RT * NT * 256 * (int)sizeof(T) / 16;             // the waves' tiles
    __shared__ typename Chunk<T>::v lds[ops > sums ? ops : sums];
    if (first >= J.n) return;
    // Rows of whole 128-byte lines are streamed past the caches (c64, 8 sources, n = 9648: 133 us, 142 through
    // them).  Otherwise neighbouring steps share lines, which the caches then serve (n = 9990: 174 us, 183).
    if (J.n % (128 / (2 * (int)sizeof(T))) == 0) {
        for (int s0 = 0; s0 < J.S; s0 += NT * kGemmS8) gemm_pass<T, RT, NT, true>(J, first, s0, lds);
    } else {
        for (int s0 = 0; s0 < J.S; s0 += NT * kGemmS8) gemm_pass<T, RT, NT, false>(J, first, s0, lds);
    }
}

// ---- launches -------------------------------------------------------------------------
//
// Work lists name (job, block of `unit` rows), the same list whatever the
// tile: `sub` workgroups share a block.  A launch whose blocks all belong to
// one job passes sub = 0: workgroup b then owns the b-th tile of that job.

struct RowRange {
    int job, first, end;
};
__device__ __forceinline__ RowRange rows_of_block(const int2* __restrict__ work, int rows, int unit, int sub) {
    if (sub == 0) return {work[0].x, (int)blockIdx.x * rows, 0x7fffffff};
    const int item = blockIdx.x / sub;
    const int2 wk = work[item];
    return {wk.x, wk.y * unit + ((int)blockIdx.x - item * sub) * rows, (wk.y + 1) * unit};
}

template <typename T, int RT, int NT>
__global__ __launch_bounds__(64 * kGemmW) void k_gemm(const MvDev* __restrict__ jobs, const SysDev* __restrict__ sys,
                                                      const int2* __restrict__ work, int unit, int sub) {
    const RowRange q = rows_of_block(work, 16 * RT, unit, sub);
    const MvDev J = jobs[q.job];
    if (J.skip >= 0 && all_done(sys[J.skip])) return;
    gemm_rows<T, RT, NT>(J, q.first);
}

template <typename T, int RT, int NT>
__global__ __launch_bounds__(64 * kGemmW) void k_gemm1(MvDev J) {
    gemm_rows<T, RT, NT>(J, blockIdx.x * 16 * RT);
}

template <typename T, int R, int SG, int U>
__global__ __launch_bounds__(kThreads) void k_gemv(const MvDev* __restrict__ jobs, const SysDev* __restrict__ sys,
                                                   const int2* __restrict__ work, int unit, int sub) {
    const RowRange q = rows_of_block(work, 4 * R, unit, sub);
    const MvDev J = jobs[q.job];
    if (J.skip >= 0 && all_done(sys[J.skip])) return;
    gemv_rows<T, R, SG, U>(J, q.first, q.end);
}

// one job passed by value
template <typename T, int R, int SG, int U>
__global__ __launch_bounds__(kThreads) void k_gemv1(MvDev J) {
    gemv_rows<T, R, SG, U>(J, blockIdx.x * 4 * R, J.n);
}

// ---- tile variants ------------------------------------------------------------------

// Variant 0 of a class is chosen per launch by size (auto_variant); the
// others fix a tile: R rows per wave and U chunks in flight (classes of one
// and two right-hand sides), or RT 16-row tiles per workgroup of the
// matrix-core product (SG = 0).
struct Variant {
    int R, SG, U;
    const char* name;
};
constexpr int kMaxVariants = 9;
const Variant kVariants[kTileClasses][kMaxVariants] = {
    {{0, 1, 0, "auto"}, {8, 1, 2, "r8u2"}, {6, 1, 2, "r6u2"}, {5, 1, 2, "r5u2"}, {4, 1, 2, "r4u2"}, {3, 1, 4, "r3u4"},
     {2, 1, 4, "r2u4"}, {1, 1, 8, "r1u8"}},
    {{0, 2, 0, "auto"}, {5, 2, 2, "r5u2"}, {4, 2, 2, "r4u2"}, {3, 2, 2, "r3u2"}, {2, 2, 4, "r2u4"}, {1, 2, 4, "r1u4"}},
    {{0, 0, 0, "auto"}, {1, 0, 0, "mfma16"}, {2, 0, 0, "mfma32"}},
    {{0, 0, 0, "auto"}, {1, 0, 0, "mfma16"}, {2, 0, 0, "mfma32"}},
};
int g_variant[2][kTileClasses] = {{0, 0, 0, 0}, {0, 0, 0, 0}};  // [es == 8][class]

// rows of a work-list block per class (c64 / c128)
constexpr int kUnit[2][kTileClasses] = {{32, 16, 128, 128}, {32, 16, 64, 64}};

inline int nvariants(int c) {
    int k = 0;
    while (k < kMaxVariants && kVariants[c][k].name) k++;
    return k;
}

int rows_of_variant(int c, int v) {
    const Variant& V = kVariants[c][v];
    return V.SG == 0 ? 16 * V.R : 4 * V.R;
}

// The tile of a launch over `rows` rows.  A CU streams at its own limit
// however many workgroups it holds, so a launch takes as long as the CU with
// the most rows: rounds = ceil(workgroups / 256) times the rows of a
// workgroup.  The tile with the smallest such count, weighted by what the tile
// itself costs, is the fastest measured one or within 4 % of it at all of the
// 27 sizes tried from 592 to 30000 rows.  us per product, this rule and the
// fixed r8u2 / 128-row tiles that served every size before: n = 592 c128 7.3 and
// 12.5, 2910 24 and 45, 4500 51 and 69, 9000 189 and 260, 20000 920 and 982; 8
// right-hand sides c64 5600 46 and 306, 9648 132 and 511, 16000 301 and 844.
double tile_weight(int c, int R, int es, long rounds) {
    if (c >= 2) return R == 1 ? 1.05 : 1.0;  // one 16-row tile reads X twice as often as two
    if (c == 0) {
        if (R == 8) return rounds <= 2 ? 1.001 : 1.0;  // r4u2 first where both fill the same rounds
        return R == 1 ? 1.12 : R == 2 ? 1.04 : 1.0;    // x is read R times less often than A
    }
    if (R == 5) return es == 8 && rounds == 1 ? 1.5 : 1.0;  // alone on a CU its loads do not cover the latency
    return R == 1 ? 1.30 : R == 2 ? 1.08 : 1.0;
}

// block: rows of a work-list block, 0 for one job.  A list splits every block by
// itself, so there only tiles that divide the block are counted rightly, and the
// others leave part-filled workgroups: 12 systems of n = 2500 (c128, 1 source;
// 948 blocks of 32) ran 24-row tiles, 24 + 8 rows per block, at 866 us per
// BiCGSTAB iteration; 785 us in 32-row tiles, 710 us in the 8-row ones that
// fill the rounds best.
int auto_variant(int c, long rows, int es, int block) {
    constexpr long kCus = 256;
    int best = 1;
    double best_cost = 1e300;
    for (int v = 1; v < nvariants(c); v++) {
        const long tile = rows_of_variant(c, v), rounds = ((rows + tile - 1) / tile + kCus - 1) / kCus;
        if (block % tile != 0) continue;
        const double cost = (double)(rounds * tile) * tile_weight(c, kVariants[c][v].R, es, rounds);
        if (cost < best_cost - 1e-9) {
            best = v;
            best_cost = cost;
        }
    }
    return best;
}
// ... for a list of nwork blocks, or for one job of single_n rows if that is not 0
int auto_variant_of(int c, int es, int nwork, int single_n) {
    const int unit = kUnit[es == 8][c];
    return single_n ? auto_variant(c, single_n, es, 0) : auto_variant(c, (long)nwork * unit, es, unit);
}

template <typename T, int R, int SG, int U>
void launch_gemv(const MvDev* jobs, const SysDev* sys, const int2* work, int unit, int sub, unsigned grid,
                 const MvDev* one, hipStream_t st) {
    if (one) hipLaunchKernelGGL((k_gemv1<T, R, SG, U>), dim3(grid), dim3(kThreads), 0, st, *one);
    else hipLaunchKernelGGL((k_gemv<T, R, SG, U>), dim3(grid), dim3(kThreads), 0, st, jobs, sys, work, unit, sub);
}

template <typename T, int RT, int NT>
void launch_gemm(const MvDev* jobs, const SysDev* sys, const int2* work, int unit, int sub, unsigned grid,
                 const MvDev* one, hipStream_t st) {
    if (one) hipLaunchKernelGGL((k_gemm1<T, RT, NT>), dim3(grid), dim3(64 * kGemmW), 0, st, *one);
    else hipLaunchKernelGGL((k_gemm<T, RT, NT>), dim3(grid), dim3(64 * kGemmW), 0, st, jobs, sys, work, unit, sub);
}

// One class of a product: the list `work` (nwork blocks; of one job of n =
// single_n rows if that is not 0), or the job `one` by value.
template <typename T>
int launch_class(int c, const MvDev* jobs, const SysDev* sys, const int2* work, int nwork, int single_n,
                 const MvDev* one, hipStream_t st) {
    const int unit = kUnit[sizeof(T) == 8][c];
    if (one) single_n = one->n;
    int v = g_variant[sizeof(T) == 8][c];
    if (v == 0) v = auto_variant_of(c, sizeof(T), nwork, single_n);
    const Variant& V = kVariants[c][v];
    const int rows = rows_of_variant(c, v);
    const int sub = single_n ? 0 : (unit + rows - 1) / rows;
    const unsigned grid = single_n ? (single_n + rows - 1) / rows : (unsigned)nwork * sub;
#define MPA_VAR(R_, SG_, U_) \
    if (V.R == R_ && V.SG == SG_) launch_gemv<T, R_, SG_, U_>(jobs, sys, work, unit, sub, grid, one, st);
#define MPA_GEMM(RT_, NT_) \
    if (V.R == RT_ && c == NT_ + 1) launch_gemm<T, RT_, NT_>(jobs, sys, work, unit, sub, grid, one, st);
    MPA_VAR(8, 1, 2) MPA_VAR(6, 1, 2) MPA_VAR(5, 1, 2) MPA_VAR(4, 1, 2)
    MPA_VAR(3, 1, 4) MPA_VAR(2, 1, 4) MPA_VAR(1, 1, 8)
    MPA_VAR(5, 2, 2) MPA_VAR(4, 2, 2) MPA_VAR(3, 2, 2) MPA_VAR(2, 2, 4) MPA_VAR(1, 2, 4)
    MPA_GEMM(1, 1) MPA_GEMM(2, 1) MPA_GEMM(1, 2) MPA_GEMM(2, 2)
#undef MPA_VAR
#undef MPA_GEMM
    MPA_LAUNCH_CHECK();
    return MPA_OK;
}

}  // namespace

int gemv_class(int S) { return S == 1 ? 0 : (S == 2 ? 1 : (S <= 8 ? 2 : 3)); }

int gemv_row_blocks(int n, int S, int es) {
    const int unit = kUnit[es == 8][gemv_class(S)];
    return (n + unit - 1) / unit;
}

int gemv_launch(int es, const MvDev* jobs, const SysDev* sys, int2* const* work, const int* nwork,
                const int* single_n, hipStream_t st) {
    ProfScope prof(es == 8 ? 0 : 1, st);
    for (int c = 0; c < kTileClasses; c++) {
        if (!nwork[c]) continue;
        const int rc = es == 8
                           ? launch_class<double>(c, jobs, sys, work[c], nwork[c], single_n[c], nullptr, st)
                           : launch_class<float>(c, jobs, sys, work[c], nwork[c], single_n[c], nullptr, st);
        if (rc) return rc;
    }
    return MPA_OK;
}

int gemv_launch1(int es, const MvDev& J, hipStream_t st) {
    ProfScope prof(es == 8 ? 0 : 1, st);
    const int c = gemv_class(J.S);
    return es == 8 ? launch_class<double>(c, nullptr, nullptr, nullptr, 0, 0, &J, st)
                   : launch_class<float>(c, nullptr, nullptr, nullptr, 0, 0, &J, st);
}

}  // namespace mpa

using namespace mpa;

extern "C" int mpa_matvec(int n, int nrhs, int dtype, const void* A, int add_identity, const void* x, void* y,
                          void* stream) {
    if (n < 1 || nrhs < 1 || !A || !x || !y || (n & 1)) {
        mpa_set_error("matvec: bad argument (n must be even and positive)");
        return MPA_ERR_ARG;
    }
    if (dtype != MPA_C128 && dtype != MPA_C64) {
        mpa_set_error("matvec: unknown dtype %d", dtype);
        return MPA_ERR_ARG;
    }
    MvDev J{A, x, y, n, nrhs, add_identity, -1};
    return gemv_launch1(dtype == MPA_C128 ? 8 : 4, J, (hipStream_t)stream);
}

// Autotuner: time every tile variant of the class of `nrhs` on the caller's
// operands (y is overwritten), keep the fastest for (dtype, class).
extern "C" int mpa_autotune_matvec(int n, int nrhs, int dtype, const void* A, const void* x, void* y, int reps,
                                   int* variant_out, double* ms_out, void* stream) {
    if (n < 2 || (n & 1) || nrhs < 1 || !A || !x || !y || reps < 1 || (dtype != MPA_C128 && dtype != MPA_C64)) {
        mpa_set_error("autotune_matvec: bad argument");
        return MPA_ERR_ARG;
    }
    const int es = dtype == MPA_C128 ? 8 : 4;
    const int c = gemv_class(nrhs);
    hipStream_t st = (hipStream_t)stream;
    MvDev J{A, x, y, n, nrhs, 0, -1};
    hipEvent_t e0, e1;
    MPA_HIP_CHECK(hipEventCreate(&e0));
    MPA_HIP_CHECK(hipEventCreate(&e1));
    int best = 0;
    double best_ms = 1e30;
    const int saved = g_variant[es == 8][c];
    int rc = MPA_OK;
    for (int v = 0; v < nvariants(c) && rc == MPA_OK; v++) {
        g_variant[es == 8][c] = v;
        rc = gemv_launch1(es, J, st);  // warm-up
        if (rc) break;
        (void)hipEventRecord(e0, st);
        for (int r = 0; r < reps && rc == MPA_OK; r++) rc = gemv_launch1(es, J, st);
        (void)hipEventRecord(e1, st);
        if (hipEventSynchronize(e1) != hipSuccess) rc = MPA_ERR_HIP;
        float ms = 0;
        if (rc == MPA_OK && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = MPA_ERR_HIP;
        if (rc == MPA_OK && ms / reps < best_ms) {
            best_ms = ms / reps;
            best = v;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    g_variant[es == 8][c] = rc == MPA_OK ? best : saved;
    if (rc) return rc;
    if (variant_out) *variant_out = best;
    if (ms_out) *ms_out = best_ms;
    return MPA_OK;
}

// Batched autotuner: every variant of the class of nrhs[0] timed on the
// batched launch over all systems of that class (the launch shape of the
// solvers: one workgroup per (system, row block)), the fastest kept.
extern "C" int mpa_autotune_matvec_batched(int count, const int* n, const int* nrhs, int dtype, const void* const* A,
                                           const void* const* x, void* const* y, int reps, int* variant_out,
                                           double* ms_out, void* stream) {
    if (count < 1 || !n || !nrhs || !A || !x || !y || reps < 1 || (dtype != MPA_C128 && dtype != MPA_C64)) {
        mpa_set_error("autotune_matvec_batched: bad argument");
        return MPA_ERR_ARG;
    }
    const int es = dtype == MPA_C128 ? 8 : 4;
    const int c = gemv_class(nrhs[0] < 1 ? 1 : nrhs[0]);
    std::vector<MvDev> jobs;
    for (int i = 0; i < count; i++) {
        if (n[i] < 2 || (n[i] & 1) || nrhs[i] < 1 || !A[i] || !x[i] || !y[i]) {
            mpa_set_error("autotune_matvec_batched: bad system %d", i);
            return MPA_ERR_ARG;
        }
        if (gemv_class(nrhs[i]) == c) jobs.push_back(MvDev{A[i], x[i], y[i], n[i], nrhs[i], 0, -1});
    }
    const int nv = nvariants(c);
    std::vector<int2> work;
    for (int j = 0; j < (int)jobs.size(); j++)
        for (int b = 0; b < gemv_row_blocks(jobs[j].n, jobs[j].S, es); b++) work.push_back(make_int2(j, b));
    order_work_longest_first(work, [&](int j) { return jobs[j].n; });  // as the solvers order it
    hipStream_t st = (hipStream_t)stream;
    MvDev* d_jobs = nullptr;
    int2* d_work = nullptr;
    MPA_HIP_CHECK(hipMalloc(&d_jobs, sizeof(MvDev) * jobs.size()));
    if (hipMalloc(&d_work, sizeof(int2) * work.size()) != hipSuccess) {
        (void)hipFree(d_jobs);
        mpa_set_error("autotune_matvec_batched: out of device memory");
        return MPA_ERR_OOM;
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = MPA_OK;
    if (hipMemcpyAsync(d_jobs, jobs.data(), sizeof(MvDev) * jobs.size(), hipMemcpyHostToDevice, st) != hipSuccess ||
        hipMemcpyAsync(d_work, work.data(), sizeof(int2) * work.size(), hipMemcpyHostToDevice, st) != hipSuccess ||
        hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
        rc = MPA_ERR_HIP;
    const int saved = g_variant[es == 8][c];
    int best = saved;
    double best_ms = 1e30;
    for (int v = 0; v < nv && rc == MPA_OK; v++) {
        g_variant[es == 8][c] = v;
        int2* wl[kTileClasses] = {nullptr, nullptr, nullptr, nullptr};
        int nw[kTileClasses] = {0, 0, 0, 0}, single[kTileClasses] = {0, 0, 0, 0};
        wl[c] = d_work;
        nw[c] = (int)work.size();
        single[c] = jobs.size() == 1 ? jobs[0].n : 0;
        rc = gemv_launch(es, d_jobs, nullptr, wl, nw, single, st);  // warm-up
        if (rc) break;
        (void)hipEventRecord(e0, st);
        for (int r = 0; r < reps && rc == MPA_OK; r++) rc = gemv_launch(es, d_jobs, nullptr, wl, nw, single, st);
        (void)hipEventRecord(e1, st);
        if (hipEventSynchronize(e1) != hipSuccess) rc = MPA_ERR_HIP;
        float ms = 0;
        if (rc == MPA_OK && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = MPA_ERR_HIP;
        if (rc == MPA_OK && ms / reps < best_ms) {
            best_ms = ms / reps;
            best = v;
        }
    }
    (void)hipStreamSynchronize(st);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(d_work);
    (void)hipFree(d_jobs);
    g_variant[es == 8][c] = rc == MPA_OK ? best : saved;
    if (rc) return rc;
    if (variant_out) *variant_out = best;
    if (ms_out) *ms_out = best_ms;
    return MPA_OK;
}

extern "C" int mpa_matvec_variant(int dtype, int nrhs, int set_to) {
    if (dtype != MPA_C128 && dtype != MPA_C64) return -1;
    const int c = gemv_class(nrhs < 1 ? 1 : nrhs);
    int& v = g_variant[dtype == MPA_C128][c];
    if (set_to >= 0 && set_to < nvariants(c)) v = set_to;
    return v;
}

extern "C" const char* mpa_matvec_variant_name(int dtype, int nrhs, int variant) {
    const int c = gemv_class(nrhs < 1 ? 1 : nrhs);
    if (variant < 0 || variant >= nvariants(c) || (dtype != MPA_C128 && dtype != MPA_C64)) return "";
    return kVariants[c][variant].name;
}

// Rows of a workgroup's tile that the size rule takes for a list of nwork
// blocks, or for one job of single_n rows (not part of the public interface).
extern "C" int mpa_internal_matvec_tile(int dtype, int nrhs, int nwork, int single_n) {
    const int c = gemv_class(nrhs);
    return rows_of_variant(c, auto_variant_of(c, dtype == MPA_C128 ? 8 : 4, nwork, single_n));
}

// Plain 16-byte copy of `bytes` (a multiple of 16): the reference point for
// scaling hardware byte counters (FETCH_SIZE / WRITE_SIZE) to HBM bytes.
__global__ __launch_bounds__(kThreads) void k_copy16(size_t nchunks, const dvec2* __restrict__ src,
                                                     dvec2* __restrict__ dst) {
    for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < nchunks; i += (size_t)gridDim.x * kThreads)
        __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
}

extern "C" int mpa_stream_copy(const void* src, void* dst, size_t bytes, void* stream) {
    if (!src || !dst || bytes % 16) {
        mpa_set_error("stream_copy: bad argument");
        return MPA_ERR_ARG;
    }
    hipLaunchKernelGGL(k_copy16, dim3(8192), dim3(kThreads), 0, (hipStream_t)stream, bytes / 16, (const dvec2*)src,
                       (dvec2*)dst);
    MPA_LAUNCH_CHECK();
    return MPA_OK;
}
