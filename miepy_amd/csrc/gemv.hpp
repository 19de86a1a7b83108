// Batched complex matvec y = (I +) A x over many systems, S RHS each.
//
// The system matrix is read from HBM once per pass: one pass for up to 8
// right-hand sides, one per 16 beyond.  It is not reused within a call, so it is
// streamed past the caches, which hold x (not by matrix-core tiles over rows
// that are no whole 128-byte lines).  One or two right-hand sides run on the
// vector units, a wave owning R consecutive rows; three and more run on the
// matrix cores, a workgroup owning 16 or 32 rows whose columns its waves split.
// Jobs whose system has converged for all right-hand sides
// return before touching the matrix.
#pragma once

#include <algorithm>
#include <vector>

#include "krylov.hpp"

namespace mpa {

// Tile classes: systems are grouped by RHS count so that every launch uses
// one kernel instance: class 0 (S = 1), 1 (S = 2), 2 (S = 3..8, one MFMA
// column tile), 3 (S >= 9, two).  The tile is chosen per launch by size; the
// autotuner (mpa_autotune_matvec) may fix one per (element type, class).
// Matrix cores from S = 3 on (n = 9648, c64 / c128): S = 4 126 / 250 us
// against 155 / 317 us for a vector tile of 4 right-hand sides, S = 8 133 / 262
// against 312 / 627 us in two such passes.
constexpr int kTileClasses = 4;
int gemv_class(int S);
// row blocks of a work list for an n-row system with S right-hand sides
// (element size es: 8 c128, 4 c64); independent of the tile in use
int gemv_row_blocks(int n, int S, int es);

// Batched matvec: one launch per non-empty class over its (job, row block)
// work list.  `sys` may be null when no job has skip >= 0.
// single_n[c]: the rows of the only job of class c's list, or 0 if it has several jobs.
int gemv_launch(int es, const MvDev* jobs, const SysDev* sys, int2* const* work, const int* nwork,
                const int* single_n, hipStream_t st);

// A batched GEMM's work list (job, row block) with the longest rows first
// (len(job) = its row length): workgroups over big matrices start early and
// those over small ones fill the tail.  Row blocks of one job keep their order.
// (batch256's FP64 batch: the c128 GEMM 396 -> 371-384 ms per step.)
template <class F>
inline void order_work_longest_first(std::vector<int2>& mw, F len) {
    std::stable_sort(mw.begin(), mw.end(), [&](const int2& a, const int2& b) { return len(a.x) > len(b.x); });
}
// The rows of a work list's only job (rows(job)), or 0 if it names several.
template <class F>
inline int single_job_rows(const std::vector<int2>& mw, F rows) {
    for (const int2& e : mw)
        if (e.x != mw[0].x) return 0;
    return mw.empty() ? 0 : rows(mw[0].x);
}
// One job without device-side descriptors.
int gemv_launch1(int es, const MvDev& J, hipStream_t st);

}  // namespace mpa
