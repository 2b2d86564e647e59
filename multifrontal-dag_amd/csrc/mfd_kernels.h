// Host-side launchers of the numeric kernels (mfd_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "mfd_plan.h"

namespace mfd {

// Zero fronts with A's entries in place (see k_assemble); scale: the 16-bit
// forms' diagonal scaling, or null.
template <typename T>
void launch_assemble(T* pool, const NodeDev* nodes, const FillTask* tasks, int count, const double* a,
                     const int64_t* dst, const int64_t* src, const int2* rc, const double* scale, hipStream_t st);
// Diagonal scaling of the 16-bit forms (powers of two: S A S is exact):
// s[j] from A(j,j) = a[diag_src[j]] so that s_j^2 A(j,j) lies in [0.5, 2);
// out = diag(s) in per right-hand side.
void launch_diag_scale(double* s, const double* a, const int64_t* diag_src, int n, hipStream_t st);
void launch_scale_rows(double* out, const double* in, const double* s, int n, int nrhs, hipStream_t st);
template <typename T>
void launch_extend_add(T* pool, const int* lidx, const NodeDev* nodes, const ExtTask* tasks, int count, hipStream_t st);
template <typename T>
void launch_pull_children(T* pool, const int* lidx, const NodeDev* nodes, const PullTask* tasks, int count,
                          const int* children, hipStream_t st);
template <typename T>
void launch_small_front(T* pool, const NodeDev* nodes, const int* tasks, int count, int* info, hipStream_t st);
// Medium fronts: the whole partial factorization of one front per
// workgroup (tasks: node ids); lowp as for launch_gemm's update tiles;
// clocks (nullable): start and end wall_clock64 per task.
template <typename T>
void launch_front_wg(T* pool, const NodeDev* nodes, const int* tasks, int count, int* info, long long* clocks,
                     hipStream_t st, int lowp = 0);
template <typename T>
void launch_diag(T* pool, const DiagTask* tasks, int count, int* info, hipStream_t st);
template <typename T>
void launch_upd_diag(T* pool, const DiagTask* diags, int ndiag, const GemmTask* tiles, int ntiles,
                     int* info, hipStream_t st);
// kind 0: panel TRSM tiles; 1: in-panel update; 2: Schur update (mode 3
// tiles read local_index from lidx).  lowp (FP32 fronts, kinds 1 and 2): 1
// multiplies FP16-rounded operands, 2 BF16-rounded ones, on the 16-bit MFMA
// with FP32 accumulation; 0 the front's own precision.
template <typename T>
void launch_gemm(T* pool, const GemmTask* tasks, int count, int kind, const int* lidx, hipStream_t st, int lowp = 0);
// 128 x 128 tiles (m, n <= 128) of modes 0 and 3 with their K chunks (16
// columns) divided evenly over `groups`
// workgroups (segments [seg_ptr[w], seg_ptr[w + 1]) each), then the nfix
// tiles whose K was split summed from their partial products in part
// (16384 entries per slot).
template <typename T>
void launch_gemm_seg(T* pool, const GemmTask* tasks, const SegTask* segs, const int* seg_ptr, int groups,
                     const FixTask* fixes, int nfix, T* part, const int* lidx, hipStream_t st, int lowp = 0);
// The superblock matrices: columns of X (wv = false), then the 64 x 64 blocks
// of W and V (wv = true, MFMA tile products).
template <typename T>
void launch_superinv(const T* pool, T* sinv, const NodeDev* nodes, const SuperInvTask* tasks, int count, bool wv,
                     hipStream_t st);
// The solves (mfd_solve.hip): tasks task0 .. task0 + ntasks - 1 for every
// group of 16 right-hand sides, one ticket word per launch.
// z: planes of zs entries, one per right-hand side; b, y, x: n x nrhs.
// flags: kSolveCtl control words, then nflags counters per group, all zero
// at the start (launch_solve_reset); err: set when a wait reached its bound.
template <typename T> struct SolveArgs {
    const T* pool;
    const T* sinv;
    double* z;
    const double* b;
    double *y, *x;
    const int2* gat;
    const int *gsrc, *grow;
    const SolveTask* tasks;
    int *flags, *err;
    int64_t zs;
    int n, nrhs, ngroups, nflags, task0, ntasks, ticket;
};
// The bottom of the tree (mfd_tree.hip).  a: caller values; entry e of A is
// a[asrc[e]] at row (apos[e] & 255), panel column (apos[e] >> 8); scale (may
// be null): the 16-bit forms' diagonal scaling, (row, column) = arc[e].  flags
// as for the solves, one counter per front; err likewise.
template <typename T> struct TreeArgs {
    T* pool;
    const double* a;
    const int *apos, *asrc, *aptr;
    const int2* arc;
    const double* scale;
    const int* lidx;
    const TreeTask* tasks;
    const TreeChild* children;
    int *flags, *err, *info;
    int ntasks;
};
template <typename T> void launch_tree(const TreeArgs<T>& A, hipStream_t st);
constexpr int kRhsGroup = 16;
// Zeroes n words; polls: the bound of a wait (kWaitPolls by default).
constexpr int kWaitPolls = 1 << 23;
void launch_solve_reset(int* flags, int64_t n, int polls, hipStream_t st);
template <typename T> void launch_solve(const SolveArgs<T>& A, hipStream_t st);
void launch_set_int(int* p, int v, hipStream_t st);
void launch_residual(double* r, const double* b, const double* x, int n, int nrhs, const int* ptr, const int* col,
                     const double* val, int64_t nnz, hipStream_t st);
// val[e] = a[src[e]] (the matrix values in CSR order) and the infinity norm
// of A into out[0] (zeroed by the caller).
void launch_gather_vals(unsigned long long* out, double* val, const double* a, const int64_t* src, int n,
                        const int* ptr, int64_t nnz, hipStream_t st);
// Partials per column of the sums of squares in launch_err_norms:
// sumsq_parts(n) <= kSumParts.
constexpr int kSumParts = 256;
int sumsq_parts(int64_t n);
// The maxima of |r|, |x|, |b| and (d != nullptr) |d| per column into out
// (at 0, nrhs, 2 nrhs, 3 nrhs; zeroed by the caller) and the sums of squares
// of r and x as sumsq_parts(n) partials per column (part, then part +
// sumsq_parts(n) nrhs), in one pass.
void launch_err_norms(unsigned long long* out, double* part, const double* r, const double* x, const double* b,
                      const double* d, int64_t n, int nrhs, hipStream_t st);
void launch_axpy(double* x, const double* d, int64_t n, hipStream_t st);
void launch_zero_u64(unsigned long long* p, int n, hipStream_t st);
void launch_gather_rows(double* out, int ld_out, const double* in, int ld_in, const int* perm, int n, int nrhs,
                        hipStream_t st);
void launch_scatter_rows(double* out, int ld_out, const double* in, int ld_in, const int* perm, int n, int nrhs,
                         hipStream_t st);

}  // namespace mfd
