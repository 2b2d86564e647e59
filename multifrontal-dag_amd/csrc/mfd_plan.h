// Task descriptors shared by the host scheduler (mfd_runtime.hip) and the
// device kernels (mfd_kernels.hip).  Every launch of the numeric schedule
// processes a contiguous range of one descriptor array that is built once per
// analysis and kept in device memory.
#pragma once
#include <cstdint>

namespace mfd {

constexpr int kTile = 64;        // edge of every front tile a workgroup owns
constexpr int kPanel = 64;       // pivot columns per panel step of a large front
constexpr int kSmallFront = 64;  // fronts up to this order are factored whole in LDS

// One front (supernode).  The front is an n x n column-major block (ld = n)
// in the front pool; its lower part holds, after factorization, L in the
// first c columns and the update matrix (Schur complement) in the trailing
// w x w block.
struct NodeDev {
    int64_t front;   // element offset of the front in the pool
    int64_t lidx;    // offset of this node's local_index (w entries) in the lidx array
    int64_t inv;     // element offset (in the pool) of the inverses of the 64 x 64 diagonal blocks
    int n, c, w;
    int parent;      // 0-based parent node, -1 for a root
    int first;       // 0-based first global (postordered) column
    int pad;
};

// kFillCols columns of a front from j0 on, zeroed, then the assembly entries
// [e0, e1) of those columns put in place.
constexpr int kFillCols = 16;
struct FillTask {
    int node, j0;
    int64_t e0, e1;
};

// The children of `node` in the bottom of the tree, entries [child, child +
// nchild) of the list of them, added into its columns [j0, j0 + kPullCols).
constexpr int kPullCols = 32;
struct PullTask {
    int node, j0, child, nchild;
};

// Extend-add of one 64 x 64 tile (ti >= tj) of child's update matrix.
struct ExtTask {
    int child, ti, tj, pad;
};

// Diagonal block [k0, k0+kb) of a large front, to be factored and
// inverted.  kprev = 0: all its updates are done.  kprev > 0: the block
// still needs the previous panel (the kprev columns to its left, block s)
// and, with kpp > 0, the kpp columns before those (panels no in-panel
// update has applied yet); the factorizing workgroup also forms the
// panel-s entries of its own rows (their TRSM with block s's inverse) and
// stores them.
// The kpp pending columns have been applied to the block itself (by the
// previous step's TRSM tile of its rows, GemmTask::syrk); the task applies
// them to its rows of block s.  The front's fields are those of its NodeDev
// (one load less before the operands'), inv the block's own inverse.
struct DiagTask {
    int64_t front, inv;
    int node, n, first;
    int k0, kb, kprev, kpp, pad;
};

// Superblocks: the solves step over 256-column superblocks u (columns B_u) of
// a front.  Fronts with many pivot columns ("super") do so through three 256
// x 256 matrices per superblock (column-major, in a separate array at xoff):
// X, the inverse of the superblock's diagonal block (zero past its width);
// at xoff + 256^2 W = X L[B_u, B_{u-1}] (u >= 1, forward); at xoff + 2 256^2
// V = L[B_{u+1}, B_u] X (B_{u+1} not empty, backward).  The others solve a
// superblock by one workgroup through the stored inverses of its 64 x 64
// diagonal blocks.
constexpr int kSuper = 256;
constexpr int64_t kSuperMats = 3 * (int64_t)kSuper * kSuper;  // entries per superblock

// A workgroup's turn in the solves (mfd_solve.hip; built by
// mfd_solve_plan.cpp).  Forward: kFwdRows / kFwdRows64, nr (<= 16 / 64) front
// rows from r0, superblocks v < nslot applied to them, sig raised; kFwdTop,
// rows r0 .. r0 + 15 of superblock u (super fronts); kFwdPiv, superblock u
// (other fronts) and then, nr > 0, the front's nr update rows, sig raised.
// Backward: kBwdPart, partial sums of the 32 columns from column nslot over
// nr rows from r0, to plane offset slot, sig raised; kBwdCols, nr
// (<= 16) columns r0 .. of superblock u, superblocks v >= grow applied to
// them, sig raised; kBwdTop, columns r0 .. r0 + 15 of superblock u; kBwdPiv,
// superblock u, before it (nr > 0) the front's nr update rows.  In kBwdCols,
// kBwdTop and kBwdPiv, nslot chunks of partial sums per 64 columns lie at
// slot.  Every task waits for counter w0 to reach w0t (w0 < 0: for nothing)
// and for the y_v (x_v) it takes up.
enum SolveKind { kFwdRows, kFwdRows64, kFwdTop, kFwdPiv, kBwdPart, kBwdCols, kBwdTop, kBwdPiv };
struct SolveTask {
    int64_t front;  // element offset of the front in the pool
    int64_t aux;    // kFwdTop, kBwdTop: superblock u's matrices; kFwdPiv, kBwdPiv: inverse of its first 64 x 64 block
    int n, c, first;  // the front; its 0-based first global column
    int z;            // front row i lies at z + i of a right-hand side's plane
    int kind, u, r0, nr;
    int goff;         // the front's gather table (gat[goff + i], row i; < 0: no children)
    int grow;         // its update rows' global rows (backward), or the first superblock of kBwdCols
    int slot, nslot;
    int w0, w0t, sig;
    int flag, fstr;   // the front's counters: asm, then z, y, p, t, x of each superblock, fstr apart; 0: one for all
    int nsup, super;  // superblocks; 1: super front
    int per;          // turns the next ticket of the workgroup takes
};
// Words before the counters in the solve's control array: the two tickets
// (whole solve or forward part; backward part), the stop word, after it the
// bound of a wait.
constexpr int kSolveTicket = 0, kSolveTicketBwd = 16, kSolveStop = 32, kSolveCtl = 64;

// Part of superblock u's matrices.  k_superinv: columns [16 j, 16 j + 16) of
// X (i unused).  k_superwv: 64 x 64 block (i, j - 4) of W, 4 <= j < 8, or
// block (i, j - 8) of V, j >= 8.
struct SuperInvTask {
    int node, u, i, j;
    int64_t xoff;
};

// A front of order <= kTreeFront all of whose children are such fronts
// (mfd_tree.hip): child .. child + nchild its children, aptr the panels'
// ranges of its entries of A, flag its counter of finished children, sig the
// parent's (-1: none, or the parent is no such front), per the turns the next
// ticket of the workgroup takes.
constexpr int kTreeFront = 128;
struct TreeTask {
    int64_t front, inv;  // element offsets in the pool
    int n, c, first;     // first: 0-based first global column
    int child, nchild, aptr;
    int flag, sig;
    int per, pad;
};
struct TreeChild {
    int64_t u;  // element offset of the child's update matrix
    int ld, w;
    int lidx, pad;
};

// mode 0: C (m x n tile, ldc) -= A (m x k, lda) * B (n x k, ldb)^T;
// mode 1: C = A B^T with B stored transposed (B[j][k] at b + j * ldb + k);
// A may be C itself: the panel TRSM X = P L^{-T}, with b the stored L^{-T}
// (column-major), whose transpose is L^{-1};
// mode 2: C = (C - A B^T) D^T with D = L^{-1} stored transposed at d
// (ld 64) and K = kd: the panel TRSM preceded by the previous panel's
// update of the same rows;
// mode 3: mode 0, and each updated entry also added into the parent front
// at p (order np) at the rows and columns local_index gives (lidx offsets
// li for the tile's rows, lj for its columns): the Schur update with the
// extend-add of its result.  Offsets are into the front pool; tri != 0
// keeps only the lower triangle (row >= col) of C.
// syrk > 0 (a TRSM tile, modes 1 and 2, whose rows are the next pivot block
// but one): afterwards the lower syrk x syrk part of the diagonal block at
// cd (ld ldc) loses R R^T, R the tile's rows over every column from A to the
// end of C (the pending panels and the panel just solved), so that the
// diagonal task of the next step finds them applied.
struct GemmTask {
    int64_t c, a, b, d, p;
    int ldc, lda, ldb;
    int m, n, k;
    int tri, mode;
    int kd, np, li, lj;
    int syrk, pad;
    int64_t cd;
};

// A run of K of one 128 x 128 tile: GEMM task `task`, K columns [k0, k1);
// slot < 0: the whole K, applied at once; otherwise its partial product goes
// to partial-product slot `slot`.
struct SegTask {
    int task, k0, k1, slot;
};
// A tile whose K was split: its partial products in slots slot0 .. slot0 +
// nslot - 1, in K order.
struct FixTask {
    int task, slot0, nslot, pad;
};

}  // namespace mfd
