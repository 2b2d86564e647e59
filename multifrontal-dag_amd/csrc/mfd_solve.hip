// The supernodal triangular solves as one dependency-driven launch, written
// for gfx950 (CDNA4, wave64).
//
// Replaces (paths relative to the reference root, src/main/):
//   seq_forward   (scatter_add, TRSV, GEMV)  seq_solve/seq_forward_m.f90:14-81
//   seq_backward  (gather, GEMV, TRSV)       seq_solve/seq_backward_m.f90:14-131
//
// A sweep is a chain of a few hundred dependent, tiny products: what bounds
// it is the time from one product's result to the next one's start, not the
// 2 nnz(L) entries it reads.  One launch per step of the chain cost 8 to 14
// us a step (the launch itself 1.8, then three dependent reads -- task, front,
// operands -- before the first multiply).  Here every task of both sweeps is
// a workgroup's turn in one launch: workgroups take tickets in task order,
// load the factor entries of their task into registers, wait on a counter in
// device memory for the vectors they need, and raise a counter when their
// own result is out; a hop from one workgroup to the next measured 1.4 us
// with one producer and 3 us with sixteen.
//
// No deadlock: a task waits only for tasks earlier in the order
// (mfd_check_schedule proves it for a built schedule), tickets are handed
// out in that order by an atomic counter, and a workgroup that holds a
// ticket is running; so the earliest unfinished task is always running and
// never waits, whatever the number of resident workgroups and whatever else
// the GPU runs.  Each wait is bounded all the same (kWaitPolls): a workgroup
// that reaches the bound raises the stop word, every other wait then ends,
// and the host reports an internal error.
//
// Values passed between tasks (y, x, the update rows Z, partial sums) are
// written and read by relaxed agent-scope accesses, which meet in memory
// common to the eight XCDs; a workgroup waits for its stores' completion
// before it raises its counter.  The factor is read through the caches.
//
// Every product runs on FP64 MFMA (FP32 factors are widened as they are
// read) with 16 right-hand sides as the second operand's columns; all sums
// have a fixed order, so results do not depend on timing.
#include <hip/hip_runtime.h>

#include "mfd_device.h"
#include "mfd_kernels.h"

namespace mfd {

namespace {

constexpr int kRhs = kRhsGroup;      // right-hand sides per group: the columns of an MFMA operand

__device__ __forceinline__ d4 mma(double a, double b, d4 c) { return Mfma<double>::mma(a, b, c); }

// The vector operand of a task's products, rows of 16 right-hand sides, and
// the four waves' partial products (which take the same place once the
// operand has been read): four workgroups per CU, of which the registers allow
// three in FP64.
union SolveLds {
    double v[kSuper][kRhs + 1];
    double red[4][16][kRhs + 1];
};

// What a task knows of its launch, its right-hand-side group and its place
// in the workgroup.
template <typename T> struct Ctx {
    const SolveArgs<T>& A;
    SolveLds& S;
    int* flags;  // the group's counters
    int rb, nr;  // its right-hand sides rb .. rb + nr - 1
    int tid, lane, wv, li, g;
};

// Waits until counter f reaches target (all threads; ends with a barrier,
// after which the values the counter stands for can be read).  SLOW: polls
// every 0.4 us at most, for tasks off the chain that many workgroups run (so
// that their polls do not delay the counter's additions).
template <typename T, bool SLOW = false>
__device__ __forceinline__ void wait_for(const Ctx<T>& C, int f, int target)
{
    if (f >= 0 && C.tid == 0) poll<SLOW>(C.flags + f, target, C.A.flags + kSolveStop, C.A.err);
    __syncthreads();
}
// Raises counters f and f2 (negative: none) once every store of the
// workgroup has completed (all threads; holds a barrier).
template <typename T> __device__ __forceinline__ void signal(const Ctx<T>& C, int f, int f2 = -1)
{
    stores_done();
    __syncthreads();
    if (C.tid == 0) {
        if (f >= 0) add_agent(C.flags + f, 1);
        if (f2 >= 0) add_agent(C.flags + f2, 1);
    }
}

// Counters of a front (SolveTask::flag, fstr): y_u and x_u of superblock u; of
// a front that has one for all (fstr 0), that one.
__device__ __forceinline__ int y_flag(const SolveTask& t, int u) { return t.flag + t.fstr * (1 + t.nsup + u); }
__device__ __forceinline__ int x_flag(const SolveTask& t, int u) { return t.flag + t.fstr * (1 + 4 * t.nsup + u); }
// Tasks that form superblock u's y (or x).
__device__ __forceinline__ int yx_target(const SolveTask& t, int u)
{
    return t.super ? (min(kSuper, t.c - kSuper * u) + 15) / 16 : 1;
}
// What the y counter has reached before those tasks: where it counts the
// children's signals too, w0t, which a task on the front's rows waits for.
__device__ __forceinline__ int before_y(const SolveTask& t) { return t.fstr == 0 ? t.w0t : 0; }

// S.v[k][r] = src[k + (rb + r) ld] for k < cnt, zero for the other k < 256
// (thread k's row; all loads before the stores of four columns).
template <typename T>
__device__ __forceinline__ void stage_rows(const Ctx<T>& C, const double* src, int64_t ld, int cnt)
{
    const int k = C.tid;
    for (int r = 0; r < C.nr; r += 4) {
        double q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            q[i] = (k < cnt && r + i < C.nr) ? ld_agent(src + k + (int64_t)(C.rb + r + i) * ld) : 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (r + i < C.nr) C.S.v[k][r + i] = q[i];
    }
}

// The children's contributions to row i of a front, in child order: table
// entry gat[goff + i] holds the plane positions of the first and the second
// (-1: none), or, where there are more, -2 - k with the list of the second
// and the others at gsrc[k] (their number, then their positions); goff < 0:
// a leaf.  Read before the wait for the children.
template <typename T> __device__ __forceinline__ int2 gather_at(const Ctx<T>& C, const SolveTask& t, int i)
{
    return t.goff < 0 ? make_int2(-1, -1) : C.A.gat[t.goff + i];
}
template <typename T> __device__ __forceinline__ double gather_list(const Ctx<T>& C, int y, int rhs, double v)
{
    const int* p = C.A.gsrc + (-2 - y);
    for (int k = 1; k <= p[0]; ++k) v += ld_agent(C.A.z + (int64_t)rhs * C.A.zs + p[k]);
    return v;
}
// Four right-hand-side entries of a front, entry e that of row i[e] (gather
// entry q[e]), column rhs[e] (live[e] false: zero): b on pivot rows, plus the
// children's contributions (scatter_add, sparse_add_subroutines_m.f90:13-30).
// begin issues the loads, end adds them up.
struct Gather4 {
    double b[4], c0[4], c1[4];
};
template <typename T>
__device__ __forceinline__ void gather_begin(const Ctx<T>& C, const SolveTask& t, const int2 (&q)[4], const int (&i)[4],
                                             const int (&rhs)[4], const bool (&live)[4], Gather4& v)
{
#pragma unroll
    for (int e = 0; e < 4; ++e)
        v.b[e] = (live[e] && i[e] < t.c) ? C.A.b[t.first + i[e] + (int64_t)rhs[e] * C.A.n] : 0.0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const double* Z = C.A.z + (int64_t)rhs[e] * C.A.zs;
        v.c0[e] = (live[e] && q[e].x >= 0) ? ld_agent(Z + q[e].x) : 0.0;
        v.c1[e] = (live[e] && q[e].y >= 0) ? ld_agent(Z + q[e].y) : 0.0;
    }
}
template <typename T>
__device__ __forceinline__ void gather_end(const Ctx<T>& C, const int2 (&q)[4], const int (&rhs)[4],
                                           const bool (&live)[4], const Gather4& v, double (&z)[4])
{
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        z[e] = v.b[e] + v.c0[e] + v.c1[e];
        if (live[e] && q[e].y < -1) z[e] = gather_list(C, q[e].y, rhs[e], z[e]);
    }
}

// 64 entries of K for 16 rows of column-major M (uniform address): lane (row
// `row`, column k0 + 4 j + g), j < 16 -- 16 consecutive rows of four columns
// per load.  cmax: the last column read.
template <typename T>
__device__ __forceinline__ void load_cols(T (&a)[16], const T* M, int row, int ld, int k0, int g, int cmax)
{
#pragma unroll
    for (int j = 0; j < 16; ++j) a[j] = ld_off(M, (unsigned)(row + min(k0 + 4 * j + g, cmax) * ld));
}
// acc += sum over j < 16 of a[j] b(j), four entries of K each, in N chains
// added pairwise and then to acc.  In one chain through all of a task's entries
// (up to 256) every product rounds at the whole sum's magnitude: over 240
// systems the backward error of an FP64 solve was 7% larger than with sums of
// 16 to 64 entries (16% on a 12^3 27-point stencil), and is 2% larger with
// these.  Four chains in the tasks that run on 16 rows or columns; two in the
// block tasks (kFwdPiv, kBwdPiv), whose three tiles in flight leave no
// registers for more (solves 5 to 15% slower at four).  One with an FP32
// factor, whose own rounding is 2^29 times that of these sums.
template <int N64, typename T, typename B> __device__ __forceinline__ void mma_chains(d4& acc, const T (&a)[16], B b)
{
    constexpr int N = sizeof(T) == 8 ? N64 : 1;
    static_assert(N == 1 || N == 2 || N == 4, "added pairwise");
    if constexpr (N == 1) {
#pragma unroll
        for (int j = 0; j < 16; ++j) acc = mma((double)a[j], b(j), acc);
        return;
    }
    d4 p[N];
#pragma unroll
    for (int j = 0; j < N; ++j) p[j] = d4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 16; ++j) p[j % N] = mma((double)a[j], b(j), p[j % N]);
    if constexpr (N == 4)
        acc += (p[0] + p[1]) + (p[2] + p[3]);
    else
        acc += p[0] + p[1];
}
// acc += a S.v[k0 ..] in load_cols's order.
template <int N = 4, typename T> __device__ __forceinline__ void mma_cols(d4& acc, const T (&a)[16], const Ctx<T>& C, int k0)
{
    const bool ok = C.li < C.nr;
    const int r = ok ? C.li : 0;
    mma_chains<N>(acc, a, [&](int j) {
        const double b = C.S.v[k0 + 4 * j + C.g][r];
        return ok ? b : 0.0;
    });
}

// 64 entries of K for 16 columns of column-major M (the transposed
// product): lane (column li) reads 16-byte pieces of its column, the four
// lanes of a column consecutive ones: rows row_of(j, g).
template <typename T> struct Piece;
template <> struct Piece<double> {
    typedef double vec __attribute__((ext_vector_type(2), aligned(8)));
    static constexpr int V = 2;
};
template <> struct Piece<float> {
    typedef float vec __attribute__((ext_vector_type(4), aligned(4)));
    static constexpr int V = 4;
};
template <typename T> __device__ __forceinline__ int row_of(int j, int g)
{
    constexpr int V = Piece<T>::V;
    return 4 * V * (j / V) + V * g + j % V;
}
// M: uniform address; col: the lane's offset from it at the product's first
// row; rows past lim give 0 (a piece that crosses lim is read whole: it lies
// inside the pool, whose stored inverses follow the fronts).
template <typename T>
__device__ __forceinline__ void load_rows(T (&a)[16], const T* M, int col, int r0, int g, int lim)
{
    constexpr int V = Piece<T>::V;
    typedef typename Piece<T>::vec vec;
#pragma unroll
    for (int j = 0; j < 16; j += V) {
        const int r = r0 + row_of<T>(j, g);
        const unsigned at = (unsigned)(col + (r < lim ? r : 0));
        const vec p = *reinterpret_cast<const vec*>(reinterpret_cast<const char*>(M) + (size_t)(at * (unsigned)sizeof(T)));
#pragma unroll
        for (int e = 0; e < V; ++e) a[j + e] = r + e < lim ? p[e] : T(0);
    }
}
template <int N = 4, typename T> __device__ __forceinline__ void mma_rows(d4& acc, const T (&a)[16], const Ctx<T>& C, int k0)
{
    const bool ok = C.li < C.nr;
    const int r = ok ? C.li : 0;
    mma_chains<N>(acc, a, [&](int j) {
        const double b = C.S.v[k0 + row_of<T>(j, C.g)][r];
        return ok ? b : 0.0;
    });
}

// The four waves' partial products added in wave order: thread (row tid /
// 16, right-hand side tid % 16) returns its entry.
template <typename T> __device__ __forceinline__ double reduce_waves(const Ctx<T>& C, d4 acc)
{
    __syncthreads();  // S.v has been read
#pragma unroll
    for (int v = 0; v < 4; ++v) C.S.red[C.wv][C.g + 4 * v][C.li] = acc[v];
    __syncthreads();
    const int row = C.tid >> 4, rhs = C.tid & 15;
    return (C.S.red[0][row][rhs] + C.S.red[1][row][rhs]) + (C.S.red[2][row][rhs] + C.S.red[3][row][rhs]);
}

// ---------------------------------------------------------------- forward
// 16 rows of a front (kFwdRows): z = their right-hand side - sum over
// superblocks v < nv of L[rows, B_v] y_v as the y_v come out, each wave a
// quarter of B_v's columns.
template <typename T> __device__ __forceinline__ void fwd_rows(const Ctx<T>& C, const SolveTask& t)
{
    const T* F = C.A.pool + t.front;
    const int nv = t.nslot, lrow = min(t.r0 + C.li, t.n - 1);
    auto load = [&](T(&a)[16], int v) {
        load_cols<T>(a, F + (int64_t)kSuper * v * t.n, lrow, t.n, 64 * C.wv, C.g, min(kSuper, t.c - kSuper * v) - 1);
    };
    T a[16], an[16];
    if (nv > 0) load(a, 0);
    const int row = C.tid >> 4, rhs = C.tid & 15, i = t.r0 + row;
    const bool live = row < t.nr && rhs < C.nr;
    const int2 q = gather_at(C, t, live ? i : t.r0);
    wait_for(C, t.w0, t.w0t);
    double z = 0.0;
    if (live) {
        const double* Z = C.A.z + (int64_t)(C.rb + rhs) * C.A.zs;
        const double bv = i < t.c ? C.A.b[t.first + i + (int64_t)(C.rb + rhs) * C.A.n] : 0.0;
        const double c0 = q.x >= 0 ? ld_agent(Z + q.x) : 0.0;
        const double c1 = q.y >= 0 ? ld_agent(Z + q.y) : 0.0;
        z = bv + c0 + c1;
        if (q.y < -1) z = gather_list(C, q.y, C.rb + rhs, z);
    }
    d4 acc = {0, 0, 0, 0};
    for (int v = 0; v < nv; ++v) {
        wait_for<T, true>(C, y_flag(t, v), before_y(t) + yx_target(t, v));
        stage_rows(C, C.A.y + t.first + kSuper * v, C.A.n, min(kSuper, t.c - kSuper * v));
        __syncthreads();
        if (v + 1 < nv) load(an, v + 1);
        mma_cols(acc, a, C, 64 * C.wv);
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = an[j];
    }
    const double s = reduce_waves(C, acc);
    if (live) st_agent(C.A.z + (int64_t)(C.rb + rhs) * C.A.zs + t.z + i, z - s);
    signal(C, t.sig);
}

// The lane's four entries of a wave's 16 x 16 result over rows r0 + rw ..,
// nr of them from r0 on (nr <= 0: none): rows and right-hand sides.
template <typename T>
__device__ __forceinline__ void own_rows(const Ctx<T>& C, const SolveTask& t, int r0, int rw, int nr, int (&at)[4],
                                         int (&rhs)[4], bool (&live)[4])
{
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int i = rw + C.g + 4 * v;
        live[v] = i < nr && C.li < C.nr;
        at[v] = live[v] ? r0 + i : 0;
        rhs[v] = C.rb + (C.li < C.nr ? C.li : 0);
    }
}
template <typename T>
__device__ __forceinline__ void gather_rows(const Ctx<T>& C, const SolveTask& t, const int (&at)[4],
                                            const bool (&live)[4], int2 (&q)[4])
{
#pragma unroll
    for (int v = 0; v < 4; ++v) q[v] = live[v] ? gather_at(C, t, at[v]) : make_int2(-1, -1);
}

// 64 rows of a front (kFwdRows64, where rows are many): each wave 16 of
// them over all columns.
template <typename T> __device__ __forceinline__ void fwd_rows64(const Ctx<T>& C, const SolveTask& t)
{
    const int rw = 16 * C.wv, nv = t.nslot, lrow = min(t.r0 + rw + C.li, t.n - 1);
    const T* F = C.A.pool + t.front;
    auto load = [&](T(&a)[16], int k0) {
        load_cols<T>(a, F + (int64_t)k0 * t.n, lrow, t.n, 0, C.g, t.c - 1 - k0);
    };
    T a[16], an[16];
    if (nv > 0) load(a, 0);
    int2 q[4];
    int at[4], rhs[4];
    bool live[4];
    own_rows(C, t, t.r0, rw, t.nr, at, rhs, live);
    gather_rows(C, t, at, live, q);
    wait_for(C, t.w0, t.w0t);
    double z[4];
    {
        Gather4 g4;
        gather_begin(C, t, q, at, rhs, live, g4);
        gather_end(C, q, rhs, live, g4, z);
    }
    d4 acc = {0, 0, 0, 0};
    for (int v = 0; v < nv; ++v) {
        const int pb = min(kSuper, t.c - kSuper * v);
        wait_for<T, true>(C, y_flag(t, v), before_y(t) + yx_target(t, v));
        stage_rows(C, C.A.y + t.first + kSuper * v, C.A.n, pb);
        __syncthreads();
        for (int k0 = 0; k0 < pb; k0 += 64) {
            const int kn = kSuper * v + k0 + 64;
            if (kn < t.c) load(an, kn);
            mma_cols(acc, a, C, k0);
#pragma unroll
            for (int j = 0; j < 16; ++j) a[j] = an[j];
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int i = rw + C.g + 4 * v;
        if (i < t.nr && C.li < C.nr)
            st_agent(C.A.z + (int64_t)(C.rb + C.li) * C.A.zs + t.z + t.r0 + i, z[v] - acc[v]);
    }
    signal(C, t.sig);
}

// S.v = the right-hand side of superblock u's rows: gathered (u has no
// earlier superblock to take off, or only the one the caller takes off) or
// from Z, where kFwdRows tasks left it.
template <typename T> __device__ __forceinline__ void stage_z(const Ctx<T>& C, const SolveTask& t, int sb, bool gather)
{
    const int k = C.tid, i = kSuper * t.u + k;
    if (gather) {
        const int2 q = gather_at(C, t, k < sb ? i : kSuper * t.u);
        const int2 qs[4] = {q, q, q, q};
        const int at[4] = {i, i, i, i};
        wait_for(C, t.w0, t.w0t);
        for (int r = 0; r < C.nr; r += 4) {
            const int rhs[4] = {C.rb + r, C.rb + r + 1, C.rb + r + 2, C.rb + r + 3};
            const bool live[4] = {k < sb, k < sb && r + 1 < C.nr, k < sb && r + 2 < C.nr, k < sb && r + 3 < C.nr};
            double z[4];
            Gather4 g4;
            gather_begin(C, t, qs, at, rhs, live, g4);
            gather_end(C, qs, rhs, live, g4, z);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (r + e < C.nr) C.S.v[k][r + e] = z[e];
        }
    } else {
        wait_for(C, t.w0, t.w0t);
        stage_rows(C, C.A.z + t.z + kSuper * t.u, C.A.zs, sb);
    }
    __syncthreads();
}

// 16 rows of superblock u through its explicit inverse (kFwdTop): y_u =
// X z_u - W y_{u-1}, z_u holding every superblock before u - 1.
template <typename T> __device__ __forceinline__ void fwd_top(const Ctx<T>& C, const SolveTask& t)
{
    const T* X = C.A.sinv + t.aux + t.r0;
    const int sb = min(kSuper, t.c - kSuper * t.u), k0 = 64 * C.wv;
    T a[16], w[16];
    load_cols<T>(a, X, C.li, kSuper, k0, C.g, kSuper - 1);
    // (W of the first superblock is unused storage)
    load_cols<T>(w, X + kSuper * kSuper, C.li, kSuper, k0, C.g, kSuper - 1);
    stage_z(C, t, sb, t.u < 2);
    d4 acc = {0, 0, 0, 0}, accw = {0, 0, 0, 0};
    if (k0 <= t.r0) mma_cols(acc, a, C, k0);  // X is lower triangular
    if (t.u > 0) {
        wait_for(C, y_flag(t, t.u - 1), yx_target(t, t.u - 1));
        stage_rows(C, C.A.y + t.first + kSuper * (t.u - 1), C.A.n, kSuper);
        __syncthreads();
        mma_cols(accw, w, C, k0);
    }
    const double y = reduce_waves(C, acc - accw);
    const int row = C.tid >> 4, rhs = C.tid & 15;
    if (t.r0 + row < sb && rhs < C.nr)
        st_agent(C.A.y + t.first + kSuper * t.u + t.r0 + row + (int64_t)(C.rb + rhs) * C.A.n, y);
    signal(C, y_flag(t, t.u));
}

// The 64 x 64 tiles a superblock's solve takes up, in order: for each block b
// its tiles (b, j), j < b, then its inverse (j = b).  Two tiles are in flight
// ahead of the one in use (their loads wait for no barrier).
constexpr int kTiles = 10;
__device__ constexpr int kTileB[kTiles] = {0, 1, 1, 2, 2, 2, 3, 3, 3, 3};
__device__ constexpr int kTileJ[kTiles] = {0, 0, 1, 0, 1, 2, 0, 1, 2, 3};

// Superblock u by one workgroup (kFwdPiv), 64 columns at a time through the
// stored inverses of the diagonal blocks: y_b = inv(L_bb) (z_b - sum_{a<b}
// L_ba y_a).  nr > 0 (fronts of one superblock): then the front's nr update
// rows as well, Z = right-hand side - L[rows, :] y.
template <typename T> __device__ __forceinline__ void fwd_piv(const Ctx<T>& C, const SolveTask& t)
{
    const int sb = min(kSuper, t.c - kSuper * t.u), nb = (sb + 63) / 64, rw = 16 * C.wv, c0 = kSuper * t.u;
    const T* F = C.A.pool + t.front + (int64_t)c0 * t.n;  // the superblock's columns
    const bool ok = C.li < C.nr;
    T buf[3][16];
    auto fetch = [&](T(&a)[16], int b, int j) {
        if (j < b)
            load_cols<T>(a, F, min(c0 + 64 * b + rw + C.li, t.n - 1), t.n, 64 * j, C.g, sb - 1);
        else  // inv[r + 64 q] = L^{-1}(q, r): the lane's row q, 16-byte pieces along r
            load_rows<T>(a, C.A.pool + t.aux + b * 4096, 64 * (rw + C.li), 0, C.g, 64);
    };
    fetch(buf[0], 0, 0);
    if (nb > 1) fetch(buf[1], 1, 0);
    int2 qr[4];  // the first update rows' gather entries
    {
        int at[4], rhs[4];
        bool live[4];
        own_rows(C, t, t.c, rw, t.nr, at, rhs, live);
        gather_rows(C, t, at, live, qr);
    }
    stage_z(C, t, sb, t.u == 0);
    d4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < kTiles; ++q) {
        const int b = kTileB[q], j = kTileJ[q];
        if (b < nb) {
            if (q + 2 < kTiles && kTileB[q + 2] < nb) fetch(buf[(q + 2) % 3], kTileB[q + 2], kTileJ[q + 2]);
            if (j < b) {
                mma_cols<2>(acc, buf[q % 3], C, 64 * j);
                if (j == b - 1) {
                    if (ok) {
#pragma unroll
                        for (int v = 0; v < 4; ++v) C.S.v[64 * b + rw + C.g + 4 * v][C.li] -= acc[v];
                    }
                    acc = d4{0, 0, 0, 0};
                    __syncthreads();
                }
            } else {
                d4 y = {0, 0, 0, 0};
                mma_rows<2>(y, buf[q % 3], C, 64 * b);
                __syncthreads();
                if (ok) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int k = 64 * b + rw + C.g + 4 * v;
                        C.S.v[k][C.li] = k < sb ? y[v] : 0.0;
                        if (k < sb) st_agent(C.A.y + t.first + c0 + k + (int64_t)(C.rb + C.li) * C.A.n, y[v]);
                    }
                }
                __syncthreads();
            }
        }
    }
    if (t.nr > 0) {
        // tiles (64 rows, 64 columns) with the next one's entries, and the
        // next rows' gather entries, in flight
        auto rows = [&](T(&a)[16], int r0, int j) {
            load_cols<T>(a, F, min(t.c + r0 + rw + C.li, t.n - 1), t.n, 64 * j, C.g, sb - 1);
        };
        int at[4], rhs[4];
        bool live[4];
        rows(buf[0], 0, 0);
        for (int r0 = 0; r0 < t.nr; r0 += 64) {
            Gather4 g4;
            own_rows(C, t, t.c + r0, rw, t.nr - r0, at, rhs, live);
            gather_begin(C, t, qr, at, rhs, live, g4);
            int2 qn[4];
            {
                int atn[4];
                bool liven[4];
                own_rows(C, t, t.c + r0 + 64, rw, t.nr - r0 - 64, atn, rhs, liven);
                gather_rows(C, t, atn, liven, qn);
            }
            acc = d4{0, 0, 0, 0};
            for (int j = 0; j < nb; ++j) {
                const bool last = j + 1 == nb;
                if (!last || r0 + 64 < t.nr) rows(buf[1], last ? r0 + 64 : r0, last ? 0 : j + 1);
                mma_cols<2>(acc, buf[0], C, 64 * j);
#pragma unroll
                for (int e = 0; e < 16; ++e) buf[0][e] = buf[1][e];
            }
            double z[4];
            gather_end(C, qr, rhs, live, g4, z);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (live[v]) st_agent(C.A.z + (int64_t)rhs[v] * C.A.zs + t.z + at[v], z[v] - acc[v]);
                qr[v] = qn[v];
            }
        }
    }
    signal(C, y_flag(t, t.u), t.sig);
}

// --------------------------------------------------------------- backward
// S.v = x at the global rows of update rows r0 .. r0 + nr - 1 (gather,
// sparse_add_subroutines_m.f90:32-49), zero past nr; the rows' positions are
// read before the wait on counter f.
template <typename T>
__device__ __forceinline__ void stage_x(const Ctx<T>& C, const SolveTask& t, int r0, int nr, int f, int target)
{
    const int k = C.tid, at = k < nr ? C.A.grow[t.grow + (r0 - t.c) + k] : 0;
    wait_for(C, f, target);
    for (int r = 0; r < C.nr; r += 4) {
        double q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            q[i] = (k < nr && r + i < C.nr) ? ld_agent(C.A.x + at + (int64_t)(C.rb + r + i) * C.A.n) : 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (r + i < C.nr) C.S.v[k][r + i] = q[i];
    }
    __syncthreads();
}

// Partial sums (kBwdPart): L[rows, 32 columns]^T x over the task's update rows
// (first column nslot of the front) into 32 entries at slot, 256 rows at a
// time (few tasks have more); a wave takes 16 of the columns and half the
// rows, so that all entries of the first 256 rows are in registers before the
// wait for x.
template <typename T> __device__ __forceinline__ void bwd_part(const Ctx<T>& C, const SolveTask& t)
{
    const int cw = 16 * (C.wv & 1), h = 128 * (C.wv >> 1), col0 = t.nslot;
    const T* F = C.A.pool + t.front + (int64_t)col0 * t.n + t.r0;
    const int lcol = min(cw + C.li, t.c - 1 - col0) * t.n;
    T a[16], an[16];
    d4 acc = {0, 0, 0, 0};
    for (int r = 0; r < t.nr; r += kSuper) {
        load_rows<T>(a, F, lcol, r + h, C.g, t.nr);
        load_rows<T>(an, F, lcol, r + h + 64, C.g, t.nr);
        stage_x(C, t, t.r0 + r, min(kSuper, t.nr - r), r == 0 ? t.w0 : -1, t.w0t);
        mma_rows(acc, a, C, h);
        mma_rows(acc, an, C, h + 64);
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v) C.S.red[C.wv][C.g + 4 * v][C.li] = acc[v];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int k = (C.tid & 15) + 16 * e, rhs = C.tid >> 4;
        if (rhs < C.nr)
            st_agent(C.A.z + (int64_t)(C.rb + rhs) * C.A.zs + t.slot + k,
                     C.S.red[e][C.tid & 15][rhs] + C.S.red[e + 2][C.tid & 15][rhs]);
    }
    signal(C, t.sig);
}

// y of column k of superblock u, right-hand sides r .. r + 3 (below lim),
// less its partial sums, in chunk order; 16 loads in flight.
template <typename T>
__device__ __forceinline__ void y_less_parts(const Ctx<T>& C, const SolveTask& t, int k, int r, int lim, double (&v)[4])
{
    const double* Y = C.A.y + t.first + kSuper * t.u + k;
    const double* P = C.A.z + t.slot + (int64_t)64 * t.nslot * (k >> 6) + (k & 63);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = r + i < lim ? ld_agent(Y + (int64_t)(r + i) * C.A.n) : 0.0;
    for (int ch = 0; ch < t.nslot; ch += 4) {
        double q[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                q[i][e] = (r + i < lim && ch + e < t.nslot) ? ld_agent(P + (int64_t)(r + i) * C.A.zs + 64 * (ch + e)) : 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i] -= q[i][e];
    }
}

// 16 columns of superblock u (kBwdCols): y less the update rows' partial
// sums and less L[B_v, columns]^T x_v for v = nsup - 1 .. vlo as the x_v come
// out, each wave a quarter of B_v's rows; the result replaces y.
template <typename T> __device__ __forceinline__ void bwd_cols(const Ctx<T>& C, const SolveTask& t)
{
    const int col0 = kSuper * t.u + t.r0, lcol = min(C.li, t.c - 1 - col0) * t.n;
    const T* F = C.A.pool + t.front + (int64_t)col0 * t.n;
    const int vlo = t.grow, r0 = 64 * C.wv;
    auto load = [&](T(&a)[16], int v) {
        load_rows<T>(a, F + kSuper * v, lcol, r0, C.g, min(kSuper, t.c - kSuper * v));
    };
    T a[16], an[16];
    load(a, t.nsup - 1);
    const int col = C.tid >> 4, rhs = C.tid & 15;
    const bool live = col < t.nr && rhs < C.nr;
    wait_for(C, t.w0, t.w0t);
    double y[4] = {0.0, 0.0, 0.0, 0.0};
    if (live) y_less_parts(C, t, t.r0 + col, C.rb + rhs, C.rb + rhs + 1, y);
    d4 acc = {0, 0, 0, 0};
    for (int v = t.nsup - 1; v >= vlo; --v) {
        wait_for(C, x_flag(t, v), yx_target(t, v));
        stage_rows(C, C.A.x + t.first + kSuper * v, C.A.n, min(kSuper, t.c - kSuper * v));
        __syncthreads();
        if (v > vlo) load(an, v - 1);
        mma_rows(acc, a, C, r0);
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = an[j];
    }
    const double s = reduce_waves(C, acc);
    if (live) st_agent(C.A.y + t.first + kSuper * t.u + t.r0 + col + (int64_t)(C.rb + rhs) * C.A.n, y[0] - s);
    signal(C, t.sig);
}

// S.v = superblock u's y less everything after it (nslot > 0: less the
// partial sums still; otherwise kBwdCols tasks have done it all).
template <typename T> __device__ __forceinline__ void stage_t(const Ctx<T>& C, const SolveTask& t, int sb)
{
    wait_for(C, t.w0, t.w0t);
    const int k = C.tid;
    if (t.nslot > 0)
        for (int r = 0; r < C.nr; r += 4) {
            double v[4] = {0.0, 0.0, 0.0, 0.0};
            if (k < sb) y_less_parts(C, t, k, C.rb + r, C.rb + C.nr, v);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (r + i < C.nr) C.S.v[k][r + i] = v[i];
        }
    else
        stage_rows(C, C.A.y + t.first + kSuper * t.u, C.A.n, sb);
    __syncthreads();
}

// 16 rows of superblock u through its explicit inverse (kBwdTop): x_u =
// X^T t_u - V^T x_{u+1}.
template <typename T> __device__ __forceinline__ void bwd_top(const Ctx<T>& C, const SolveTask& t)
{
    const int sb = min(kSuper, t.c - kSuper * t.u), k0 = 64 * C.wv;
    const bool next = t.u + 1 < t.nsup;
    const T* X = C.A.sinv + t.aux + kSuper * t.r0;
    T a[16], w[16];
    load_rows<T>(a, X, kSuper * C.li, k0, C.g, kSuper);
    if (next) load_rows<T>(w, X + 2 * kSuper * kSuper, kSuper * C.li, k0, C.g, kSuper);
    stage_t(C, t, sb);
    d4 acc = {0, 0, 0, 0}, accv = {0, 0, 0, 0};
    if (k0 + 64 > t.r0) mma_rows(acc, a, C, k0);  // X is lower triangular
    if (next) {
        wait_for(C, x_flag(t, t.u + 1), yx_target(t, t.u + 1));
        stage_rows(C, C.A.x + t.first + kSuper * (t.u + 1), C.A.n, min(kSuper, t.c - kSuper * (t.u + 1)));
        __syncthreads();
        mma_rows(accv, w, C, k0);
    }
    const double x = reduce_waves(C, acc - accv);
    const int row = C.tid >> 4, rhs = C.tid & 15;
    if (t.r0 + row < sb && rhs < C.nr)
        st_agent(C.A.x + t.first + kSuper * t.u + t.r0 + row + (int64_t)(C.rb + rhs) * C.A.n, x);
    signal(C, x_flag(t, t.u));
}

// Superblock u by one workgroup (kBwdPiv): x_b = inv(L_bb)^T (t_b -
// sum_{a>b} L_ab^T x_a), tiles in fwd_piv's order counted from the last
// block.  nr > 0 (fronts of one superblock): the front's nr update rows
// first, t = y - L[rows, :]^T x.
template <typename T> __device__ __forceinline__ void bwd_piv(const Ctx<T>& C, const SolveTask& t)
{
    const int sb = min(kSuper, t.c - kSuper * t.u), nb = (sb + 63) / 64, cw = 16 * C.wv, c0 = kSuper * t.u;
    const T* F = C.A.pool + t.front + (int64_t)c0 * t.n;
    const bool ok = C.li < C.nr;
    T buf[3][16];
    if (t.nr > 0) {
        d4 acc[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
        auto rows = [&](T(&a)[16], int r, int b) {  // rows r .. r + 63 of the update part, column block b
            load_rows<T>(a, F + t.c, min(64 * b + cw + C.li, sb - 1) * t.n, r, C.g, t.nr);
        };
        rows(buf[0], 0, 0);
        for (int r0 = 0; r0 < t.nr; r0 += kSuper) {
            const int nr = min(kSuper, t.nr - r0);
            stage_x(C, t, t.c + r0, nr, r0 == 0 ? t.w0 : -1, t.w0t);
            for (int q = 0; q < nr; q += 64) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (b >= nb) continue;
                    const bool last = b + 1 >= nb;
                    if (!last || r0 + q + 64 < t.nr) rows(buf[1], r0 + q + (last ? 64 : 0), last ? 0 : b + 1);
                    mma_rows<2>(acc[b], buf[0], C, q);
#pragma unroll
                    for (int e = 0; e < 16; ++e) buf[0][e] = buf[1][e];
                }
            }
            __syncthreads();
        }
        const double* Y = C.A.y + t.first + (int64_t)(C.rb + (ok ? C.li : 0)) * C.A.n;
        double y[4][4];
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int k = 64 * b + cw + C.g + 4 * v;
                y[b][v] = ok && k < sb ? ld_agent(Y + k) : 0.0;
            }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if (b >= nb || !ok) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int k = 64 * b + cw + C.g + 4 * v;
                C.S.v[k][C.li] = k < sb ? y[b][v] - acc[b][v] : 0.0;
            }
        }
    }
    auto fetch = [&](T(&a)[16], int bq, int jq) {
        const int b = nb - 1 - bq, j = nb - 1 - jq;
        if (jq < bq)
            load_rows<T>(a, F + c0, (64 * b + cw + C.li) * t.n, 64 * j, C.g, sb);
        else
            load_cols<T>(a, C.A.pool + t.aux + b * 4096, cw + C.li, 64, 0, C.g, 63);
    };
    fetch(buf[0], 0, 0);
    if (nb > 1) fetch(buf[1], 1, 0);
    if (t.nr > 0)
        __syncthreads();
    else
        stage_t(C, t, sb);
    d4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < kTiles; ++q) {
        const int bq = kTileB[q], jq = kTileJ[q];
        if (bq < nb) {
            const int b = nb - 1 - bq, j = nb - 1 - jq;
            if (q + 2 < kTiles && kTileB[q + 2] < nb) fetch(buf[(q + 2) % 3], kTileB[q + 2], kTileJ[q + 2]);
            if (jq < bq) {
                mma_rows<2>(acc, buf[q % 3], C, 64 * j);
                if (jq == bq - 1) {
                    if (ok) {
#pragma unroll
                        for (int v = 0; v < 4; ++v) C.S.v[64 * b + cw + C.g + 4 * v][C.li] -= acc[v];
                    }
                    acc = d4{0, 0, 0, 0};
                    __syncthreads();
                }
            } else {
                d4 x = {0, 0, 0, 0};
                mma_cols<2>(x, buf[q % 3], C, 64 * b);
                __syncthreads();
                if (ok) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int k = 64 * b + cw + C.g + 4 * v;
                        C.S.v[k][C.li] = x[v];
                        if (k < sb) st_agent(C.A.x + t.first + c0 + k + (int64_t)(C.rb + C.li) * C.A.n, x[v]);
                    }
                }
                __syncthreads();
            }
        }
    }
    signal(C, x_flag(t, t.u));
}

}  // namespace

template <typename T> __global__ __launch_bounds__(kThreads, sizeof(T) == 8 ? 3 : 4) void k_solve(SolveArgs<T> A)
{
    __shared__ SolveLds S;
    __shared__ int ticket;
    const int tid = threadIdx.x;
    int* counter = A.flags + A.ticket;
    // a ticket: the next `per` turns (turn k: task k / ngroups for group k %
    // ngroups); per is the last task's, 1 where a level's tasks are few
    int per = 1, k0 = 0;
    for (;;) {
        if (tid == 0) ticket = add_agent(counter, per);
        __syncthreads();
        k0 = __builtin_amdgcn_readfirstlane(ticket);
        const int k1 = min(k0 + per, A.ntasks * A.ngroups);
        if (k0 >= k1) return;
        SolveTask next = ld_scalar(A.tasks + A.task0 + k0 / A.ngroups);
        for (int k = k0; k < k1; ++k) {
            const SolveTask t = next;
            const int grp = k % A.ngroups;
            per = t.per;
            if (k + 1 < k1) next = ld_scalar(A.tasks + A.task0 + (k + 1) / A.ngroups);
            // hidden from the compiler, which would otherwise compute every
            // kind's lane offsets once, before the loop, and spill them
            int lid = tid;
            asm volatile("" : "+v"(lid));
            const Ctx<T> C{A,
                           S,
                           A.flags + kSolveCtl + (int64_t)grp * A.nflags,
                           kRhs * grp,
                           min(kRhs, A.nrhs - kRhs * grp),
                           lid,
                           lid & 63,
                           __builtin_amdgcn_readfirstlane(lid >> 6),
                           lid & 15,
                           (lid >> 4) & 3};
            switch (t.kind) {
            case kFwdRows: fwd_rows(C, t); break;
            case kFwdRows64: fwd_rows64(C, t); break;
            case kFwdTop: fwd_top(C, t); break;
            case kFwdPiv: fwd_piv(C, t); break;
            case kBwdPart: bwd_part(C, t); break;
            case kBwdCols: bwd_cols(C, t); break;
            case kBwdTop: bwd_top(C, t); break;
            default: bwd_piv(C, t); break;
            }
            // (each ends with a barrier after its last use of S and ticket)
        }
    }
}

__global__ __launch_bounds__(kThreads) void k_solve_reset(int* p, int64_t n, int polls)
{
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        p[i] = i == kSolveStop + 1 ? polls : 0;
}

void launch_solve_reset(int* flags, int64_t n, int polls, hipStream_t st)
{
    if (n > 0)
        hipLaunchKernelGGL(k_solve_reset, dim3((unsigned)std::min<int64_t>((n + kThreads - 1) / kThreads, 512)),
                           dim3(kThreads), 0, st, flags, n, polls);
}
// Four workgroups per CU (in FP64, where the chip holds three, the last quarter
// finds the tickets gone); fewer tickets, fewer.
template <typename T> void launch_solve(const SolveArgs<T>& A, hipStream_t st)
{
    const int64_t total = (int64_t)A.ntasks * A.ngroups;
    if (total > 0)
        hipLaunchKernelGGL(k_solve<T>, dim3((unsigned)std::min<int64_t>(total, 1024)), dim3(kThreads), 0, st, A);
}
template void launch_solve<double>(const SolveArgs<double>&, hipStream_t);
template void launch_solve<float>(const SolveArgs<float>&, hipStream_t);

}  // namespace mfd
