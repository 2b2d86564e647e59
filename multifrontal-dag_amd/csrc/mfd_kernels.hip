// HIP kernels of the numeric phase, written for gfx950 (CDNA4, wave64).
//
// Fronts live in one pool, each an n x n column-major block (see NodeDev in
// mfd_plan.h).  Every kernel processes one range of a task array; a
// workgroup owns one task, so no two workgroups of one launch write the same
// entry and the results do not depend on scheduling.
//
// Reference operations these kernels replace (paths relative to the
// reference root, src/main/):
//   k_assemble      set_zero + set_coefficient        zero_setter_m.f90:12-31, coefficient_setter_m.f90:15-50
//   k_extend_add,   extend_add_tri / extend_add_rect  seq_factorize/kernel/extend_add_kernel_m.f90:6-34
//   k_pull_children (children that are not large; k_gemm mode 3 for the others)
//   k_small_front   the per-front tile loop           seq_factorize_m.f90:31-79
//   k_diag,         DPOTRF("U") of a diagonal block,  seq_factorize/kernel/factorize_kernel_m.f90:4-16,
//   k_upd_diag      with its panel's DTRSM tiles      border_kernel_m.f90:9-30
//   k_gemm          DTRSM (modes 1, 2), DSYRK / DGEMM factorize_kernel_m.f90:11-33, border_kernel_m.f90:21-30,
//                   updates (modes 0, 3)              border_subroutines_m.f90:41-73
// The solves are in mfd_solve.hip, the bottom of the tree in mfd_tree.hip.
#include <hip/hip_runtime.h>

#include "mfd_device.h"
#include "mfd_kernels.h"

namespace mfd {

namespace {

// 16-bit operands with FP32 accumulation (the FP16_IR / BF16_IR forms):
// D(16x16) += A(16x16) B(16x16); lane l supplies A[l%16][4(l/16) + i] and
// B[4(l/16) + i][l%16], i < 4; the accumulator layout is the f32 one above.
// Operands are rounded to nearest even from FP32.
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef short s4 __attribute__((ext_vector_type(4)));
enum LowPrec { kNative = 0, kF16 = 1, kBF16 = 2 };
__device__ __forceinline__ short bf16_bits(float x)
{
    unsigned u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even (finite inputs)
    return (short)(u >> 16);
}
template <int LP> struct Mfma16;
template <> struct Mfma16<kF16> {
    typedef h4 op_t;
    static __device__ _Float16 cvt(float x) { return (_Float16)x; }
    static __device__ f4 mma(op_t a, op_t b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0); }
};
template <> struct Mfma16<kBF16> {
    typedef s4 op_t;
    static __device__ short cvt(float x) { return bf16_bits(x); }
    static __device__ f4 mma(op_t a, op_t b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }
};


// ------------------------------------------- dense 64 x 64 partial Cholesky
// A front (or diagonal block) of order n <= 64 in LDS, factored in its first
// c columns by a blocked right-looking algorithm with 16-column panels:
//   - each panel is factored by one wave, one row per lane, in a 16-step
//     chain: the pivot and the finished column's entry of the next column's
//     row come from their lanes by readlane, the entries the later columns
//     need are read back from LDS, where each column is stored as soon as it
//     is finished;
//   - the panel's 16 x 16 diagonal block is inverted by another wave during
//     the next panel's chain (lane r solves L u = e_r);
//   - the rank-16 update of the trailing blocks runs on MFMA across the four
//     waves;
//   - the off-diagonal 16 x 16 blocks of L^{-1} follow on MFMA, by distance
//     from the diagonal: X_ij = -inv(L_ii) sum_{k=j}^{i-1} L_ik X_kj.
// Layout: A[col][row] holds the lower triangle (zero past n); afterwards it
// holds L in columns < c and the Schur complement in the trailing block.
// X[col][row] = L^{-1}[row][col] for row, col < c (other entries are
// scratch).  Upper-triangle entries of A are scratch too.  rs[k] = 1 / L_kk.
template <typename T> struct Front64 {
    T A[64][65];
    T X[64][65];
    T Ts[4][16][17];
    T rs[64];
};

// Panel b16 .. b16 + cb - 1 (cb <= 16; FULL: cb == 16) by one wave, rows
// b16 .. 63 on their lanes.  Column k: d = x_k on lane k, rs = 1 / sqrt(d),
// L_kk = sqrt(d), l = x_k / L_kk (quot: exact whenever the quotient is
// representable).  Every lane forms row k+1's quotient too, from the entry its
// lane had before (by readlane, beside the chain), and updates column k+1 at
// once (the next pivot needs it): by the finished entries, so that where the
// factor is representable the pivots are exact, and zero where they are zero.
// The column goes to LDS, and its entries for rows k+2 .. 15 are read back
// (the wave's LDS accesses complete in issue order, so the reads see the
// column) and applied to those columns in step k+1, by when the reads have
// landed.  A partial panel also updates the block's columns past cb (trailing
// columns of the front) by all of its columns, and stores them.  After the
// first panel the 16 lanes past row 63 hold the unit vectors, which the same
// operations turn into the rows of L_bb^{-T}: the diagonal block's inverse
// (column id of it to X[b16 + id]; in a partial panel the rows past its cb
// pivots are not used, and its columns past them are zero in the others).
// Every x_j receives its updates in column order, as in the plain loop.  The first
// non-positive pivot is recorded (each pivot stays on its row's lane; one look
// at all of them at the end).
// One wave issues at most an instruction every four cycles, so the panel is
// bound by its instruction count as much as by the chain: 3960 cycles for 16
// columns in FP64, 3320 in FP32; with a check per pivot and masked stores
// 4810 and 4020.  (Updating column k+1 by x_k rs times its entry's, not yet
// corrected, takes 3760 and 3070 and lets singular matrices pass.)
template <typename T, bool FULL>
__device__ __forceinline__ void panel16(Front64<T>& S, int b16, int cb, int n, int* info, int col0)
{
    int r = threadIdx.x & 63, diag = 66 * b16;
    pin(r);  // (the comparisons with it stay here: hoisted, their masks spill)
    pin(diag);
    T* const Ad = &S.A[0][0] + diag;  // the panel's diagonal block, by vector address
    const int row = b16 + r;
    const bool live = row < n;
    const int at = live ? row : 64;  // (column slot 64 of a row is not used)
    const int id = row - 64;         // the unit vector on this lane
    T x[16], v[16], piv = T(1);
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = S.A[b16 + j][at];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        pin(x[j]);  // (read by every lane: no branch around each)
        x[j] = (live && (r >= 16 || j <= r)) ? x[j] : id == j ? T(1) : T(0);
        v[j] = T(0);
    }
    T lp = T(0);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (FULL || k < cb) {  // no early exit: the loop stays unrolled, x and v in registers
            const T d = bcast(x[k], k), rs = rsqrt_nr(d), sd = sqrt_from_rs(d, rs), q = quot(x[k], sd, rs);
            // column k-1's updates of columns k+1 .. 15 (its entries read in
            // step k-1), with column k's of column k+1
            if (k + 1 < 16) {
                const T u = quot(bcast(x[k], k + 1), sd, rs);
                x[k + 1] -= lp * v[k + 1];
                if (FULL || k + 1 < cb) x[k + 1] -= q * u;
                pin(x[k + 1]);
            }
            piv = r == k ? d : piv;
            pin(piv);
            const T l = r == k ? sd : q;
            x[k] = l;
            S.A[b16 + k][at] = l;
            S.rs[b16 + k] = rs;
#pragma unroll
            for (int j = k + 2; j < 16; ++j) {
                x[j] -= lp * v[j];
                pin(x[j]);
            }
            lp = l;
            __builtin_amdgcn_wave_barrier();  // the reads below stay after the store above
#pragma unroll
            for (int j = k + 2; j < 16; ++j) v[j] = Ad[65 * k + j];
            if (!FULL && k + 1 == cb && k + 1 < 16) v[k + 1] = Ad[65 * k + k + 1];
        }
    }
    if (!FULL) {
        if (r == 0)
            for (int k = cb; k < 16; ++k) S.rs[b16 + k] = T(1);  // finite stand-ins for the block's inverse
        // the last column's updates of the block's columns past cb
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (j >= cb) x[j] -= lp * v[j];
        if (live) {
#pragma unroll
            for (int j = 0; j < 16; ++j)
                if (j >= cb) S.A[b16 + j][row] = x[j];
        }
    }
    if (id >= 0 && id < 16) {
#pragma unroll
        for (int j = 0; j < 16; ++j) S.X[b16 + id][b16 + j] = x[j];
    }
    const unsigned long long bad = __ballot(!(piv > T(0)));
    if (bad && r == 0) atomicMin(info, col0 + b16 + __ffsll(bad));
}

// Inverse of panel b16's 16 x 16 diagonal block of L (one wave; the first
// panel's, whose 64 rows leave panel16 no lanes for it): lane r < 16
// solves L u = e_r by forward substitution, u = column r of the inverse,
// stored as X[b16 + r][b16 + k] = u_k.  For a partial panel the rows and
// columns past its cb pivots are finite stand-ins (rs = 1 there; the
// entries of L in them are trailing-block values), which no stored
// inverse entry uses: the inverse's row k < cb depends only on the rows
// and columns <= k.
template <typename T>
__device__ __forceinline__ void diaginv16(Front64<T>& S, int b16)
{
    const int r = threadIdx.x & 63;
    T y[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) y[j] = j == r ? T(1) : T(0);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const T y0 = y[k] * S.rs[b16 + k];
        y[k] = y0;
#pragma unroll
        for (int j = k + 1; j < 16; ++j) y[j] -= y0 * S.A[b16 + k][b16 + j];
    }
    if (r < 16) {
#pragma unroll
        for (int k = 0; k < 16; ++k) S.X[b16 + r][b16 + k] = y[k];
    }
}

// A_IJ -= L_Ib L_Jb^T over the cb pivot columns of panel b (one wave).
template <typename T>
__device__ __forceinline__ void trailing16(Front64<T>& S, int b16, int cb, int I, int J)
{
    typedef typename Mfma<T>::acc_t acc_t;
    const int lane = threadIdx.x & 63, li = lane & 15;
    // two chains of products, subtracted at the end: added to A_IJ one by one
    // they would round at its magnitude each time
    acc_t acc = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0}, old;
#pragma unroll
    for (int v = 0; v < 4; ++v) old[v] = S.A[16 * J + li][16 * I + Mfma<T>::row(lane, v)];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int kk = 4 * q + (lane >> 4);
        const bool ok = kk < cb;
        const T a = ok ? S.A[b16 + kk][16 * I + li] : T(0);
        const T b = ok ? S.A[b16 + kk][16 * J + li] : T(0);
        if (q & 1)
            acc2 = Mfma<T>::mma(a, b, acc2);
        else
            acc = Mfma<T>::mma(a, b, acc);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) S.A[16 * J + li][16 * I + Mfma<T>::row(lane, v)] = old[v] - (acc[v] + acc2[v]);
}

// X_ij = -inv(L_ii) sum_{k=j}^{i-1} L_ik X_kj (one wave; staging in Ts[w]).
template <typename T>
__device__ __forceinline__ void inverse16(Front64<T>& S, int i, int j, int w)
{
    typedef typename Mfma<T>::acc_t acc_t;
    const int lane = threadIdx.x & 63, li = lane & 15;
    acc_t acc = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0};  // two chains of products
    for (int k = j; k < i; ++k) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int kk = 4 * q + (lane >> 4);
            const T a = S.A[16 * k + kk][16 * i + li], b = S.X[16 * j + li][16 * k + kk];
            if (q & 1)
                acc2 = Mfma<T>::mma(a, b, acc2);
            else
                acc = Mfma<T>::mma(a, b, acc);
        }
    }
    wave_sync();
#pragma unroll
    for (int v = 0; v < 4; ++v) S.Ts[w][Mfma<T>::row(lane, v)][li] = acc[v] + acc2[v];
    wave_sync();
    acc = acc2 = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int m = 4 * q + (lane >> 4);
        const T a = S.X[16 * i + m][16 * i + li], b = S.Ts[w][m][li];
        if (q & 1)
            acc2 = Mfma<T>::mma(a, b, acc2);
        else
            acc = Mfma<T>::mma(a, b, acc);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) S.X[16 * j + li][16 * i + Mfma<T>::row(lane, v)] = -(acc[v] + acc2[v]);
}

// All 256 threads: loads the lower n x n block at g (leading dimension ld),
// factors its first c columns, writes L and the Schur complement back and
// stores L^{-T} of the c x c factor column-major at inv (64 x 64,
// zero-padded: inv[r + 64 q] = L^{-1}[q][r]).  A pivot that is not positive
// records the global column col0 + k + 1 in *info (smallest wins).
// Same, with S.A already holding the block (lower part, zero past row n)
// and S.X zero above the diagonal blocks, both visible to the workgroup.
// pre(w), w = 0 .. 2: what three waves do during the first panel's chain.
template <typename T, typename Pre>
__device__ __forceinline__ void factor_dense64_loaded(Front64<T>& S, T* g, int64_t ld, int n, int c, int* info,
                                                      int col0, T* inv, Pre pre)
{
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const int nblk = (c + 15) >> 4, nall = (n + 15) >> 4, last = nblk - 1;
    // columns 16 jb .. of L (or of the trailing block) and rows 16 ib .. of
    // the inverse to memory, by wave w of nw
    auto put_cols = [&](int jb, int w, int nw) {
#pragma unroll 4
        for (int q = w; q < 16; q += nw) {
            const int col = 16 * jb + q;
            if (lane < n && col <= lane) g[lane + (int64_t)col * ld] = S.A[col][lane];
        }
    };
    auto put_inv = [&](int ib, int w, int nw) {
#pragma unroll 4
        for (int q = 16 * ib + w; q < 16 * ib + 16; q += nw)
            inv[lane + 64 * q] = (lane < c && q < c) ? S.X[lane][q] : T(0);
    };
    // Phase b: wave 0 runs panel b's chain, which also inverts its diagonal
    // block (b > 0); beside it the other waves finish panel b-1's update
    // (block column b, which the chain needs, came before), form row b-1 of
    // the inverse's off-diagonal blocks and store what is final: block column
    // b-1 of L, block row b-2 of the inverse.  Then all waves apply panel b to
    // block column b+1.  Phase nblk has the last row of the inverse alone.
    // Only the last panel can be partial.
    for (int b = 0; b <= nblk; ++b) {
        const int b16 = 16 * b, cb = min(16, c - b16);
        if (wv == 0 && b < nblk) {
            if (cb == 16)
                panel16<T, true>(S, b16, 16, n, info, col0);
            else
                panel16<T, false>(S, b16, cb, n, info, col0);
        } else if (b == 0) {
            pre(wv - 1);
        } else {
            if (b == 1 && wv == 1) diaginv16<T>(S, 0);
            const int j = b < nblk ? wv - 2 : wv;
            if (j >= 0 && j < b - 1) inverse16<T>(S, b - 1, j, wv);
            int idx = 0;
            for (int J = b + 1; b < nblk && J < nall; ++J)
                for (int I = J; I < nall; ++I, ++idx)
                    if (1 + (idx + b) % 3 == wv) trailing16<T>(S, b16 - 16, 16, I, J);
            if (wv == (b == 3 && b < nblk ? 1 : 3)) {
                for (int jb = b - 1; jb < (b < nblk ? b : nall); ++jb) put_cols(jb, 0, 1);
                if (b >= 2) put_inv(b - 2, 0, 1);
            }
        }
        if (b == nblk) break;
        __syncthreads();
        if (b + 1 < nall) {
            int idx = 0;
            for (int J = b + 1; J < (b < last ? b + 2 : nall); ++J)
                for (int I = J; I < nall; ++I, ++idx)
                    if ((idx & 3) == wv) trailing16<T>(S, b16, cb, I, J);
            __syncthreads();
        }
    }
    __syncthreads();
    for (int ib = max(last, 0); ib < 4; ++ib) put_inv(ib, wv, 4);
}
template <typename T>
__device__ __forceinline__ void factor_dense64(Front64<T>& S, T* g, int64_t ld, int n, int c, int* info, int col0,
                                               T* inv)
{
    // every load from a clamped in-bounds position, all issued before the
    // masked stores (no branch around each load)
    T v[16];
    const int row = threadIdx.x & 63, rc = min(row, n - 1);
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = ld_off(g, (unsigned)(rc + min((int)(threadIdx.x >> 6) + 4 * j, n - 1) * ld));
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int col = (threadIdx.x >> 6) + 4 * j;
        S.A[col][row] = (row < n && col <= row) ? v[j] : T(0);
        S.X[col][row] = T(0);
    }
    __syncthreads();
    factor_dense64_loaded<T>(S, g, ld, n, c, info, col0, inv, [](int) {});
}

}  // namespace

// ---------------------------------------------------------------- assembly
// The lower part (row >= col; the upper part of a front is never read) of
// kFillCols columns of one front: zero, but for the stored A entries, each of
// which lands on exactly one front position (coefficient_setter_m.f90:26-50
// in the front layout): entry k of the task goes to pool[dst[k]], from
// a[src[k]], with scale != nullptr (the 16-bit forms) times s[r] s[c], (r, c) =
// rc[k] its global (postordered, 0-based) row and column.  Bound by its
// stores; a wave takes whole columns, so that columns of a few hundred
// entries keep its lanes busy.  (Zeroing 64 columns a workgroup and scattering
// A in a second launch, one pair of launches per level, took 13 + 4 us and
// two launch gaps for a level of a 23 x 19 x 17 grid.)
template <typename T>
__global__ __launch_bounds__(kThreads) void k_assemble(T* pool, const NodeDev* nodes, const FillTask* tasks,
                                                       const double* a, const int64_t* dst, const int64_t* src,
                                                       const int2* rc, const double* scale)
{
    const FillTask t = tasks[blockIdx.x];
    const NodeDev nd = nodes[t.node];
    const int n = nd.n, jend = min(t.j0 + kFillCols, n), lane = threadIdx.x & 63;
    constexpr int V = 16 / sizeof(T);  // elements per 16-byte store
    T* g = pool + nd.front;
    for (int j = t.j0 + (threadIdx.x >> 6); j < jend; j += kThreads / 64) {
        // rows [j, n) of column j: scalar head up to a 16-byte boundary,
        // 16-byte stores, scalar tail
        T* col = g + (int64_t)j * n;
        const int head = min((int)((V - ((reinterpret_cast<uintptr_t>(col + j) / sizeof(T)) % V)) % V), n - j);
        const int i0 = j + head, nv = (n - i0) / V, tail = i0 + nv * V;
        if (lane < head) col[j + lane] = T(0);
        uint4* v = reinterpret_cast<uint4*>(col + i0);
        for (int p = lane; p < nv; p += 64) v[p] = make_uint4(0u, 0u, 0u, 0u);
        if (lane < n - tail) col[tail + lane] = T(0);
    }
    if (t.e0 == t.e1) return;
    stores_done();
    __syncthreads();
    for (int64_t k = t.e0 + threadIdx.x; k < t.e1; k += kThreads) {
        double v = a[src[k]];
        if (scale) {
            const int2 q = rc[k];
            v = v * scale[q.x] * scale[q.y];
        }
        pool[dst[k]] = (T)v;
    }
}

// Diagonal scaling of the 16-bit forms: s[j] = 2^-e with e = floor(E / 2)
// for A(j,j) = m 2^E (0.5 <= m < 1), so that s_j^2 A(j,j) lies in [0.5, 2);
// a diagonal that is not positive and finite keeps s[j] = 1.  Powers of two
// make the scaled matrix S A S exact.  diag_src[j]: caller index of A(j,j)
// (j postordered).
__global__ __launch_bounds__(kThreads) void k_diag_scale(double* s, const double* a, const int64_t* diag_src, int n)
{
    const int j = blockIdx.x * kThreads + threadIdx.x;
    if (j >= n) return;
    const double d = a[diag_src[j]];
    double v = 1.0;
    if (d > 0.0 && d <= 1.7976931348623157e308) {
        int E;
        (void)frexp(d, &E);
        const int e = E >= 0 ? E / 2 : -((1 - E) / 2);  // floor(E / 2)
        v = ldexp(1.0, -e);
    }
    s[j] = v;
}

// out[i + k n] = s[i] in[i + k n] (out may be in).
__global__ __launch_bounds__(kThreads) void k_scale_rows(double* out, const double* in, const double* s, int n, int nrhs)
{
    const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (e >= (int64_t)n * nrhs) return;
    out[e] = s[e % n] * in[e];
}

// ------------------------------------------------------------- extend-add
// One 64 x 64 tile (ti >= tj) of the child's update matrix, lower part only,
// added into the parent front at the rows/columns local_index gives (used
// for the children of order <= 64; the Schur tiles of larger children add
// their results themselves).  The map is injective within a child and one
// launch carries at most one child per parent, so the read-modify-write is
// race-free; a launch per child rank keeps the order of the additions fixed.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_extend_add(T* pool, const int* lidx, const NodeDev* nodes,
                                                         const ExtTask* tasks)
{
    const ExtTask t = tasks[blockIdx.x];
    const NodeDev ch = nodes[t.child];
    const NodeDev pa = nodes[ch.parent];
    __shared__ int64_t colmap[kTile];
    const int tid = threadIdx.x;
    const int i0 = t.ti * kTile, j0 = t.tj * kTile;
    if (tid < kTile) {
        int j = j0 + tid;
        colmap[tid] = j < ch.w ? (int64_t)(lidx[ch.lidx + j] - 1) * pa.n : 0;
    }
    __syncthreads();
    const int i = i0 + (tid & 63);
    if (i >= ch.w) return;
    const int64_t prow = lidx[ch.lidx + i] - 1;
    const T* src = pool + ch.front + (int64_t)(ch.c + i) + (int64_t)ch.c * ch.n;
    T* dst = pool + pa.front + prow;
    for (int jj = tid >> 6; jj < kTile; jj += 4) {
        int j = j0 + jj;
        if (j >= ch.w || j > i) break;
        dst[colmap[jj]] += src[(int64_t)j * ch.n];
    }
}

// The update matrices of children in the bottom of the tree (order <= 128),
// added into kPullCols columns of their parent, child after child: all of them
// in one launch after k_tree, where a launch per level and child rank took
// 8 to 15 us each (44 of them for 512 systems).  A child's columns that fall
// into the task's are consecutive (local_index ascends), a wave takes every
// fourth, and the loads of all of them are in flight together.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_pull_children(T* pool, const int* lidx, const NodeDev* nodes,
                                                            const PullTask* tasks, const int* children)
{
    const PullTask t = tasks[blockIdx.x];
    const NodeDev pa = nodes[t.node];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    T* dst = pool + pa.front;
    for (int k = 0; k < t.nchild; ++k) {
        const NodeDev ch = nodes[children[t.child + k]];
        const int* li = lidx + ch.lidx;
        // the first update column at or past parent column j0 (lanes 0 .. 63
        // and 64 .. 127 of the order look at one each)
        const int l0 = lane < ch.w ? li[lane] - 1 : INT_MAX, l1 = lane + 64 < ch.w ? li[lane + 64] - 1 : INT_MAX;
        const int q0 = __popcll(__ballot(l0 < t.j0)) + __popcll(__ballot(l1 < t.j0));
        const int q1 = __popcll(__ballot(l0 < t.j0 + kPullCols)) + __popcll(__ballot(l1 < t.j0 + kPullCols));
        const T* src = pool + ch.front + ch.c + (int64_t)ch.c * ch.n;
        constexpr int G = 4;
        for (int qb = q0 + wv; qb < q1; qb += 4 * G) {
            T* p[2 * G];
            T c[2 * G], v[2 * G];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int q = min(qb + 4 * g, q1 - 1);
                T* col = dst + (int64_t)(li[q] - 1) * pa.n;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    // (lanes without an entry read the column's diagonal one)
                    const int i = lane + 64 * h;
                    const bool on = i >= q && i < ch.w;
                    p[2 * g + h] = col + (on ? (h ? l1 : l0) : li[q] - 1);
                    c[2 * g + h] = src[(on ? i : q) + (int64_t)q * ch.n];
                    v[2 * g + h] = *p[2 * g + h];
                }
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int q = qb + 4 * g;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int i = lane + 64 * h;
                    if (q < q1 && i >= q && i < ch.w) *p[2 * g + h] = v[2 * g + h] + c[2 * g + h];
                }
            }
        }
        if (k + 1 < t.nchild) {
            stores_done();
            __syncthreads();
        }
    }
}

// -------------------------------------------------------- small fronts
// Whole partial factorization of a front with n <= 64 in one workgroup: L in
// the first c columns, the Schur complement in the trailing block, and the
// inverse of the c x c diagonal block for the solves.  As many workgroups per
// CU as k_diag.
template <typename T>
__global__ __launch_bounds__(kThreads, sizeof(T) == 8 ? 2 : 4) void k_small_front(T* pool, const NodeDev* nodes, const int* tasks, int* info)
{
    const NodeDev nd = nodes[tasks[blockIdx.x]];
    __shared__ Front64<T> S;
    factor_dense64<T>(S, pool + nd.front, nd.n, nd.n, nd.c, info, nd.first, pool + nd.inv);
}

// ------------------------------------------------------ large fronts
// LDS staging of one 64 x 64 MFMA tile product: NB chunks of 16 columns.
template <typename T, int NB = 1> struct TileLds {
    T As[NB][16][kTile + 4];
    T Bs[NB][16][kTile + 4];
};

// sum_kk A[row][kk] B[col][kk] over a 64 x 64 tile (rows past m and columns
// past n give 0), FP64/FP32 MFMA 16x16x4.  Four waves each own a 32 x 32
// quarter (2 x 2 MFMA blocks c[i][j]: rows wr + 16 i, columns wc + 16 j).  K
// is staged through LDS in chunks of 16, the global loads two chunks ahead
// of their MFMAs; with NB = 2 the chunks alternate between two buffers and
// one barrier a chunk is enough (Schur updates of the 64^3 workload: 8.4 ms
// with one chunk ahead and two barriers, 8.1 so; the matrix cores were busy
// 59% of that time).  Every read of A and B happens before the function
// returns (it ends with a barrier), so the caller may overwrite A afterwards.
//
// tb != 0 takes B transposed in memory (B[col][kk] at B + col * ldb + kk);
// its chunks are then read 16 entries at a time along kk.
//
// LP = kF16 / kBF16 (FP32 operands only) rounds each operand to 16 bits as
// it leaves LDS and multiplies on the 16-bit MFMA with FP32 accumulation.
// TB: 0 = B stored like A (B[col + kk * ldb]), 1 = B transposed in memory,
// -1 = as the runtime flag tb says (the panel TRSM kernel holds both).
// OWN: also the rows' product with themselves, own[i][j] += sum_kk A[row][kk]
// A[col][kk] (the block at wr = 0, wc = 32 above the diagonal left out).
template <typename T, int LP = kNative, int TB = -1, int NB = 1, bool OWN = false>
__device__ __forceinline__ void tile_mma(const T* A, int lda, const T* B, int ldb, bool tb, int m, int n, int k,
                                         TileLds<T, NB>& L, typename Mfma<T>::acc_t (&c)[2][2],
                                         typename Mfma<T>::acc_t (&own)[2][2], int tid = threadIdx.x)
{
    static_assert(LP == kNative || sizeof(T) == 4, "16-bit operands come from FP32 fronts");
    typedef typename Mfma<T>::acc_t acc_t;
    const bool trb = TB < 0 ? tb : TB == 1;
    const int lane = tid & 63, wv = tid >> 6;
    const int wr = (wv & 1) * 32, wc = (wv >> 1) * 32;
    const int li = tid & 63, lp = tid >> 6;
    acc_t c00 = {0, 0, 0, 0}, c01 = {0, 0, 0, 0}, c10 = {0, 0, 0, 0}, c11 = {0, 0, 0, 0};
    T ra[2][4], rb[2][4];
    // transposed-B chunk: element e = tid + 256 p is (col e / 16, kk e % 16)
    const int tcol = tid >> 4, tkk = tid & 15;
    // Every load from a clamped in-bounds position (m, n, k >= 1), its value
    // kept raw and masked only as it is stored to LDS: no branch around the
    // loads, which all go out together.
    const int lic = min(li, m - 1), lib = min(li, n - 1);
    auto load = [&](int k0, T (&xa)[4], T (&xb)[4]) {
        // uniform bases, 32-bit offsets within the chunk: one VGPR an address
        const T* Ak = A + (int64_t)k0 * lda;
        const T* Bk = trb ? B + k0 : B + (int64_t)k0 * ldb;
        const int kl = k - 1 - k0;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int kc = min(lp + 4 * p, kl);
            xa[p] = ld_off(Ak, (unsigned)(lic + kc * lda));
            if (trb)
                xb[p] = ld_off(Bk, (unsigned)(min(tcol + 16 * p, n - 1) * ldb + min(tkk, kl)));
            else
                xb[p] = ld_off(Bk, (unsigned)(lib + kc * ldb));
        }
    };
    auto store = [&](int k0, int buf, const T (&xa)[4], const T (&xb)[4]) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int kk = k0 + lp + 4 * p;
            L.As[buf][lp + 4 * p][li] = (li < m && kk < k) ? xa[p] : T(0);
            if (trb) {
                const int col = tcol + 16 * p;
                L.Bs[buf][tkk][col] = (col < n && k0 + tkk < k) ? xb[p] : T(0);
            } else {
                L.Bs[buf][lp + 4 * p][li] = (li < n && kk < k) ? xb[p] : T(0);
            }
        }
    };
    auto multiply = [&](int buf) {
        if constexpr (LP == kNative) {
            // the operands of the chunk's four k-steps, then its 16 MFMAs (the
            // compiler interleaves the reads with the MFMAs)
            T a0[4], a1[4], b0[4], b1[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int kr = q * 4 + (lane >> 4);
                a0[q] = L.As[buf][kr][wr + (lane & 15)];
                a1[q] = L.As[buf][kr][wr + 16 + (lane & 15)];
                b0[q] = L.Bs[buf][kr][wc + (lane & 15)];
                b1[q] = L.Bs[buf][kr][wc + 16 + (lane & 15)];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                c00 = Mfma<T>::mma(a0[q], b0[q], c00);
                c01 = Mfma<T>::mma(a0[q], b1[q], c01);
                c10 = Mfma<T>::mma(a1[q], b0[q], c10);
                c11 = Mfma<T>::mma(a1[q], b1[q], c11);
            }
            if (OWN && wc <= wr) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int kr = q * 4 + (lane >> 4);
                    const T w0 = L.As[buf][kr][wc + (lane & 15)], w1 = L.As[buf][kr][wc + 16 + (lane & 15)];
                    own[0][0] = Mfma<T>::mma(a0[q], w0, own[0][0]);
                    own[0][1] = Mfma<T>::mma(a0[q], w1, own[0][1]);
                    own[1][0] = Mfma<T>::mma(a1[q], w0, own[1][0]);
                    own[1][1] = Mfma<T>::mma(a1[q], w1, own[1][1]);
                }
            }
        } else {
            typedef Mfma16<LP> M16;
            typename M16::op_t a0, a1, b0, b1;
            const int kr = 4 * (lane >> 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a0[i] = M16::cvt(L.As[buf][kr + i][wr + (lane & 15)]);
                a1[i] = M16::cvt(L.As[buf][kr + i][wr + 16 + (lane & 15)]);
                b0[i] = M16::cvt(L.Bs[buf][kr + i][wc + (lane & 15)]);
                b1[i] = M16::cvt(L.Bs[buf][kr + i][wc + 16 + (lane & 15)]);
            }
            c00 = M16::mma(a0, b0, c00);
            c01 = M16::mma(a0, b1, c01);
            c10 = M16::mma(a1, b0, c10);
            c11 = M16::mma(a1, b1, c11);
        }
    };
    // chunk k0 is in LDS, chunk k0 + 16 on its way in (xa, xb), chunk k0 + 32
    // is sent for in (ya, yb); the main loop without conditions, which would
    // make the wait for (xa, xb) a wait for every load
    auto step = [&](int k0, int buf, bool inner, T (&xa)[4], T (&xb)[4], T (&ya)[4], T (&yb)[4]) {
        if (inner || k0 + 32 < k) load(k0 + 32, ya, yb);
        multiply(NB == 2 ? buf : 0);
        if (NB == 1) __syncthreads();
        if (inner || k0 + 16 < k) store(k0 + 16, NB == 2 ? buf ^ 1 : 0, xa, xb);
        __syncthreads();
    };
    load(0, ra[0], rb[0]);
    if (k > 16) load(16, ra[1], rb[1]);
    store(0, 0, ra[0], rb[0]);
    __syncthreads();
    int k0 = 0;
    for (; k0 + 48 < k; k0 += 32) {
        step(k0, 0, true, ra[1], rb[1], ra[0], rb[0]);
        step(k0 + 16, 1, true, ra[0], rb[0], ra[1], rb[1]);
    }
    for (; k0 < k; k0 += 32) {
        step(k0, 0, false, ra[1], rb[1], ra[0], rb[0]);
        if (k0 + 16 < k) step(k0 + 16, 1, false, ra[0], rb[0], ra[1], rb[1]);
    }
    c[0][0] = c00;
    c[0][1] = c01;
    c[1][0] = c10;
    c[1][1] = c11;
}
// Cs[col][row] = c, in the layout of tile_mma's result.
template <typename T>
__device__ __forceinline__ void stage_acc(const typename Mfma<T>::acc_t (&c)[2][2], T (*Cs)[kTile + 1])
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int wr = (wv & 1) * 32, wc = (wv >> 1) * 32, q0 = wc + (lane & 15);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) Cs[q0 + 16 * j][wr + 16 * i + Mfma<T>::row(lane, v)] = c[i][j][v];
}

// The same product staged as Cs[col][row]; ends with a barrier.
template <typename T, int LP = kNative, int TB = -1, int NB = 1>
__device__ __forceinline__ void tile_product(const T* A, int lda, const T* B, int ldb, bool tb, int m, int n, int k,
                                             TileLds<T, NB>& L, T (*Cs)[kTile + 1])
{
    typename Mfma<T>::acc_t c[2][2];
    tile_mma<T, LP, TB, NB>(A, lda, B, ldb, tb, m, n, k, L, c, c);
    stage_acc<T>(c, Cs);
    __syncthreads();
}

// The same wave layout with A in LDS (Am[kk][row], zero past row m and column
// k) and B (transposed in memory) in registers: rb[4 i + p] is entry (column
// tid / 16 + 16 p, kk 16 i + tid % 16), staged through L.Bs in chunks of 16.
// Ends with a barrier.
template <typename T>
__device__ __forceinline__ void load_tb(const T* B, int ldb, int n, int k, T (&rb)[16])
{
    const int tcol = threadIdx.x >> 4, tkk = threadIdx.x & 15;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int p = 0; p < 4; ++p)
            rb[4 * i + p] = ld_off(B, (unsigned)(min(tcol + 16 * p, n - 1) * ldb + min(16 * i + tkk, k - 1)));
}
template <typename T, int NB>
__device__ __forceinline__ void tile_mma_ldsA(const T (*Am)[kTile + 1], const T (&rb)[16], int n, int k,
                                              TileLds<T, NB>& L, typename Mfma<T>::acc_t (&c)[2][2])
{
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wr = (wv & 1) * 32, wc = (wv >> 1) * 32, tcol = tid >> 4, tkk = tid & 15;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) c[i][j] = typename Mfma<T>::acc_t{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (16 * i < k) {
            const int buf = NB == 2 ? i & 1 : 0;
#pragma unroll
            for (int p = 0; p < 4; ++p)
                L.Bs[buf][tkk][tcol + 16 * p] = (tcol + 16 * p < n && 16 * i + tkk < k) ? rb[4 * i + p] : T(0);
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int kr = q * 4 + (lane >> 4);
                const T a0 = Am[16 * i + kr][wr + (lane & 15)], a1 = Am[16 * i + kr][wr + 16 + (lane & 15)];
                const T b0 = L.Bs[buf][kr][wc + (lane & 15)], b1 = L.Bs[buf][kr][wc + 16 + (lane & 15)];
                c[0][0] = Mfma<T>::mma(a0, b0, c[0][0]);
                c[0][1] = Mfma<T>::mma(a0, b1, c[0][1]);
                c[1][0] = Mfma<T>::mma(a1, b0, c[1][0]);
                c[1][1] = Mfma<T>::mma(a1, b1, c[1][1]);
            }
            if (NB == 1) __syncthreads();
        }
    }
    if (NB == 2) __syncthreads();
}

// One GemmTask per workgroup (see mfd_plan.h): C -= A B^T (mode 0: the
// DSYRK/DGEMM updates) or C = A B^T with B transposed in memory (mode 1: the
// panel TRSM as a product with the stored L^{-T} of the diagonal block, C
// and A the same rows).
// The result goes through LDS so the write of C is coalesced along columns.
// KIND only names the instance after the kernel class that launches it
// (TRSM, in-panel update, Schur update), so that profiles tell them apart.
// The result goes through LDS so the write of C is coalesced along columns
// (written straight from the accumulators it would be 32-byte pieces).
template <typename T, int LP = kNative, bool PRE = true, int TB = -1, int NB = 1, bool SYRK = false>
__device__ __forceinline__ void gemm_task(T* pool, const GemmTask& t, TileLds<T, NB>& L, T (*Cs)[kTile + 1],
                                          const int* lidx = nullptr)
{
    T* C = pool + t.c;
    const int tid = threadIdx.x, row = tid & 63;
    // the entries of C this thread reads afterwards (row, column tid / 64 +
    // 4 j), loaded before the K loop so that their latency hides behind it
    // (from clamped positions, masked where used); PRE = false (the update
    // and Schur tiles, four workgroups per CU, where the registers they would
    // hold are those of the second chunk in flight) loads them after it
    T cpre[16];
    if (PRE && t.mode != 1) {
        const int rc = min(row, t.m - 1);
#pragma unroll
        for (int j = 0; j < 16; ++j) cpre[j] = C[rc + (int64_t)min((tid >> 6) + 4 * j, t.n - 1) * t.ldc];
    }
    // the stored inverse of the second product (mode 2), early where
    // registers are plenty
    constexpr bool kEarly = PRE && NB == 2, kTrsm = TB != 0;
    T rb[16];
    if (kEarly && kTrsm && t.mode == 2) load_tb(pool + t.d, kPanel, t.n, t.kd, rb);
    typename Mfma<T>::acc_t acc[2][2], own[2][2] = {{{0, 0, 0, 0}, {0, 0, 0, 0}}, {{0, 0, 0, 0}, {0, 0, 0, 0}}};
    T dpre[16];
    auto load_d = [&]() {
        const int rd = min(row, t.syrk - 1);
#pragma unroll
        for (int j = 0; j < 16; ++j)
            dpre[j] = ld_off((const T*)pool + t.cd, (unsigned)(rd + min((tid >> 6) + 4 * j, rd) * t.ldc));
    };
    if constexpr (SYRK && kEarly) load_d();
    tile_mma<T, LP, TB, NB, SYRK>(pool + t.a, t.lda, pool + t.b, t.ldb, t.mode == 1, t.m, t.n, t.k, L, acc, own);
    // the parent positions of this thread's row and columns (local_index)
    int lrow = 1, lcol[16];
    if (t.mode == 3) {
        lrow = lidx[t.li + min(row, t.m - 1)];
#pragma unroll
        for (int j = 0; j < 16; ++j) lcol[j] = lidx[t.lj + min((tid >> 6) + 4 * j, t.n - 1)];
    }
    if (!PRE && t.mode != 1) {
        const int rc = min(row, t.m - 1);
#pragma unroll
        for (int j = 0; j < 16; ++j) cpre[j] = C[rc + (int64_t)min((tid >> 6) + 4 * j, t.n - 1) * t.ldc];
    }
    stage_acc<T>(acc, Cs);
    __syncthreads();
    if (kTrsm && t.mode == 2) {
        // Cs = C - A B^T, then C = Cs D^T (D = L^{-1}, stored transposed)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int col = (tid >> 6) + 4 * j;
            Cs[col][row] = (row < t.m && col < t.n) ? cpre[j] - Cs[col][row] : T(0);
        }
        __syncthreads();
        if (!kEarly) load_tb(pool + t.d, kPanel, t.n, t.kd, rb);
        tile_mma_ldsA<T, NB>(Cs, rb, t.n, t.kd, L, acc);
        stage_acc<T>(acc, Cs);
        __syncthreads();
    }
    if constexpr (SYRK) {
        // the diagonal block at cd loses R R^T over its lower syrk x syrk part,
        // R = the tile's rows over the pending panels (own, formed as they
        // passed through LDS) and the panel just solved (Cs, zero past the
        // tile's rows and columns)
        const int lane = tid & 63, wr = ((tid >> 6) & 1) * 32 + (lane & 15), wc = (tid >> 7) * 32 + (lane & 15);
        if (!kEarly) load_d();
        if (t.mode == 1)  // no pending panels: A was the panel itself, unsolved
#pragma unroll
            for (int i = 0; i < 2; ++i) own[i][0] = own[i][1] = typename Mfma<T>::acc_t{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int col = (tid >> 6) + 4 * j;
            if (row < t.m && col < t.n) C[row + (int64_t)col * t.ldc] = Cs[col][row];
        }
        if (wc <= wr) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const T* r = Cs[4 * q + (lane >> 4)];
                const T a0 = r[wr], a1 = r[wr + 16], b0 = r[wc], b1 = r[wc + 16];
                own[0][0] = Mfma<T>::mma(a0, b0, own[0][0]);
                own[0][1] = Mfma<T>::mma(a0, b1, own[0][1]);
                own[1][0] = Mfma<T>::mma(a1, b0, own[1][0]);
                own[1][1] = Mfma<T>::mma(a1, b1, own[1][1]);
            }
        }
        __syncthreads();
        stage_acc<T>(own, Cs);
        __syncthreads();
        T* D = pool + t.cd;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int col = (tid >> 6) + 4 * j;
            if (row < t.syrk && col <= row) D[row + (int64_t)col * t.ldc] = dpre[j] - Cs[col][row];
        }
        return;
    }
    if (row >= t.m) return;
    if (t.mode == 3 || t.mode == 0) {
        // C -= the product; mode 3 also adds the new entry into the parent
        // (one launch holds at most one child of each parent, and local_index
        // is injective within a child: no two lanes add into one entry).
        // Their loads (from clamped columns) are all issued before the stores,
        // which may alias them as far as the compiler knows: sixteen columns
        // at a time, four where C has been kept since before the K loop.
        const bool ea = t.mode == 3;
        T* P = ea ? pool + t.p + (lrow - 1) : C;
        constexpr int G = PRE ? 4 : 16;
#pragma unroll
        for (int k = 0; k < 16; k += G) {
            const int c0 = (tid >> 6) + 4 * k;
            if (c0 >= t.n) break;
            T pv[G];
            T* pp[G];
#pragma unroll
            for (int q = 0; q < G; ++q) {
                pp[q] = P + (ea ? (int64_t)(lcol[k + q] - 1) * t.np : 0);
                pv[q] = ea ? *pp[q] : T(0);
            }
#pragma unroll
            for (int q = 0; q < G; ++q) {
                const int col = c0 + 4 * q;
                if (col < t.n && (!t.tri || row >= col)) {
                    const T v = cpre[k + q] - Cs[col][row];
                    C[row + (int64_t)col * t.ldc] = v;
                    if (ea) *pp[q] = pv[q] + v;
                }
            }
        }
    } else {
        for (int col = tid >> 6; col < t.n; col += 4) C[row + (int64_t)col * t.ldc] = Cs[col][row];
    }
}

// LP != kNative: the update and Schur tiles (KIND 1, 2) of the FP16_IR /
// BF16_IR forms multiply 16-bit operands.
template <typename T, int KIND, int LP = kNative>
__global__ __launch_bounds__(kThreads, KIND == 0 ? 3 : 4) void k_gemm(T* pool, const GemmTask* tasks, const int* lidx)
{
    static_assert(LP == kNative || KIND != 0, "the panel TRSM stays in the front's precision");
    if constexpr (KIND == 0) {
        // panel TRSM tiles (modes 1 and 2): mode 2 keeps its first product
        // in Cs while staging the inverse through L, so the two are separate
        __shared__ TileLds<T> L;
        __shared__ T Cs[kTile][kTile + 1];
        const GemmTask t = tasks[blockIdx.x];
        if (t.syrk > 0)
            gemm_task<T, kNative, false, -1, 1, true>(pool, t, L, Cs);
        else
            gemm_task<T>(pool, t, L, Cs);
    } else {
        // modes 0 and 3 (B never transposed): the staged result Cs is written
        // after the last read of the operand staging L, so the two share LDS
        // (four workgroups per CU instead of three)
        __shared__ union {
            TileLds<T, 2> L;
            T Cs[kTile][kTile + 1];
        } u;
        gemm_task<T, LP, false, 0, 2>(pool, tasks[blockIdx.x], u.L, u.Cs, lidx);
    }
}

// One launch per panel step s of the large fronts: GemmTasks from workgroup
// ndiag on (the panel TRSM of the rows after block s+1, preceded by the
// update of those rows by the panels still pending for block column s, and,
// where small, the periodic in-panel update of the column blocks after s+1)
// and, below ndiag, the factorization of block s+1.  A diagonal workgroup
// applies the pending panels and panel s to its own block itself, forming
// (and storing) its rows' panel-s entries on the way, so no task of the
// launch reads what another one writes: the chain of diagonal blocks, the
// critical path, advances one block per launch.
//
// The diagonal task sends for all its operands at once and multiplies in
// strips: a wave has 16 rows of the block, so that its rows go from product
// to product without a barrier, and L_s^{-T}'s zeros and the block's upper
// triangle are left out (40 and at most 48 products of 16 x 16 x 4 a wave
// where whole squares take 64; 64 cycles each in FP64).  A step with nothing
// beside it takes 25 us in FP64 (30.5 with the operands in two batches, whole
// squares and every store at the end), 19 in FP32 (23).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_upd_diag(T* pool, const DiagTask* diags, int ndiag, const GemmTask* tiles,
                                                       int* info)
{
    __shared__ Front64<T> S;
    __shared__ union {
        TileLds<T, 2> L;      // GEMM tasks
        T B[2][64][kTile + 1];  // diagonal task: L_s^{-T}; block s's rows in the pending panels
    } U;
    if ((int)blockIdx.x >= ndiag) {
        const GemmTask g = tiles[blockIdx.x - ndiag];
        if (g.syrk > 0)
            gemm_task<T, kNative, true, -1, 2, true>(pool, g, U.L, S.A);
        else
            gemm_task<T, kNative, true, -1, 2>(pool, g, U.L, S.A);
        return;
    }
    typedef typename Mfma<T>::acc_t acc_t;
    const DiagTask t = diags[blockIdx.x];
    const int n = t.n, kb = t.kb, kp = t.kprev, kpp = t.kpp;
    T* front = pool + t.front;
    const T* C = front + t.k0 + (int64_t)t.k0 * n;                         // block s+1
    T* Pg = front + t.k0 + (int64_t)(t.k0 - kp) * n;                       // its rows in panel s
    const T* Xd = front + t.k0 + (int64_t)(t.k0 - kp - kpp) * n;          // its rows in the pending panels
    const T* Xs = front + (t.k0 - kp) + (int64_t)(t.k0 - kp - kpp) * n;   // block s's rows in them
    const T* inv = pool + t.inv - kPanel * kPanel;                         // L_s^{-T}
    const int tid = threadIdx.x, row = tid & 63, c4 = tid >> 6;
    const int lane = tid & 63, li = lane & 15, kl = lane >> 4, r0 = 16 * c4;  // the wave's strip of rows
    // Entry (row, c4 + 4 j) of each 64 x 64 block, and of the strip's rows of
    // the pending panels the MFMA operands (r0 + li, 4 q + kl); positions past
    // the block read entry 0 and are masked after the loads.
    const unsigned ra = row < kb ? row : 0u, rb = row < kp ? row : 0u, rx = r0 + li < kb ? r0 + li : 0u;
    auto load_pending = [&](int q0, T (&xs)[16], T (&xd)[16]) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int cs = q0 + c4 + 4 * j, cd = q0 + 4 * j + kl;
            xs[j] = ld_off(Xs, rb + (cs < kpp ? cs : 0u) * (unsigned)n);
            xd[j] = ld_off(Xd, rx + (cd < kpp ? cd : 0u) * (unsigned)n);
        }
    };
    auto stage_pending = [&](int q0, const T (&xs)[16]) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int col = c4 + 4 * j;
            U.B[1][col][row] = (row < kp && q0 + col < kpp) ? xs[j] : T(0);
        }
    };
    T xs[16], xd[16], rc[16], rp[16], ri[16];
    if (kpp > 0) load_pending(0, xs, xd);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int col = c4 + 4 * j;
        rp[j] = ld_off((const T*)Pg, ra + (col < kp ? col : 0u) * (unsigned)n);
        ri[j] = ld_off(inv, (unsigned)(tid + kThreads * j));
        rc[j] = ld_off(C, ra + (col <= row && row < kb ? col : 0u) * (unsigned)n);
    }
    if (kpp > 0) stage_pending(0, xs);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int col = c4 + 4 * j, e = tid + kThreads * j, k = e & 63, i = e >> 6;
        S.X[col][row] = (row < kb && col < kp) ? rp[j] : T(0);
        U.B[0][k][i] = (k < kp && i < kp) ? ri[j] : T(0);  // B[k][j] = L_s^{-1}[j][k] = inv[k + 64 j]
        S.A[col][row] = (row < kb && col <= row) ? rc[j] : T(0);
    }
    __syncthreads();
    // the pending panels (64 columns per round): S.X -= Xd Xs^T (they have
    // been applied to the block itself by the TRSM tile of its rows)
    if (kpp > 0) {
        acc_t c[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
        for (int q0 = 0; q0 < kpp; q0 += 64) {
            if (q0 > 0) {
                load_pending(q0, xs, xd);
                __syncthreads();
                stage_pending(q0, xs);
                __syncthreads();
            }
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const T a = (r0 + li < kb && q0 + 4 * q + kl < kpp) ? xd[q] : T(0);
#pragma unroll
                for (int j = 0; j < 4; ++j) c[j] = Mfma<T>::mma(a, U.B[1][4 * q + kl][16 * j + li], c[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) S.X[16 * j + li][r0 + Mfma<T>::row(lane, v)] -= c[j][v];
        wave_sync();
    }
    // X = S.X L_s^{-T}, whose column block j has rows up to its own
    {
        acc_t c[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const T a = S.X[4 * q + kl][r0 + li];
#pragma unroll
            for (int j = q / 4; j < 4; ++j) c[j] = Mfma<T>::mma(a, U.B[0][4 * q + kl][16 * j + li], c[j]);
        }
        wave_sync();
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) S.X[16 * j + li][r0 + Mfma<T>::row(lane, v)] = c[j][v];
    }
    __syncthreads();
    // S.A -= X X^T: the ten lower 16 x 16 blocks from three block rows of X a
    // wave, (o0, o1), (o0, o2) and (o2, o2) of (3, 0, 1), (3, 3, 2), (2, 0, 1),
    // (1, 0, 0)
    {
        const int o0 = 16 * (0x1233 >> 4 * c4 & 3), o1 = 16 * (0x0030 >> 4 * c4 & 3), o2 = 16 * (0x0121 >> 4 * c4 & 3);
        acc_t c[3] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const T* x = S.X[4 * q + kl] + li;
            const T x0 = x[o0], x1 = x[o1], x2 = x[o2];
            c[0] = Mfma<T>::mma(x0, x1, c[0]);
            if (c4 != 3) c[1] = Mfma<T>::mma(x0, x2, c[1]);
            if (c4 != 2) c[2] = Mfma<T>::mma(x2, x2, c[2]);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = Mfma<T>::row(lane, v);
            S.A[o1 + li][o0 + r] -= c[0][v];
            if (c4 != 3) S.A[o2 + li][o0 + r] -= c[1][v];
            if (c4 != 2) S.A[o2 + li][o2 + r] -= c[2][v];
        }
    }
    __syncthreads();
    // during the first panel's chain: X into the front (these rows are this
    // task's), then zero where the inverse is, above its diagonal blocks
    auto put_x = [&](int w) {
#pragma unroll 4
        for (int col = w; col < 64; col += 3) {
            if (row < kb && col < kp) Pg[row + (int64_t)col * n] = S.X[col][row];
            if (row < (col & ~15)) S.X[col][row] = T(0);
        }
    };
    factor_dense64_loaded<T>(S, front + t.k0 + (int64_t)t.k0 * n, n, kb, kb, info, t.first + t.k0, pool + t.inv, put_x);
}

// C -= A B^T on 128 x 128 tiles (GemmTask with m, n <= 128, mode 0 or 3):
// the Schur update of fronts with many update rows (and their extend-add,
// mode 3).  Each of the four waves owns a 64 x 64 quarter as 4 x 4 MFMA
// 16x16x4 blocks, so every operand read from LDS feeds four MFMAs (half the
// LDS reads and half the L2 traffic per flop of the 64 x 64 tile).  K is
// staged through LDS in chunks of 16, double buffered: chunk j+1's global
// loads are issued before chunk j's MFMAs and stored to the other buffer
// after them, one barrier per chunk.  A diagonal tile (tri) skips the
// quarter above the diagonal.  The result goes back one quarter at a time
// through LDS (coalesced along columns); mode 3 also adds each new entry
// into the parent front at the rows and columns local_index gives (one
// launch holds at most one child of each parent).
template <typename T> struct WideLds {
    union {
        struct {
            T As[2][16][132];
            T Bs[2][16][132];
        } k;
        T Cs[64][65];
    };
};
template <typename T> using WideAcc = typename Mfma<T>::acc_t[4][4];

// acc = sum over K columns [k0, k1) of A B^T (a multiple of 16 apart, or k1
// = K); ends with a barrier.
template <typename T, int LP>
__device__ __forceinline__ void wide_product(const T* pool, const GemmTask& t, int k0, int k1, WideAcc<T>& acc,
                                             WideLds<T>& u)
{
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15;
    const int wr = (wv & 1) * 64, wc = (wv >> 1) * 64;
    const bool skip = t.tri && wc > wr;  // quarter strictly above the diagonal
    const T* A = pool + t.a;
    const T* B = pool + t.b;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = typename Mfma<T>::acc_t{0, 0, 0, 0};
    const int lr = tid & 127, lk = tid >> 7;
    T ra[8], rb[8];
    auto load = [&](int kc) {
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            const int kk = kc + lk + 2 * p;
            ra[p] = (lr < t.m && kk < k1) ? A[lr + (int64_t)kk * t.lda] : T(0);
            rb[p] = (lr < t.n && kk < k1) ? B[lr + (int64_t)kk * t.ldb] : T(0);
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            u.k.As[buf][lk + 2 * p][lr] = ra[p];
            u.k.Bs[buf][lk + 2 * p][lr] = rb[p];
        }
    };
    load(k0);
    store(0);
    __syncthreads();
    const int nch = (k1 - k0 + 15) / 16;
    for (int j = 0; j < nch; ++j) {
        const int buf = j & 1;
        if (j + 1 < nch) load(k0 + 16 * (j + 1));
        if (!skip) {
            if constexpr (LP == kNative) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int kr = 4 * q + (lane >> 4);
                    T a[4], b[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        a[i] = u.k.As[buf][kr][wr + 16 * i + li];
                        b[i] = u.k.Bs[buf][kr][wc + 16 * i + li];
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int jj = 0; jj < 4; ++jj) acc[i][jj] = Mfma<T>::mma(a[i], b[jj], acc[i][jj]);
                }
            } else {
                typedef Mfma16<LP> M16;
                const int kr = 4 * (lane >> 4);
                typename M16::op_t a[4], b[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        a[i][e] = M16::cvt(u.k.As[buf][kr + e][wr + 16 * i + li]);
                        b[i][e] = M16::cvt(u.k.Bs[buf][kr + e][wc + 16 * i + li]);
                    }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int jj = 0; jj < 4; ++jj) acc[i][jj] = M16::mma(a[i], b[jj], acc[i][jj]);
            }
        }
        if (j + 1 < nch) store(buf ^ 1);
        __syncthreads();
    }
}

// C -= acc (and, mode 3, each new entry added into the parent front), or,
// with part != nullptr, acc stored as partial product `part` (four 64 x 64
// quarters, column-major); both through LDS one quarter at a time; ends with
// a barrier.
template <typename T>
__device__ __forceinline__ void wide_apply(T* pool, const GemmTask& t, const int* lidx, const WideAcc<T>& acc,
                                           WideLds<T>& u, T* part)
{
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15;
    T* C = pool + t.c;
    const bool ea = t.mode == 3;
    for (int w = 0; w < 4; ++w) {
        const int qr = (w & 1) * 64, qc = (w >> 1) * 64;
        if ((t.tri && qc > qr) || qr >= t.m || qc >= t.n) continue;  // uniform
        if (wv == w) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                    for (int v = 0; v < 4; ++v) u.Cs[16 * jj + li][16 * i + Mfma<T>::row(lane, v)] = acc[i][jj][v];
        }
        __syncthreads();
        const int row = tid & 63, gr = qr + row;
        if (part) {
            T* Q = part + w * 4096 + row;
            for (int col = tid >> 6; col < 64; col += 4) Q[col * 64] = u.Cs[col][row];
        } else if (gr < t.m) {
            T* P = ea ? pool + t.p + (lidx[t.li + gr] - 1) : C;
            for (int c0 = tid >> 6; c0 < 64; c0 += 16) {
                T cv[4], pv[4];
                int64_t po[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int gc = min(qc + c0 + 4 * q, t.n - 1);
                    cv[q] = C[gr + (int64_t)gc * t.ldc];
                    po[q] = ea ? (int64_t)(lidx[t.lj + gc] - 1) * t.np : 0;
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) pv[q] = ea ? P[po[q]] : T(0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int col = c0 + 4 * q, gc = qc + col;
                    if (gc < t.n && (!t.tri || gr >= gc)) {
                        const T v = cv[q] - u.Cs[col][row];
                        C[gr + (int64_t)gc * t.ldc] = v;
                        if (ea) P[po[q]] = pv[q] + v;
                    }
                }
            }
        }
        __syncthreads();
    }
}

// The tiles' K loops divided evenly over the workgroups (every workgroup
// takes a run of 16-column K chunks, which may start and end inside a
// tile), so that a launch has no partly filled last round: workgroup w
// takes segments [seg_ptr[w], seg_ptr[w + 1]).  A segment covering its
// tile's whole K applies its product at once; the others store their
// partial products (slot: four 64 x 64 quarters, column-major, staged
// through LDS) for k_gemm_fix, which adds them in segment order and applies
// the sum.  Nothing waits on another workgroup.
template <typename T, int LP = kNative>
__global__ __launch_bounds__(kThreads, 2) void k_gemm_seg(T* pool, const GemmTask* tasks, const SegTask* segs,
                                                          const int* seg_ptr, T* part, const int* lidx)
{
    __shared__ WideLds<T> u;
    for (int s = seg_ptr[blockIdx.x]; s < seg_ptr[blockIdx.x + 1]; ++s) {
        const SegTask g = segs[s];
        const GemmTask t = tasks[g.task];
        WideAcc<T> acc;
        wide_product<T, LP>(pool, t, g.k0, g.k1, acc, u);
        wide_apply<T>(pool, t, lidx, acc, u, g.slot < 0 ? nullptr : part + (int64_t)g.slot * 16384);
    }
}

// Tiles whose K was split: C -= the partial products of slots slot0 ..
// slot0 + nslot - 1 added in that order (and, mode 3, each new entry added
// into the parent front), quarter by quarter like wide_apply.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_gemm_fix(T* pool, const GemmTask* tasks, const FixTask* fixes,
                                                       const T* part, const int* lidx)
{
    const FixTask f = fixes[blockIdx.x];
    const GemmTask t = tasks[f.task];
    const int tid = threadIdx.x, row = tid & 63;
    T* C = pool + t.c;
    const bool ea = t.mode == 3;
    for (int w = 0; w < 4; ++w) {
        const int qr = (w & 1) * 64, qc = (w >> 1) * 64, gr = qr + row;
        if ((t.tri && qc > qr) || qr >= t.m || qc >= t.n || gr >= t.m) continue;
        const T* Q = part + (int64_t)f.slot0 * 16384 + w * 4096 + row;
        T* P = ea ? pool + t.p + (lidx[t.li + gr] - 1) : C;
        for (int col = tid >> 6; col < 64; col += 4) {
            const int gc = qc + col;
            if (gc >= t.n || (t.tri && gr < gc)) continue;
            T sum = Q[col * 64];
            for (int sl = 1; sl < f.nslot; ++sl) sum += Q[(int64_t)sl * 16384 + col * 64];
            const T v = C[gr + (int64_t)gc * t.ldc] - sum;
            C[gr + (int64_t)gc * t.ldc] = v;
            if (ea) {
                T* pp = P + (int64_t)(lidx[t.lj + gc] - 1) * t.np;
                *pp = *pp + v;
            }
        }
    }
}

// Diagonal block [k0, k0+kb) of a large front, already updated by every
// earlier panel (DPOTRF("U"), factorize_kernel_m.f90:4-9): L written back
// into the front, and the inverse of L stored for the panel TRSM and the
// solves.  As many workgroups per CU as its LDS allows: two in FP64, four in
// FP32.
template <typename T>
__global__ __launch_bounds__(kThreads, sizeof(T) == 8 ? 2 : 4) void k_diag(T* pool, const DiagTask* tasks, int* info)
{
    const DiagTask t = tasks[blockIdx.x];
    __shared__ Front64<T> S;
    factor_dense64<T>(S, pool + t.front + t.k0 + (int64_t)t.k0 * t.n, t.n, t.kb, t.kb, info, t.first + t.k0,
                      pool + t.inv);
}

// ---------------------------------------------------------- medium fronts
// The whole partial factorization of one front per workgroup, for fronts
// larger than one 64 x 64 LDS block whose 64-column steps would leave most
// of the chip idle (many such fronts share a level): panel by panel,
//   1. the kb x kb diagonal block factored and inverted in LDS
//      (factor_dense64: DPOTRF, factorize_kernel_m.f90:4-9), its inverse
//      stored for the solves;
//   2. the rows below it solved against that inverse, in place, one 64-row
//      MFMA tile at a time (the panel TRSM, factorize_kernel_m.f90:11-16);
//   3. the trailing lower triangle -- pivot columns and update matrix --
//      updated by the panel, one 64 x 64 MFMA tile at a time with K = kb
//      (DSYRK / DGEMM, factorize_kernel_m.f90:18-33).
// The workgroup owns its front, so workgroup barriers order the phases; no
// tile of a phase reads what another tile of it writes.  LP rounds the
// update tiles' operands to 16 bits (the FP16_IR / BF16_IR forms).  With
// clocks != nullptr, task i's start and end (wall_clock64, 100 MHz) go to
// clocks[2 i], clocks[2 i + 1]: the per-front timings of the schedule tuner.
template <typename T> union FrontLds {
    Front64<T> D;
    struct {
        TileLds<T, 2> L;
        T Cs[kTile][kTile + 1];
    } G;
};
// One tile of k_front_wg, kept out of line: the medium-front kernel's
// registers are then those of its diagonal phase (the call's saved registers
// on the stack) instead of the sum of both phases.  The LDS comes by its own
// address space: through generic pointers each access to it would count as a
// memory access and wait for the loads of the next chunks.  In FP64 the tile's
// entries of C come before its K loop (24^3 grid, one front after another:
// 10.6 ms against 11.3 after it); in FP32, where the loop is shorter than the
// loads, after it (9.1 against 9.3).
template <typename T, int LP>
__device__ __attribute__((noinline)) void front_tile(T* pool, GemmTask g, __attribute__((address_space(3))) FrontLds<T>* U)
{
    FrontLds<T>* u = (FrontLds<T>*)U;
    gemm_task<T, LP, sizeof(T) == 8, -1, 2>(pool, g, u->G.L, u->G.Cs);
}
// Two workgroups per CU, in both types: left to itself the compiler takes
// registers for one, with which 256 systems of a batch, all their fronts
// medium, take 9.2 ms in FP64 and 7.4 in FP32 instead of 7.25 and 5.4.
template <typename T, int LP>
__global__ __launch_bounds__(kThreads, 2) void k_front_wg(T* pool, const NodeDev* nodes, const int* tasks, int* info,
                                                       long long* clocks)
{
    long long t_start = 0;
    if (clocks) t_start = wall_clock64();
    const NodeDev nd = nodes[tasks[blockIdx.x]];
    __shared__ FrontLds<T> U;
    auto* lds = (__attribute__((address_space(3))) FrontLds<T>*)&U;
    const int n = nd.n, c = nd.c;
    for (int k0 = 0; k0 < c; k0 += kPanel) {
        const int kb = min(kPanel, c - k0);
        const int64_t inv = nd.inv + (int64_t)(k0 / kPanel) * kPanel * kPanel;
        factor_dense64<T>(U.D, pool + nd.front + k0 + (int64_t)k0 * n, n, kb, kb, info, nd.first + k0, pool + inv);
        __syncthreads();
        for (int r0 = k0 + kb; r0 < n; r0 += kTile) {
            GemmTask g{};
            g.c = g.a = nd.front + r0 + (int64_t)k0 * n;
            g.ldc = g.lda = n;
            g.b = inv;  // L^{-T}, read transposed
            g.ldb = kPanel;
            g.m = min(kTile, n - r0);
            g.n = g.k = kb;
            g.mode = 1;
            front_tile<T, kNative>(pool, g, lds);
            __syncthreads();
        }
        for (int c0 = k0 + kb; c0 < n; c0 += kTile)
            for (int r0 = c0; r0 < n; r0 += kTile) {
                GemmTask g{};
                g.c = nd.front + r0 + (int64_t)c0 * n;
                g.a = nd.front + r0 + (int64_t)k0 * n;
                g.b = nd.front + c0 + (int64_t)k0 * n;
                g.ldc = g.lda = g.ldb = n;
                g.m = min(kTile, n - r0);
                g.n = min(kTile, n - c0);
                g.k = kb;
                g.tri = r0 == c0;
                front_tile<T, LP>(pool, g, lds);
                __syncthreads();
            }
    }
    if (clocks && threadIdx.x == 0) {
        clocks[2 * blockIdx.x] = t_start;
        clocks[2 * blockIdx.x + 1] = wall_clock64();
    }
}

// ------------------------------------------------------------ superblocks
// The three 256 x 256 matrices of superblock u, column-major, X at xoff, W
// at xoff + 256^2 (u >= 1), V at xoff + 2 256^2 (superblock u+1 not empty):
//   X = inverse of the superblock's diagonal block of L (zero past its
//       width sb), by 64 x 64 blocks (i, j), j <= i: X_ii is the stored
//       64 x 64 inverse (j = i; the row's blocks above the diagonal cleared,
//       the whole row past sb) and X_ij = -X_ii sum_{k=j}^{i-1} L_ik X_kj;
//   W = X L[B_u, B_{u-1}] (4 <= j < 8: block (i, j - 4)), the coupling of
//       the superblock to the previous one, so that y_u = X z_u - W y_{u-1};
//   V = L[B_{u+1}, B_u] X (j >= 8: block (i, j - 8), rows of superblock
//       u+1), so that x_u = X^T (y_u - q_u) - V^T x_{u+1}.
// A task forms 16 columns of X from block row j = t.j / 4 down, one row after
// another (they depend on no other column): the columns so far are in LDS, a
// wave has 16 rows of the block row in work and takes the blocks of L and the
// stored inverse straight into MFMA operands, a block ahead.  Bound by the
// latency of that chain (up to nine products of 64 x 16 x 64).  As a launch
// per block distance with a whole 64 x 64 block a workgroup, off the matrix
// cores, the last front's superblocks took 110 us (one superblock) to 185 us
// (64^3 workload, 122 of them) in FP64 where this takes 18 and 106.  The W and
// V blocks follow in one launch of k_superwv.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_superinv(const T* pool, T* sinv, const NodeDev* nodes,
                                                       const SuperInvTask* tasks)
{
    typedef typename Mfma<T>::acc_t acc_t;
    const SuperInvTask t = tasks[blockIdx.x];
    const NodeDev nd = nodes[t.node];
    const int n = nd.n, c0 = kSuper * t.u, sb = min(kSuper, nd.c - c0), j = t.j >> 2, s0 = 16 * (t.j & 3);
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kl = lane >> 4, r0 = 16 * (tid >> 6);
    T* X = sinv + t.xoff + kSuper * (64 * j + s0);  // the task's columns
    __shared__ T Xs[4][64][17];  // X, block row, row, column
    __shared__ T Ss[64][17];     // sum_k L_ik X_kj
    const T* inv = pool + nd.inv + (int64_t)(c0 / 64) * 4096;  // block i's: inv[4096 i + r + 64 q] = L^{-1}(q, r)
    const int nblk = (sb + 63) / 64;                           // block rows in use
    // X_jj from the stored inverse; zero above it and past the superblock
    for (int e = tid; e < kSuper * 16; e += kThreads) {
        const int r = e & 255, col = e >> 8, i = r >> 6, kb = min(64, sb - 64 * j);
        if (i > j && i < nblk) continue;
        T v = T(0);
        if (i == j && (r & 63) < kb && s0 + col < kb) v = inv[4096 * j + (s0 + col) + 64 * (r & 63)];
        if (i == j) Xs[j][r & 63][col] = v;
        X[r + kSuper * col] = v;
    }
    __syncthreads();
    for (int i = j + 1; i < nblk; ++i) {
        const int kbi = min(64, sb - 64 * i);
        // entry (r0 + li, 4 q + kl) of L_ik, rows past kbi masked
        const T* Lr = pool + nd.front + c0 + 64 * i + min(r0 + li, kbi - 1) + (int64_t)(c0 + kl) * n;
        T a[16], an[16];
        auto load = [&](T (&x)[16], int k) {
#pragma unroll
            for (int q = 0; q < 16; ++q) x[q] = Lr[(int64_t)(64 * k + 4 * q) * n];
        };
        load(a, j);
        acc_t acc = {0, 0, 0, 0};
        for (int k = j; k < i; ++k) {
            if (k + 1 < i)
                load(an, k + 1);
            else
#pragma unroll
                for (int q = 0; q < 16; ++q) an[q] = inv[4096 * i + 4 * q + kl + 64 * (r0 + li)];
#pragma unroll
            for (int q = 0; q < 16; ++q)
                acc = Mfma<T>::mma(r0 + li < kbi ? a[q] : T(0), Xs[k][4 * q + kl][li], acc);
#pragma unroll
            for (int q = 0; q < 16; ++q) a[q] = an[q];
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) Ss[r0 + Mfma<T>::row(lane, v)][li] = acc[v];
        __syncthreads();
        acc = {0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < 16; ++q) acc = Mfma<T>::mma(a[q], Ss[4 * q + kl][li], acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = r0 + Mfma<T>::row(lane, v);
            Xs[i][r][li] = -acc[v];
            X[64 * i + r + kSuper * li] = -acc[v];
        }
        __syncthreads();
    }
}

// The W and V blocks of the superblock matrices (tasks with j >= 4, see
// k_superinv) as single MFMA tile products with K up to 256:
//   W block (i, j - 4) = X[block row i, :] L[B_u, B_{u-1} block j - 4]
//       (X is zero right of its diagonal block, so K = min(64 (i + 1), sb));
//   V block (i, j - 8) = L[B_{u+1} block i, B_u from block j - 8]
//       X[B_u from block j - 8, block j - 8] (X is zero above it).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_superwv(const T* pool, T* sinv, const NodeDev* nodes,
                                                      const SuperInvTask* tasks)
{
    const SuperInvTask t = tasks[blockIdx.x];
    const NodeDev nd = nodes[t.node];
    T* X = sinv + t.xoff;
    const int n = nd.n, c0 = kSuper * t.u, sb = min(kSuper, nd.c - c0), i = t.i;
    const T* F = pool + nd.front;
    __shared__ union {
        TileLds<T> L;
        T Cs[kTile][kTile + 1];
    } u;
    T* dst;
    const int row = threadIdx.x & 63;
    if (t.j >= 8) {
        const int jv = t.j - 8, rv = c0 + kSuper + 64 * i;
        const int m = min(64, nd.c - rv);
        if (m < 1) {  // past a partial superblock's last row
            dst = X + 2 * kSuper * kSuper + 64 * i + kSuper * 64 * jv;
            for (int col = threadIdx.x >> 6; col < 64; col += 4) dst[row + kSuper * col] = T(0);
            return;
        }
        tile_product<T, kNative, 1>(F + rv + (int64_t)(c0 + 64 * jv) * n, n, X + kSuper * 64 * jv + 64 * jv, kSuper, true, m, 64,
                        kSuper - 64 * jv, u.L, u.Cs);
        dst = X + 2 * kSuper * kSuper + 64 * i + kSuper * 64 * jv;
    } else {
        const int jw = t.j - 4, cp = c0 - kSuper;
        tile_product<T, kNative, 1>(X + 64 * i, kSuper, F + c0 + (int64_t)(cp + 64 * jw) * n, n, true, 64, 64, min(64 * (i + 1), sb),
                        u.L, u.Cs);
        dst = X + kSuper * kSuper + 64 * i + kSuper * 64 * jw;
    }
    for (int col = threadIdx.x >> 6; col < 64; col += 4) dst[row + kSuper * col] = u.Cs[col][row];
}

// ----------------------------------------------- permutations and residual
// out[i + r*ld_out] = in[perm[i] + r*ld_in] (perm 0-based)
__global__ __launch_bounds__(kThreads) void k_gather_rows(double* out, int ld_out, const double* in, int ld_in,
                                                          const int* perm, int n, int nrhs)
{
    int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (e >= (int64_t)n * nrhs) return;
    int i = (int)(e % n), r = (int)(e / n);
    out[i + (int64_t)r * ld_out] = in[perm[i] + (int64_t)r * ld_in];
}
// out[perm[i] + r*ld_out] = in[i + r*ld_in]
__global__ __launch_bounds__(kThreads) void k_scatter_rows(double* out, int ld_out, const double* in, int ld_in,
                                                           const int* perm, int n, int nrhs)
{
    int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (e >= (int64_t)n * nrhs) return;
    int i = (int)(e % n), r = (int)(e / n);
    out[perm[i] + (int64_t)r * ld_out] = in[i + (int64_t)r * ld_in];
}

// ------------------------------------------------------ FP64 refinement
// r = b - A x over the full symmetric matrix in CSR order (val: the values
// in that order, gathered once per factorization), four right-hand sides per
// pass over a row.  G lanes take a row's entries G apart, so that a wave reads
// consecutive entries of 64 / G rows, and their sums are added pairwise (a
// fixed order).  What bounds it is the entries' 12 bytes each, once from
// memory: one lane per row read every line of them 64 / G times over and
// took 506 us on the 40^3 three-unknown stencil (15.0M entries).
template <int G>
__global__ __launch_bounds__(kThreads) void k_residual(double* r, const double* b, const double* x, int n, int nrhs,
                                                       const int* ptr, const int* col, const double* val)
{
    const int row = blockIdx.x * (kThreads / G) + (int)threadIdx.x / G, g = threadIdx.x % G;
    const int at = min(row, n - 1);  // lanes past the last row repeat it and store nothing
    const int e0 = ptr[at], e1 = ptr[at + 1];
    for (int k0 = 0; k0 < nrhs; k0 += 4) {
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        for (int e = e0 + g; e < e1; e += G) {
            const double v = val[e];
            const double* xc = x + col[e] + (int64_t)k0 * n;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (k0 + q < nrhs) acc[q] += v * xc[(int64_t)q * n];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int off = G / 2; off > 0; off >>= 1) acc[q] += __shfl_xor(acc[q], off);
            if (g == 0 && row < n && k0 + q < nrhs)
                r[row + (int64_t)(k0 + q) * n] = b[row + (int64_t)(k0 + q) * n] - acc[q];
        }
    }
}

// Maximum over the workgroup, then one atomic per workgroup (as IEEE bits:
// order-preserving for non-negative doubles, so the result is exact).
__device__ __forceinline__ void block_max_to(unsigned long long* out, double m)
{
    __shared__ double wmax[kThreads / 64];
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; ++w) m = fmax(m, wmax[w]);
        atomicMax(out, (unsigned long long)__double_as_longlong(m));
    }
}

// The norms a backward error needs, in one pass, per column k (blockIdx.y)
// of the n x nrhs vectors r, x, b and (if not null) d, ld n: the maxima of
// |r|, |x|, |b|, |d| into out[k], out[nrhs + k], out[2 nrhs + k], out[3 nrhs
// + k] (IEEE bits, one atomic per workgroup: order-preserving for
// non-negative doubles, so exact), and the sums of squares of r and x as
// per-workgroup partials part[k parts + w], part[(nrhs + k) parts + w] (parts
// = gridDim.x), which the caller adds in order, so the sums do not depend on
// the timing of the workgroups.
__global__ __launch_bounds__(kThreads) void k_err_norms(unsigned long long* out, double* part, const double* r,
                                                        const double* x, const double* b, const double* d, int64_t n,
                                                        int nrhs)
{
    __shared__ double red[6][kThreads / 64];
    const int k = blockIdx.y;
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};  // max |r|, |x|, |b|, |d|; sum r^2, x^2
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        const int64_t e = i + (int64_t)k * n;
        const double rv = r[e], xv = x[e], bv = b[e], dv = d ? d[e] : 0.0;
        v[0] = fmax(v[0], fabs(rv));
        v[1] = fmax(v[1], fabs(xv));
        v[2] = fmax(v[2], fabs(bv));
        v[3] = fmax(v[3], fabs(dv));
        v[4] += rv * rv;
        v[5] += xv * xv;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const double o = __shfl_xor(v[q], off);
            v[q] = q < 4 ? fmax(v[q], o) : v[q] + o;
        }
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int q = 0; q < 6; ++q) red[q][threadIdx.x >> 6] = v[q];
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; ++w)
#pragma unroll
            for (int q = 0; q < 6; ++q) v[q] = q < 4 ? fmax(v[q], red[q][w]) : v[q] + red[q][w];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q < 3 || d) atomicMax(out + q * nrhs + k, (unsigned long long)__double_as_longlong(v[q]));
        part[(int64_t)k * gridDim.x + blockIdx.x] = v[4];
        part[(int64_t)(nrhs + k) * gridDim.x + blockIdx.x] = v[5];
    }
}

// val[e] = a[src[e]], the caller's values in CSR order, and out[0] = max over
// rows of sum_e |val[e]|, the infinity norm of A (zeroed by the caller), in
// one pass over the entries, G lanes per row as in k_residual (apart, and one
// lane per row for the norm, they took 82 and 78 us on the 40^3 three-unknown
// stencil).
template <int G>
__global__ __launch_bounds__(kThreads) void k_gather_vals(unsigned long long* out, double* val, const double* a,
                                                          const int64_t* src, int n, const int* ptr)
{
    const int g = threadIdx.x % G;
    double m = 0.0;
    for (int row = blockIdx.x * (kThreads / G) + (int)threadIdx.x / G; row < n; row += gridDim.x * (kThreads / G)) {
        double s = 0.0;
        for (int e = ptr[row] + g; e < ptr[row + 1]; e += G) {
            const double v = a[src[e]];
            val[e] = v;
            s += fabs(v);
        }
#pragma unroll
        for (int off = G / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
        m = fmax(m, s);
    }
    block_max_to(out, m);
}

__global__ __launch_bounds__(kThreads) void k_axpy(double* x, const double* d, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < n) x[i] += d[i];
}

__global__ void k_zero_u64(unsigned long long* p, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0ull;
}

// Lanes per row of the CSR kernels: about a third of a row's entries, so that
// few lanes idle on the last ones (4 for the 7-point grids, 8 and 32 for the
// 27-point ones with one and three unknowns, 16 with two).  A band of 150,000
// rows, four right-hand sides: 45 entries a row 63 us with 32 lanes, 43 with
// 16; 59 entries 66 and 53; 41 entries 42 with 8.
static int row_lanes(int n, int64_t nnz)
{
    const int64_t per = nnz / n;
    return per <= 12 ? 4 : per <= 40 ? 8 : per <= 72 ? 16 : 32;
}
void launch_residual(double* r, const double* b, const double* x, int n, int nrhs, const int* ptr, const int* col,
                     const double* val, int64_t nnz, hipStream_t st)
{
    if (n <= 0) return;
    const int g = row_lanes(n, nnz);
    const dim3 grid((unsigned)(((int64_t)n * g + kThreads - 1) / kThreads)), block(kThreads);
    if (g == 4)
        hipLaunchKernelGGL(k_residual<4>, grid, block, 0, st, r, b, x, n, nrhs, ptr, col, val);
    else if (g == 8)
        hipLaunchKernelGGL(k_residual<8>, grid, block, 0, st, r, b, x, n, nrhs, ptr, col, val);
    else if (g == 16)
        hipLaunchKernelGGL(k_residual<16>, grid, block, 0, st, r, b, x, n, nrhs, ptr, col, val);
    else
        hipLaunchKernelGGL(k_residual<32>, grid, block, 0, st, r, b, x, n, nrhs, ptr, col, val);
}
// (at most 2048 workgroups, each one atomic on the norm)
void launch_gather_vals(unsigned long long* out, double* val, const double* a, const int64_t* src, int n,
                        const int* ptr, int64_t nnz, hipStream_t st)
{
    if (n <= 0) return;
    const int g = row_lanes(n, nnz);
    const dim3 grid((unsigned)std::min<int64_t>(((int64_t)n * g + kThreads - 1) / kThreads, 2048)), block(kThreads);
    if (g == 4)
        hipLaunchKernelGGL(k_gather_vals<4>, grid, block, 0, st, out, val, a, src, n, ptr);
    else if (g == 8)
        hipLaunchKernelGGL(k_gather_vals<8>, grid, block, 0, st, out, val, a, src, n, ptr);
    else if (g == 16)
        hipLaunchKernelGGL(k_gather_vals<16>, grid, block, 0, st, out, val, a, src, n, ptr);
    else
        hipLaunchKernelGGL(k_gather_vals<32>, grid, block, 0, st, out, val, a, src, n, ptr);
}
// at least 8 entries per thread: few workgroups per column, so few atomics
// on each maximum and a short read-back of the partial sums
int sumsq_parts(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(n / (8 * kThreads), kSumParts)); }
void launch_err_norms(unsigned long long* out, double* part, const double* r, const double* x, const double* b,
                      const double* d, int64_t n, int nrhs, hipStream_t st)
{
    if (n > 0)
        hipLaunchKernelGGL(k_err_norms, dim3(sumsq_parts(n), nrhs), dim3(kThreads), 0, st, out, part, r, x, b, d, n, nrhs);
}
void launch_axpy(double* x, const double* d, int64_t n, hipStream_t st)
{
    if (n > 0) hipLaunchKernelGGL(k_axpy, dim3((unsigned)((n + kThreads - 1) / kThreads)), dim3(kThreads), 0, st, x, d, n);
}
void launch_zero_u64(unsigned long long* p, int n, hipStream_t st)
{
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, st, p, n);
}

__global__ void k_set_int(int* p, int v) { *p = v; }

// ------------------------------------------------------------- launchers
void launch_set_int(int* p, int v, hipStream_t st) { hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, st, p, v); }

template <typename T>
void launch_assemble(T* pool, const NodeDev* nodes, const FillTask* tasks, int count, const double* a,
                     const int64_t* dst, const int64_t* src, const int2* rc, const double* scale, hipStream_t st)
{
    if (count > 0)
        hipLaunchKernelGGL(k_assemble<T>, dim3(count), dim3(kThreads), 0, st, pool, nodes, tasks, a, dst, src, rc,
                           scale);
}
template <typename T>
void launch_pull_children(T* pool, const int* lidx, const NodeDev* nodes, const PullTask* tasks, int count,
                          const int* children, hipStream_t st)
{
    if (count > 0)
        hipLaunchKernelGGL(k_pull_children<T>, dim3(count), dim3(kThreads), 0, st, pool, lidx, nodes, tasks, children);
}
template <typename T>
void launch_extend_add(T* pool, const int* lidx, const NodeDev* nodes, const ExtTask* tasks, int count, hipStream_t st)
{
    if (count > 0) hipLaunchKernelGGL(k_extend_add<T>, dim3(count), dim3(kThreads), 0, st, pool, lidx, nodes, tasks);
}
template <typename T>
void launch_small_front(T* pool, const NodeDev* nodes, const int* tasks, int count, int* info, hipStream_t st)
{
    if (count > 0) hipLaunchKernelGGL(k_small_front<T>, dim3(count), dim3(kThreads), 0, st, pool, nodes, tasks, info);
}
template <typename T>
void launch_front_wg(T* pool, const NodeDev* nodes, const int* tasks, int count, int* info, long long* clocks,
                     hipStream_t st, int lowp)
{
    if (count <= 0) return;
    if constexpr (sizeof(T) == 4) {
        if (lowp == kF16) {
            hipLaunchKernelGGL((k_front_wg<T, kF16>), dim3(count), dim3(kThreads), 0, st, pool, nodes, tasks, info, clocks);
            return;
        }
        if (lowp == kBF16) {
            hipLaunchKernelGGL((k_front_wg<T, kBF16>), dim3(count), dim3(kThreads), 0, st, pool, nodes, tasks, info,
                               clocks);
            return;
        }
    }
    hipLaunchKernelGGL((k_front_wg<T, kNative>), dim3(count), dim3(kThreads), 0, st, pool, nodes, tasks, info, clocks);
}
template <typename T>
void launch_diag(T* pool, const DiagTask* tasks, int count, int* info, hipStream_t st)
{
    if (count > 0) hipLaunchKernelGGL(k_diag<T>, dim3(count), dim3(kThreads), 0, st, pool, tasks, info);
}
template <typename T>
void launch_upd_diag(T* pool, const DiagTask* diags, int ndiag, const GemmTask* tiles, int ntiles,
                     int* info, hipStream_t st)
{
    if (ndiag + ntiles > 0)
        hipLaunchKernelGGL(k_upd_diag<T>, dim3(ndiag + ntiles), dim3(kThreads), 0, st, pool, diags, ndiag, tiles,
                           info);
}
template <typename T>
void launch_gemm(T* pool, const GemmTask* tasks, int count, int kind, const int* lidx, hipStream_t st, int lowp)
{
    if (count <= 0) return;
    if constexpr (sizeof(T) == 4) {
        if (lowp == kF16 && kind != 0) {
            if (kind == 1)
                hipLaunchKernelGGL((k_gemm<T, 1, kF16>), dim3(count), dim3(kThreads), 0, st, pool, tasks, lidx);
            else
                hipLaunchKernelGGL((k_gemm<T, 2, kF16>), dim3(count), dim3(kThreads), 0, st, pool, tasks, lidx);
            return;
        }
        if (lowp == kBF16 && kind != 0) {
            if (kind == 1)
                hipLaunchKernelGGL((k_gemm<T, 1, kBF16>), dim3(count), dim3(kThreads), 0, st, pool, tasks, lidx);
            else
                hipLaunchKernelGGL((k_gemm<T, 2, kBF16>), dim3(count), dim3(kThreads), 0, st, pool, tasks, lidx);
            return;
        }
    }
    if (kind == 0)
        hipLaunchKernelGGL((k_gemm<T, 0>), dim3(count), dim3(kThreads), 0, st, pool, tasks, lidx);
    else if (kind == 1)
        hipLaunchKernelGGL((k_gemm<T, 1>), dim3(count), dim3(kThreads), 0, st, pool, tasks, lidx);
    else
        hipLaunchKernelGGL((k_gemm<T, 2>), dim3(count), dim3(kThreads), 0, st, pool, tasks, lidx);
}
void launch_diag_scale(double* s, const double* a, const int64_t* diag_src, int n, hipStream_t st)
{
    if (n > 0) hipLaunchKernelGGL(k_diag_scale, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, st, s, a, diag_src, n);
}
void launch_scale_rows(double* out, const double* in, const double* s, int n, int nrhs, hipStream_t st)
{
    const int64_t m = (int64_t)n * nrhs;
    if (m > 0)
        hipLaunchKernelGGL(k_scale_rows, dim3((unsigned)((m + kThreads - 1) / kThreads)), dim3(kThreads), 0, st, out, in,
                           s, n, nrhs);
}
template <typename T>
void launch_gemm_seg(T* pool, const GemmTask* tasks, const SegTask* segs, const int* seg_ptr, int groups,
                     const FixTask* fixes, int nfix, T* part, const int* lidx, hipStream_t st, int lowp)
{
    if (groups <= 0) return;
    if constexpr (sizeof(T) == 4) {
        if (lowp == kF16)
            hipLaunchKernelGGL((k_gemm_seg<T, kF16>), dim3(groups), dim3(kThreads), 0, st, pool, tasks, segs, seg_ptr,
                               part, lidx);
        else if (lowp == kBF16)
            hipLaunchKernelGGL((k_gemm_seg<T, kBF16>), dim3(groups), dim3(kThreads), 0, st, pool, tasks, segs, seg_ptr,
                               part, lidx);
        else
            hipLaunchKernelGGL((k_gemm_seg<T, kNative>), dim3(groups), dim3(kThreads), 0, st, pool, tasks, segs,
                               seg_ptr, part, lidx);
    } else {
        hipLaunchKernelGGL((k_gemm_seg<T, kNative>), dim3(groups), dim3(kThreads), 0, st, pool, tasks, segs, seg_ptr,
                           part, lidx);
    }
    if (nfix > 0)
        hipLaunchKernelGGL(k_gemm_fix<T>, dim3(nfix), dim3(kThreads), 0, st, pool, tasks, fixes, part, lidx);
}
template <typename T>
void launch_superinv(const T* pool, T* sinv, const NodeDev* nodes, const SuperInvTask* tasks, int count, bool wv,
                     hipStream_t st)
{
    if (count <= 0) return;
    if (wv)
        hipLaunchKernelGGL(k_superwv<T>, dim3(count), dim3(kThreads), 0, st, pool, sinv, nodes, tasks);
    else
        hipLaunchKernelGGL(k_superinv<T>, dim3(count), dim3(kThreads), 0, st, pool, sinv, nodes, tasks);
}
void launch_gather_rows(double* out, int ld_out, const double* in, int ld_in, const int* perm, int n, int nrhs,
                        hipStream_t st)
{
    int64_t tot = (int64_t)n * nrhs;
    if (tot > 0)
        hipLaunchKernelGGL(k_gather_rows, dim3((unsigned)((tot + kThreads - 1) / kThreads)), dim3(kThreads), 0, st, out,
                           ld_out, in, ld_in, perm, n, nrhs);
}
void launch_scatter_rows(double* out, int ld_out, const double* in, int ld_in, const int* perm, int n, int nrhs,
                         hipStream_t st)
{
    int64_t tot = (int64_t)n * nrhs;
    if (tot > 0)
        hipLaunchKernelGGL(k_scatter_rows, dim3((unsigned)((tot + kThreads - 1) / kThreads)), dim3(kThreads), 0, st,
                           out, ld_out, in, ld_in, perm, n, nrhs);
}

#define MFD_INSTANTIATE(T)                                                                                             \
    template void launch_assemble<T>(T*, const NodeDev*, const FillTask*, int, const double*, const int64_t*,          \
                                     const int64_t*, const int2*, const double*, hipStream_t);                         \
    template void launch_pull_children<T>(T*, const int*, const NodeDev*, const PullTask*, int, const int*,            \
                                          hipStream_t);                                                                \
    template void launch_extend_add<T>(T*, const int*, const NodeDev*, const ExtTask*, int, hipStream_t);              \
    template void launch_small_front<T>(T*, const NodeDev*, const int*, int, int*, hipStream_t);                       \
    template void launch_front_wg<T>(T*, const NodeDev*, const int*, int, int*, long long*, hipStream_t, int);           \
    template void launch_diag<T>(T*, const DiagTask*, int, int*, hipStream_t);                                        \
    template void launch_upd_diag<T>(T*, const DiagTask*, int, const GemmTask*, int, int*, hipStream_t);                \
    template void launch_gemm<T>(T*, const GemmTask*, int, int, const int*, hipStream_t, int);                         \
    template void launch_superinv<T>(const T*, T*, const NodeDev*, const SuperInvTask*, int, bool, hipStream_t);      \
    template void launch_gemm_seg<T>(T*, const GemmTask*, const SegTask*, const int*, int, const FixTask*, int, T*,  \
                                     const int*, hipStream_t, int);
MFD_INSTANTIATE(double)
MFD_INSTANTIATE(float)

}  // namespace mfd
