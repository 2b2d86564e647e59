// The fronts at the bottom of the elimination tree, written for gfx950
// (CDNA4, wave64): every front of order <= 128 whose children are such fronts
// too, assembled and factored in one dependency-driven launch.
//
// Replaces, for those fronts (paths relative to the reference root,
// src/main/): set_zero + set_coefficient (zero_setter_m.f90:12-31,
// coefficient_setter_m.f90:15-50), the extend-add (extend_add_kernel_m.f90:
// 6-34) and the tile loop of a front (seq_factorize_m.f90:31-79).
//
// A front of this size is some ten microseconds of dependent arithmetic (the
// pivot chain) on a few tens of kilobytes, so what bounds a tree of them is
// how many are in flight at a time and how often their entries pass through
// memory.  Level by level a front took a zeroing, a scatter, one extend-add
// per child rank, a diagonal, a panel and an update launch, two to four
// workgroups per CU.  Here a workgroup takes a front from start to end: its
// lower triangle lives in registers as 16 x 16 MFMA accumulators (36 tiles
// over four waves), the children's update matrices are added as they are
// read, A's entries go in with their panel, and L, the update matrix and the
// diagonal-block inverses are written once; only a 16-column panel is in LDS,
// which leaves room for three workgroups per CU.  Fronts are handed out by
// tickets in the order of their height and wait for their children by a
// counter (as in mfd_solve.hip, whose argument why no wait lasts for ever
// holds here as it stands).
#include <hip/hip_runtime.h>

#include "mfd_device.h"
#include "mfd_kernels.h"

namespace mfd {

namespace {

constexpr int kNT = kTreeFront / 16;              // 16 x 16 tiles along a front
constexpr int kOwn = (kNT * (kNT + 1) / 2 + 3) / 4;  // lower tiles of one wave
// P[col][row]; 16 modulo 32, so that the four columns of an operand read use
// different halves of the banks
constexpr int kPitch = kTreeFront + 16;

template <typename T> struct TreeLds {
    T P[16][kPitch];   // the panel in work
    T X[6][16][17];    // rows 0 .. 2 of the 64-block's inverse, tile (i, j) at i (i + 1) / 2 + j, [col][row]
    T Xl[16][17];      // its last diagonal tile
    T D[16][17];       // the previous panel's diagonal tile of L, [col][row]
    T Ts[3][16][17];   // staging of the inverse's products
    T rs[16], rsd[16];  // 1 / L_kk of the panel, and of the previous one
    short map[kTreeFront];  // front row -> update row of the child being added, -1
    int ticket;
};

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The workgroup's LDS as the out-of-line functions take it.  Out of line, the
// chain and the inverse keep their registers to themselves: inlined, they
// were added to the 72 of the tiles and spilled.
template <typename T> using Lds = __attribute__((address_space(3))) TreeLds<T>*;

// Columns b16 .. b16 + cb - 1 of the panel in P: lanes 0 .. 15 of each wave
// hold the diagonal block's rows, its other lanes 48 of the rows below, so
// each of up to three waves (w) runs the same chain on its own, with panel16's
// arithmetic and order of updates (see there).  (One wave for the chain and
// another for the rows past its 64 afterwards took longer: 20 more us for a
// front of order 110.)  One copy of the code serves whole and partial panels:
// short fronts are bound by instruction fetch as much as by the chain.  Holds
// one barrier, between the reads of the panel and the first write to it.
template <typename T>
__device__ __attribute__((noinline)) void tree_panel(Lds<T> Sp, int w, int b16, int cb, int n, int* info, int col0)
{
    // (arguments of a call come in vector registers)
    w = uniform(w), b16 = uniform(b16), cb = uniform(cb), n = uniform(n), col0 = uniform(col0);
    const int r = threadIdx.x & 63, row = r < 16 ? b16 + r : b16 + r + 48 * w, at = min(row, n - 1);
    const bool live = row < n;
    T x[16], v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const T p = Sp->P[j][at];
        x[j] = (live && (r >= 16 || j <= r)) ? p : T(0);
        v[j] = T(0);
    }
    __syncthreads();  // every wave has its copy of the diagonal block's rows
    T lp = T(0), piv = T(1);
    const int to = live ? row : kTreeFront;  // (past the last row: not used)
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (k < cb) {
            const T d = bcast(x[k], k), rs = rsqrt_nr(d), sd = sqrt_from_rs(d, rs), q = quot(x[k], sd, rs);
            if (k + 1 < 16) {
                const T u = quot(bcast(x[k], k + 1), sd, rs);
                x[k + 1] -= lp * v[k + 1];
                if (k + 1 < cb) x[k + 1] -= q * u;
                pin(x[k + 1]);
            }
            piv = r == k ? d : piv;
            pin(piv);
            const T l = r == k ? sd : q;
            x[k] = l;
            Sp->P[k][to] = l;
            Sp->rs[k] = rs;
#pragma unroll
            for (int j = k + 2; j < 16; ++j) {
                x[j] -= lp * v[j];
                pin(x[j]);
            }
            lp = l;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = k + 2; j < 16; ++j) v[j] = Sp->P[k][b16 + j];
            if (k + 1 == cb && k + 1 < 16) v[k + 1] = Sp->P[k][b16 + k + 1];
        }
    }
    if (cb < 16) {
        if (w == 0 && r == 0)
            for (int k = cb; k < 16; ++k) Sp->rs[k] = T(1);  // finite stand-ins for the inverse
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (j >= cb) {
                x[j] -= lp * v[j];
                if (live) Sp->P[j][row] = x[j];
            }
    }
    const unsigned long long bad = __ballot(!(piv > T(0)));
    if (w == 0 && bad && r == 0) atomicMin(info, col0 + b16 + __ffsll(bad));
}

// Row p of the inverse of panel p's 64-column block, by one wave: the 16 x 16
// inverse of the diagonal tile in D (as diaginv16, entries read a column
// ahead), X_ij = -inv(L_ii) sum_{j<=k<i} L_ik X_kj (as
// inverse16, L_ik read back from the front; the tiles j side by side), all
// stored at inv (inv[r + 64 q] = L^{-1}(q, r), zero elsewhere); last: the
// block's rows after p are zero.
template <typename T>
__device__ __attribute__((noinline)) void tree_inverse(Lds<T> Sp, const T* F, int n, T* inv, int p, int cb, int last)
{
    typedef typename Mfma<T>::acc_t acc_t;
    n = uniform(n), p = uniform(p), cb = uniform(cb), last = uniform(last);
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4, i = p & 3, blk = p >> 2;
    T* out = inv + (int64_t)blk * 4096;
    T lik[3][4];
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (k < i) {
#pragma unroll
            for (int q = 0; q < 4; ++q) lik[k][q] = F[min(16 * p + li, n - 1) + (int64_t)(64 * blk + 16 * k + 4 * q + g) * n];
        }
    // In 32 bits each entry of the next column of D is read as this column's
    // is used; in 64 bits that read-ahead costs the registers that hold the
    // caller's accumulators (22.8 us a front against 20.2 without it).
    constexpr bool kAhead = sizeof(T) == 4;
    T y[16], d[16], rk = Sp->rsd[0], rn = T(0);
#pragma unroll
    for (int j = 0; j < 16; ++j) y[j] = j == li ? T(1) : T(0);
    if constexpr (kAhead) {
#pragma unroll
        for (int j = 1; j < 16; ++j) d[j] = Sp->D[0][j];
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (!kAhead) __builtin_amdgcn_sched_barrier(0);
        if (k < 15) rn = Sp->rsd[k + 1];
        const T y0 = y[k] * rk;
        y[k] = y0;
#pragma unroll
        for (int j = k + 1; j < 16; ++j) {
            y[j] -= y0 * (kAhead ? d[j] : Sp->D[k][j]);
            pin(y[j]);
            if constexpr (kAhead) {
                if (j > k + 1) d[j] = Sp->D[k + 1][j];
                if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);
            }
        }
        rk = rn;
    }
    __builtin_amdgcn_sched_barrier(0);
    typedef __attribute__((address_space(3))) T (*Tile)[17];
    const Tile Xi = i < 3 ? Sp->X[i * (i + 1) / 2 + i] : Sp->Xl;
    if (lane < 16) {
#pragma unroll
        for (int k = 0; k < 16; ++k) Xi[li][k] = y[k];
    }
    acc_t acc[3] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (k < i) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int j = 0; j <= k; ++j)
                    acc[j] = Mfma<T>::mma(lik[k][q], Sp->X[k * (k + 1) / 2 + j][li][4 * q + g], acc[j]);
        }
#pragma unroll
    for (int j = 0; j < 3; ++j)
        if (j < i) {
#pragma unroll
            for (int v = 0; v < 4; ++v) Sp->Ts[j][Mfma<T>::row(lane, v)][li] = acc[j][v];
        }
    wave_sync();
    T xi[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) xi[q] = Xi[4 * q + g][li];
#pragma unroll
    for (int j = 0; j < 3; ++j) acc[j] = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (j < i) acc[j] = Mfma<T>::mma(xi[q], Sp->Ts[j][4 * q + g][li], acc[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        T xv[4] = {T(0), T(0), T(0), T(0)};
        if (j < 3 && j < i) {
#pragma unroll
            for (int v = 0; v < 4; ++v) xv[v] = -acc[j < 3 ? j : 0][v];
            if (i < 3) {
#pragma unroll
                for (int v = 0; v < 4; ++v) Sp->X[i * (i + 1) / 2 + j][li][Mfma<T>::row(lane, v)] = xv[v];
            }
        } else if (j == i) {
#pragma unroll
            for (int v = 0; v < 4; ++v) xv[v] = Xi[li][Mfma<T>::row(lane, v)];
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int q = Mfma<T>::row(lane, v);
            out[(16 * j + li) + 64 * (16 * i + q)] = (q < cb && (j < i || li < cb)) ? xv[v] : T(0);
        }
    }
    if (last)
        for (int q = 16 * (i + 1) + g; q < 64; q += 4)
#pragma unroll
            for (int j = 0; j < 4; ++j) out[(16 * j + li) + 64 * q] = T(0);
}

template <typename T> __device__ __forceinline__ void tree_front(const TreeArgs<T>& A, const TreeTask& t, TreeLds<T>& S, int tid0)
{
    typedef typename Mfma<T>::acc_t acc_t;
    int tid = tid0, lane = tid & 63, li = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the wave's role in a panel (0 .. 2 the chain, 3 the inverse), turned by one from each workgroup of a CU to the next so that
    // their chains need not share a SIMD
    const int rv = (wv + (blockIdx.x >> 3) + (blockIdx.x >> 8)) & 3;
    // lane offsets of the code that follows are computed there, not before
    auto fresh = [&]() {
        tid = tid0;
        pin(tid);
        lane = tid & 63;
        li = lane & 15;
        g = lane >> 4;
    };
    const int n = t.n, c = t.c, nt = (n + 15) >> 4, np = (c + 15) >> 4;
    T* F = A.pool + t.front;
    T* inv = A.pool + t.inv;
    // the wave's tiles: tile q = 4 s + wave of the lower triangle by rows,
    // row I and column J (I = 255 past the front)
    int ti[kOwn], tj[kOwn];
    acc_t acc[kOwn];
#pragma unroll
    for (int s = 0; s < kOwn; ++s) {
        const int q = 4 * s + wv;
        int I = 0;
#pragma unroll
        for (int k = 1; k <= kNT; ++k) I += q >= k * (k + 1) / 2;
        tj[s] = q - I * (I + 1) / 2;
        ti[s] = I < nt ? I : 255;
        acc[s] = acc_t{0, 0, 0, 0};
    }
    // A's entries of a panel, one per thread ahead of time (position row +
    // 256 col in the panel; the value, scaled in the 16-bit forms)
    auto entry = [&](int e, int& pos, T& val) {
        pos = A.apos[e];
        double a = A.a[A.asrc[e]];
        if (A.scale) {
            const int2 rc = A.arc[e];
            a = a * A.scale[rc.x] * A.scale[rc.y];
        }
        val = (T)a;
    };
    int e0 = ld_scalar(A.aptr + t.aptr), e1 = ld_scalar(A.aptr + t.aptr + 1), pos = 0;
    T val = T(0);
    if (e0 + tid < e1) entry(e0 + tid, pos, val);

    // the children's update matrices, child by child (extend-add)
    for (int k = 0; k < t.nchild; ++k) {
        const TreeChild ch = ld_scalar(A.children + t.child + k);
        const int at = tid < ch.w ? A.lidx[ch.lidx + tid] - 1 : -1;
        __syncthreads();  // the previous child's map has been read
        if (tid < kTreeFront) S.map[tid] = -1;
        __syncthreads();
        if (at >= 0) S.map[at] = (short)tid;
        if (k == 0 && tid == 0) poll(A.flags + kSolveCtl + t.flag, t.nchild, A.flags + kSolveStop, A.err);
        __syncthreads();
        const T* U = A.pool + ch.u;
        fresh();
#pragma unroll
        for (int s0 = 0; s0 < kOwn; s0 += 3) {
            T u[3][4];
#pragma unroll
            for (int s = s0; s < s0 + 3; ++s) {
                const int I = ti[s], J = tj[s];
#pragma unroll
                for (int v = 0; v < 4; ++v) u[s - s0][v] = T(0);
                if (I == 255) continue;
                const int jj = S.map[16 * J + li];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = Mfma<T>::row(lane, v), ii = S.map[16 * I + r];
                    if (jj >= 0 && ii >= 0 && (I > J || r >= li)) u[s - s0][v] = ld_off(U, (unsigned)(ii + jj * ch.ld));
                }
            }
#pragma unroll
            for (int s = s0; s < s0 + 3; ++s)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[s][v] += u[s - s0][v];
        }
    }

    for (int b = 0; b < np; ++b) {
        const int b16 = 16 * b, cb = min(16, c - b16);
        fresh();
        // the panel's tiles to P
#pragma unroll
        for (int s = 0; s < kOwn; ++s)
            if (tj[s] == b && ti[s] != 255) {
#pragma unroll
                for (int v = 0; v < 4; ++v) S.P[li][16 * ti[s] + Mfma<T>::row(lane, v)] = acc[s][v];
            }
        __syncthreads();
        // its entries of A
        if (e0 + tid < e1) S.P[pos >> 8][pos & 255] += val;
        for (int e = e0 + tid + kThreads; e < e1; e += kThreads) {
            int q;
            T a;
            entry(e, q, a);
            S.P[q >> 8][q & 255] += a;
        }
        if (b + 1 < np) {  // the next panel's
            e0 = e1;
            e1 = ld_scalar(A.aptr + t.aptr + b + 2);
            if (e0 + tid < e1) entry(e0 + tid, pos, val);
        }
        __syncthreads();
        if (rv == 0 || (rv < 3 && b16 + 16 + 48 * rv < n)) {
            tree_panel<T>((Lds<T>)&S, rv, b16, cb, n, A.info, t.first);  // (holds one barrier)
        } else {
            __syncthreads();
            if (rv == 3 && b > 0) tree_inverse<T>((Lds<T>)&S, F, n, inv, b - 1, 16, false);
        }
        __syncthreads();
        fresh();
        // (the next panel's entries have arrived: waited for here, before the
        // stores, so that no later wait for a load waits for those too)
        pin(val);
        pin(pos);
        // the panel's product off the tiles to the right (summed by itself:
        // accumulated onto the tile it would round at the tile's magnitude
        // four times instead of once), its diagonal tile
        // to D, and the panel to the front (past the pivots: update columns,
        // which the parent's workgroup reads) by the chain's waves: the
        // inverse's wave reads the front next
#pragma unroll
        for (int s = 0; s < kOwn; ++s)
            if (tj[s] > b && ti[s] != 255) {
                typename Mfma<T>::acc_t d = {0, 0, 0, 0};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int k = 4 * q + g;
                    const T x = S.P[k][16 * ti[s] + li], y = S.P[k][16 * tj[s] + li];
                    d = Mfma<T>::mma(k < cb ? x : T(0), k < cb ? y : T(0), d);
                }
                acc[s] -= d;
            }
        S.D[tid >> 4][tid & 15] = S.P[tid >> 4][b16 + (tid & 15)];
        if (tid < 16) S.rsd[tid] = S.rs[tid];
        if (rv < 3) {
#pragma unroll
            for (int k0 = 0; k0 < 6; k0 += 2) {
                T w[2][kTreeFront / 64];
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int h = 0; h < kTreeFront / 64; ++h) w[k][h] = S.P[min(rv + 3 * (k0 + k), 15)][64 * h + lane];
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int h = 0; h < kTreeFront / 64; ++h) {
                        const int row = 64 * h + lane, col = rv + 3 * (k0 + k);
                        if (col < 16 && row < n && b16 + col <= row) {
                            T* p = F + row + (int64_t)(b16 + col) * n;
                            if (col < cb)
                                *p = w[k][h];
                            else
                                st_agent(p, w[k][h]);
                        }
                    }
            }
        }
        __syncthreads();
    }
    fresh();
    // the update matrix, a tile at a time through a piece of P of the wave's own
    T* W = &S.P[0][0] + wv * 272;
#pragma unroll
    for (int s = 0; s < kOwn; ++s)
        if (tj[s] >= np && ti[s] != 255) {
            wave_sync();
#pragma unroll
            for (int v = 0; v < 4; ++v) W[li * 17 + Mfma<T>::row(lane, v)] = acc[s][v];
            wave_sync();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = 16 * ti[s] + li, col = 16 * tj[s] + 4 * q + g;
                if (row < n && col <= row) st_agent(F + row + (int64_t)col * n, W[(4 * q + g) * 17 + li]);
            }
        }
    if (t.sig >= 0) stores_done();
    __syncthreads();
    if (t.sig >= 0 && tid == 0) add_agent(A.flags + kSolveCtl + t.sig, 1);
    // the last row of the inverse beside the start of the workgroup's next
    // front (which uses none of its staging before its own panels)
    if (rv == 3) tree_inverse<T>((Lds<T>)&S, F, n, inv, np - 1, c - 16 * (np - 1), true);
}

}  // namespace

template <typename T> __global__ __launch_bounds__(kThreads, sizeof(T) == 8 ? 3 : 5) void k_tree(TreeArgs<T> A)
{
    __shared__ TreeLds<T> S;
    const int tid = threadIdx.x;
    int per = 1;
    for (;;) {
        if (tid == 0) S.ticket = add_agent(A.flags + kSolveTicket, per);
        __syncthreads();
        const int k0 = __builtin_amdgcn_readfirstlane(S.ticket), k1 = min(k0 + per, A.ntasks);
        if (k0 >= k1) return;
        for (int k = k0; k < k1; ++k) {
            const TreeTask t = ld_scalar(A.tasks + k);
            per = t.per;
            tree_front<T>(A, t, S, tid);
        }
    }
}

// As many workgroups as the chip holds (three, FP32 five, per CU).
template <typename T> void launch_tree(const TreeArgs<T>& A, hipStream_t st)
{
    if (A.ntasks > 0)
        hipLaunchKernelGGL(k_tree<T>, dim3((unsigned)std::min(A.ntasks, 256 * (sizeof(T) == 8 ? 3 : 5))), dim3(kThreads), 0, st, A);
}
template void launch_tree<double>(const TreeArgs<double>&, hipStream_t);
template void launch_tree<float>(const TreeArgs<float>&, hipStream_t);

}  // namespace mfd
