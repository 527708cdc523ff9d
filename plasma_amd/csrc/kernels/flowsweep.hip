// flowsweep.hip -- a triangular sweep of potrs / posv in one launch.
//
// L Y = B (forward) or L^T X = Y (backward), the reference's pztrsm sweeps
// (compute/pztrsm.c:113-177), with the diagonal-tile inverses W_kk.  The
// per-step form (solve.hip) takes two dependent launches per tile, about 22
// us for 2 us of work.  Here every block row is one workgroup per 16
// right-hand sides: it subtracts L(m, k) Y_k for k = 0 .. m - 1 as the Y_k
// are published, multiplies by W_mm and publishes Y_m.  What remains serial
// per tile is: see the flag, fetch Y_k, one 128 x 128 x 16 product, the
// product with W_mm, store Y_m, set the flag.  The next tile of L (or W_mm)
// is already in registers by then.
//
// Progress: block rows are handed out by a ticket in the order of their
// dependences, so a workgroup only ever waits for workgroups that started
// before it; the first waits for nobody.  A workgroup that finds the status
// word set publishes its block row unsolved: others may have started before the
// word was set and wait for it (what they go on to compute is not used).
//
// Visibility between workgroups (on different XCDs, with an L2 each): Y is
// stored and read by relaxed agent-scope atomics, which go through to memory
// and past the caches; a workgroup's stores are complete (vmcnt 0 in every
// wave, then a barrier) before one thread sets its flag, and its readers
// issue their loads after they have seen the flag.  No cache is flushed or
// invalidated, so the tiles of L stay cached.
//
// Measured (both sweeps of dposv n = 8192, nrhs 64): 1.25 ms, per-step form
// 2.9 ms; per tile and sweep about 4.5 us in FP32 and 8.7 us in FP64.  Whole
// solves, per-step form and this one: dposv n = 300 346, 277 us; n = 2000 and
// nrhs 128 1721, 1266 us; n = 16384 and nrhs 128 42.0, 38.7 ms; sposv n =
// 8192 6.73, 4.99 ms.  It is used up to FLOW_SWEEP_NRHS = 128 right-hand sides,
// which is not where it stops winning, although it reads L once per 16 of them:
// potrs n = 2000 with 256 and 768 right-hand sides 826, 368 and 954, 577 us; n =
// 8192 3.89, 2.51 and 6.18, 6.00 ms; in FP32 n = 8192 2.97, 1.35 and 4.10, 3.03
// ms.
//
// Eight waves; wave w holds rows 16 w .. of the block row (tiles of order
// <= 128).  The operand that MFMA needs row by row (L or W) goes straight
// from memory to registers (dg::Operand); Y_k (128 x 16) through LDS.
#include "common.hip.h"
#include "directgemm.hip.h"
#include "plasma_kernels.h"

namespace {

constexpr int FS_NT = 512;
constexpr int FS_NB = 128;              // largest tile
constexpr int FS_NC = 16;               // right-hand sides per workgroup
constexpr int FS_LD = FS_NC + 1;        // LDS row stride

// 16 rows x 128 k values of an MFMA operand in registers
template <typename T> struct Frag {
    static constexpr int N = FS_NB / dg::Chunk<T>::KC;
    dg::Regs<T, 1> c[N];
};

// All chunks of K k values.  A last, partial chunk is read KC values before
// the end, so it repeats values of the chunk before it, whose counterparts in
// LDS are zero (k_pos); chunks past K repeat it and are not used.  Only a K
// below one chunk takes checked loads.
template <typename T, bool UNIT>
__device__ __forceinline__ void load_frag(Frag<T> &f, const View<T> &A,
                                          int row0, int rows, int K)
{
    constexpr int KC = dg::Chunk<T>::KC;
    dg::Operand<T, 1, UNIT> o;
    o.init(A, row0, rows);
    if (K >= KC) {
#pragma unroll
        for (int i = 0; i < Frag<T>::N; i++)
            o.load(f.c[i], min(i * KC, K - KC));
    }
    else {
        o.load_tail(f.c[0], 0, K);
    }
}

// LDS row of k value r of K (r >= K: a row that must hold zeros, if any)
template <typename T> __device__ __forceinline__ int k_pos(int r, int K)
{
    constexpr int KC = dg::Chunk<T>::KC;
    const int full = K / KC * KC, end = full + KC;
    if (K < KC || K == full || r < full || r >= end) return r;
    return r < K ? r + end - K : r + full - K;
}

// acc + A (16 x K, in f) Y (K x 16, in LDS) over the chunks [lo, hi).  The
// product is summed on its own (in two chains) before it meets acc: adding
// every term to a block row of n terms would round n / 4 times at its size
// (sposv n = 6000: error 2.4e-6 instead of 1.4e-6).
template <typename T>
__device__ __forceinline__ typename Mfma<T>::acc_t mul_frag(
    typename Mfma<T>::acc_t acc, const Frag<T> &f, const T *y, int lo, int hi)
{
    constexpr int V = dg::Chunk<T>::V, KC = dg::Chunk<T>::KC;
    const int lane = threadIdx.x & 63;
    const T *p = y + V * (lane / 16) * FS_LD + lane % 16;
    typename Mfma<T>::acc_t s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < Frag<T>::N; i++)
        if (i >= lo && i < hi)
#pragma unroll
            for (int v = 0; v < V; v++) {
                const T x = f.c[i].v[0][v], b = p[(i * KC + v) * FS_LD];
                if (v & 1) s1 = Mfma<T>::mma(x, b, s1);
                else       s0 = Mfma<T>::mma(x, b, s0);
            }
#pragma unroll
    for (int q = 0; q < 4; q++) acc[q] += s0[q] + s1[q];
    return acc;
}

// BACK: L^T X = Y.  UPPER: the factor is stored as U = L^T.  sync: a ticket
// per launch and mt flags per group of right-hand sides, zero on entry.
template <typename T, bool BACK, bool UPPER>
__global__ __launch_bounds__(FS_NT) void flow_sweep_kernel(
    plasma_desc_t A, plasma_desc_t B, const T *inv, int gpt, int *sync,
    const int *status)
{
    constexpr bool UL = BACK == UPPER;      // L operand: contiguous rows
    constexpr int KC = dg::Chunk<T>::KC;
    typedef typename Mfma<T>::acc_t acc_t;
    __shared__ T sy[2][FS_NB * FS_LD];
    __shared__ int s_ticket;
    if (threadIdx.x == 0) s_ticket = atomicAdd(sync, 1);
    const bool stop = block_should_stop(status);    // and the ticket's barrier
    const int ticket = dg::uni(s_ticket);
    const int ngrp = B.nt * gpt;
    const int t = ticket / ngrp, g = ticket % ngrp;
    const int mt = B.mt;
    if (t >= mt) return;
    const int tn = g / gpt, c0 = (g % gpt) * FS_NC;
    const int nv = plasma_tile_nview(B, tn) - c0;
    if (nv <= 0) return;                    // an empty group: nobody waits
    int *flags = sync + 1 + (size_t)g * mt;
    if (stop) {
        if (threadIdx.x == 0) agent_store(&flags[t], 1);
        return;
    }
    const int m = BACK ? mt - 1 - t : t;
    const int mv = plasma_tile_mview(B, m);
    const int lane = threadIdx.x & 63;
    const int wave = dg::uni(threadIdx.x >> 6);
    const int row0 = 16 * wave;
    const bool active = row0 < mv;

    // operand tile of step s: L(m, s) forward, L(mt - 1 - s, m)^T backward;
    // the last one (s == t) is W_mm or W_mm^T
    auto load = [&](Frag<T> &f, int s) {
        if (!active) return;
        const int k = BACK ? mt - 1 - s : s;
        if (s == t) {
            View<T> W;
            W.p = const_cast<T *>(inv) + (size_t)m * A.mb * A.mb;
            W.rs = BACK ? A.mb : 1;
            W.cs = BACK ? 1 : A.mb;
            load_frag<T, !BACK>(f, W, row0, mv, mv);
        }
        else {
            const View<T> L = BACK ? lower_view<T>(A, UPPER, k, m)
                                   : lower_view<T>(A, UPPER, m, k);
            View<T> X = L;
            if (BACK) {
                X.rs = L.cs;
                X.cs = L.rs;
            }
            load_frag<T, UL>(f, X, row0, mv, plasma_tile_mview(B, k));
        }
    };
    // -Y_k into sy[buf]; rows and right-hand sides past the end are zero
    auto fetch = [&](int s, int buf) {
        const int k = BACK ? mt - 1 - s : s;
        const View<T> Y = tile_view<T>(B, k, tn);
        const int kv = plasma_tile_mview(B, k);
        constexpr int IT = FS_NB * FS_NC / FS_NT;
        T x[IT];
#pragma unroll
        for (int u = 0; u < IT; u++) {
            const int r = threadIdx.x % FS_NB;
            const int c = threadIdx.x / FS_NB + u * (FS_NT / FS_NB);
            x[u] = T(0);
            if (r < kv && c < nv) x[u] = agent_load(&Y.at(r, c0 + c));
        }
#pragma unroll
        for (int u = 0; u < IT; u++) {
            const int r = threadIdx.x % FS_NB;
            const int c = threadIdx.x / FS_NB + u * (FS_NT / FS_NB);
            sy[buf][k_pos<T>(r, kv) * FS_LD + c] = -x[u];
        }
    };

    // the block row itself
    const View<T> Bm = tile_view<T>(B, m, tn);
    acc_t acc;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int r = row0 + Mfma<T>::row(lane, q), c = lane % 16;
        acc[q] = T(0);
        if (r < mv && c < nv) acc[q] = Bm.at(r, c0 + c);
    }
    Frag<T> f0, f1;
    load(f0, 0);
    // step s with the operand in fa, the next one loading into fb
    auto step = [&](int s, const Frag<T> &fa, Frag<T> &fb) {
        load(fb, s + 1);
        if (threadIdx.x == 0)
            while (agent_load(&flags[s]) == 0) __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
        __syncthreads();
        fetch(s, s & 1);
        __syncthreads();
        const int kv = plasma_tile_mview(B, BACK ? mt - 1 - s : s);
        if (active)
            acc = mul_frag<T>(acc, fa, sy[s & 1], 0, (kv + KC - 1) / KC);
    };
    // Y_m = W_mm (or W_mm^T) times the block row, through LDS
    auto finish = [&](const Frag<T> &w) {
        T *st = sy[t & 1];
        if (active)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = row0 + Mfma<T>::row(lane, q);
                st[k_pos<T>(r, mv) * FS_LD + lane % 16] =
                    r < mv ? acc[q] : T(0);
            }
        __syncthreads();
        if (!active) return;
        // W is lower triangular: k <= row forward, k >= row backward
        const int hi = (mv + KC - 1) / KC;
        acc = mul_frag<T>(acc_t{0, 0, 0, 0}, w, st, BACK ? row0 / KC : 0,
                          BACK ? hi : min((row0 + 16 + KC - 1) / KC, hi));
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = row0 + Mfma<T>::row(lane, q), c = lane % 16;
            if (r < mv && c < nv) agent_store(&Bm.at(r, c0 + c), acc[q]);
        }
    };
    int s = 0;
    for (; s + 2 <= t; s += 2) {
        step(s, f0, f1);
        step(s + 1, f1, f0);
    }
    if (s < t) {
        step(s, f0, f1);
        finish(f1);
    }
    else {
        finish(f0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) agent_store(&flags[t], 1);
}

template <typename T>
int launch_flow(plasma_enum_t uplo, int backward, plasma_desc_t A,
                plasma_desc_t B, const void *inv, int *sync,
                const int *status, hipStream_t s)
{
    const int gpt = (B.nb + FS_NC - 1) / FS_NC;
    const dim3 grid((unsigned)B.mt * B.nt * gpt), block(FS_NT);
    const bool up = uplo == PlasmaUpper;
    const void *fn = backward
        ? (up ? (const void *)flow_sweep_kernel<T, true, true>
              : (const void *)flow_sweep_kernel<T, true, false>)
        : (up ? (const void *)flow_sweep_kernel<T, false, true>
              : (const void *)flow_sweep_kernel<T, false, false>);
    int gp = gpt;
    const T *w = (const T *)inv;
    void *args[] = {&A, &B, &w, &gp, &sync, &status};
    return hipLaunchKernel(fn, grid, block, args, 0, s) == hipSuccess
               ? 0 : PlasmaErrorInternal;
}

}  // namespace

extern "C" int plasma_flow_sweep_ok(plasma_desc_t A, int nrhs)
{
    return (A.precision == PlasmaRealDouble ||
            A.precision == PlasmaRealFloat) &&
           A.mb == A.nb && A.mb <= FS_NB && nrhs <= FLOW_SWEEP_NRHS;
}

extern "C" size_t plasma_flow_sweep_ints(plasma_desc_t B)
{
    return 1 + (size_t)B.mt * B.nt * ((B.nb + FS_NC - 1) / FS_NC);
}

extern "C" int plasma_kern_flow_sweep(plasma_enum_t uplo, int backward,
                                      plasma_desc_t A, plasma_desc_t B,
                                      const void *inv, int *sync,
                                      const int *status, hipStream_t s)
{
    if (B.mb != A.mb || !plasma_flow_sweep_ok(A, B.n))
        return PlasmaErrorNotSupported;
    if (B.mt <= 0 || B.nt <= 0) return 0;
    if (A.precision == PlasmaRealDouble)
        return launch_flow<double>(uplo, backward, A, B, inv, sync, status, s);
    return launch_flow<float>(uplo, backward, A, B, inv, sync, status, s);
}
