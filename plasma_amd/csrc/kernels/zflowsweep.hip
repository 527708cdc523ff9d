// zflowsweep.hip -- a triangular sweep of the complex potrs / posv in one
// launch: L Y = B (forward) or L^H X = Y (backward).
//
// The scheme, its tickets, flags and visibility are those of the real sweep
// (flowsweep.hip): a workgroup per block row and group of right-hand sides
// subtracts L(m, k) Y_k as the Y_k are published, multiplies by W_mm and
// publishes Y_m.
//
// A group is 8 right-hand sides, one MFMA block of 16 real columns [Re | Im].
// In LDS stand Y1 = [Yr | Yi] and Y2 = [-Yi | Yr], so that Xr Y1 + Xi Y2 is
// the complex product X Y (Xr Y1 - Xi Y2 that of conj X): two real products
// per tile where 16 right-hand sides would take four, half the serial time.
// A tile row is 128 registers per lane in FP64; the operand is loaded in two
// halves of K, each of them again as soon as it has been used.
//
// Measured, zposv n = 5001 and nrhs 32: both sweeps 1.1 ms, per-step form
// (zchol.hip, two dependent launches of about 40 us per tile and sweep) 6.4
// ms.  Whole solves, per-step form and this one: n = 300, nrhs 3 843, 596 us;
// n = 2000, nrhs 128 5.60, 3.49 ms; n = 10000, nrhs 128 60.6, 49.7 ms; cposv
// n = 4000, nrhs 32 8.99, 5.97 ms.  It is used up to ZFLOW_SWEEP_NRHS = 128
// right-hand sides, which is not where it stops winning, although it reads L once
// per 8 of them: potrs n = 2000 with 256 and 768 right-hand sides 2.89, 0.86 and
// 3.04, 1.48 ms; n = 5000 7.46, 2.84 and 9.88, 6.85 ms.
#include "common.hip.h"
#include "directgemm.hip.h"
#include "plasma_kernels.h"
#include "zview.hip.h"

namespace {

constexpr int ZF_NT = 512;
constexpr int ZF_NB = 128;              // largest tile
constexpr int ZF_NC = 8;                // right-hand sides per workgroup
constexpr int ZF_LD = 2 * ZF_NC + 1;    // LDS row stride
constexpr int ZF_Y2 = ZF_NB * ZF_LD;    // Y2 after Y1
constexpr int ZF_CH = ZF_NB / 8;        // 4-deep MFMA steps per half

// 16 rows x 64 k values of an operand: lane l holds (l % 16, 4 i + l / 16)
template <typename R> struct ZFrag {
    R re[ZF_CH], im[ZF_CH];
};

// Half h of the rows row0.. of X (UNIT: contiguous rows, else contiguous k;
// the other stride is ld), K values in all.  A last, partial group of 4 is
// read from K - 4 on, so it repeats values whose counterparts in LDS are zero
// (zk_pos); groups past K repeat it and are not used.  Only K < 4 takes
// checked loads.
template <typename R, bool UNIT>
__device__ __forceinline__ void load_half(ZFrag<R> &f, const cx<R> *p0,
                                          int ld, int row0, int rows, int K,
                                          int h)
{
    typedef R pair_t __attribute__((ext_vector_type(2)));
    const int lane = threadIdx.x & 63, lk = lane / 16;
    const int r = min(row0 + lane % 16, rows - 1);
    if (8 * ZF_CH * h >= 2 * K) return;
    const DG_GLOBAL cx<R> *p = (const DG_GLOBAL cx<R> *)dg::uni(p0);
    ld = dg::uni(ld);
    if (K < 4) {
        const cx<R> z = lk < K ? p0[UNIT ? r + lk * ld : r * ld + lk]
                               : czero<R>();
        f.re[0] = z.re;
        f.im[0] = z.im;
        return;
    }
    const unsigned off =
        (UNIT ? r + lk * ld : r * ld + lk) * (unsigned)sizeof(cx<R>);
#pragma unroll
    for (int i = 0; i < ZF_CH; i++) {
        const int kc = min(4 * (ZF_CH * h + i), K - 4);
        const DG_GLOBAL cx<R> *q = dg::scalar(p + (UNIT ? kc * ld : kc));
        const pair_t z = *(const DG_GLOBAL pair_t *)((const DG_GLOBAL char *)q
                                                     + off);
        f.re[i] = z[0];
        f.im[i] = z[1];
    }
}

// LDS row of k value r of K (r >= K: a row that must hold zeros, if any)
__device__ __forceinline__ int zk_pos(int r, int K)
{
    const int full = K & ~3, end = full + 4;
    if (K < 4 || K == full || r < full || r >= end) return r;
    return r < K ? r + end - K : r + full - K;
}

// s + Xr Y1 + Xi Y2 over the groups [lo, hi) of half h of X.  As in the real
// sweep the product of a whole tile is summed on its own before it meets the
// block row; it is one sum in the order of k (two or four interleaved ones
// are no faster and cost accuracy: n = 5001, error of X 9.0e-16 instead of
// 7.9e-16).
template <typename R>
__device__ __forceinline__ typename Mfma<R>::acc_t mul_half(
    typename Mfma<R>::acc_t s, const ZFrag<R> &f, const R *y, int h, int lo,
    int hi)
{
    const int lane = threadIdx.x & 63;
    const R *p = y + (4 * ZF_CH * h + lane / 16) * ZF_LD + lane % 16;
    lo -= ZF_CH * h;
    hi -= ZF_CH * h;
    if (lo >= ZF_CH || hi <= 0) return s;
#pragma unroll
    for (int i = 0; i < ZF_CH; i++)
        if (i >= lo && i < hi) {
            s = Mfma<R>::mma(f.re[i], p[4 * i * ZF_LD], s);
            s = Mfma<R>::mma(f.im[i], p[4 * i * ZF_LD + ZF_Y2], s);
        }
    return s;
}

// BACK: L^H X = Y.  UPPER: the factor is stored as U = L^H.  sync: a ticket
// per launch and mt flags per group of right-hand sides, zero on entry.
template <typename R, bool BACK, bool UPPER>
__global__ __launch_bounds__(ZF_NT) void zflow_sweep_kernel(
    plasma_desc_t A, plasma_desc_t B, const cx<R> *inv, int gpt, int *sync,
    const int *status)
{
    // L operand: contiguous rows, not conjugated; else contiguous k, conj
    constexpr bool UL = BACK == UPPER;
    typedef typename Mfma<R>::acc_t acc_t;
    __shared__ R sy[2 * ZF_Y2];
    __shared__ int s_ticket;
    if (threadIdx.x == 0) s_ticket = atomicAdd(sync, 1);
    const bool stop = block_should_stop(status);    // and the ticket's barrier
    const int ticket = dg::uni(s_ticket);
    const int ngrp = B.nt * gpt;
    const int t = ticket / ngrp, g = ticket % ngrp;
    const int mt = B.mt;
    if (t >= mt) return;
    const int tn = g / gpt, c0 = (g % gpt) * ZF_NC;
    const int nv = plasma_tile_nview(B, tn) - c0;
    if (nv <= 0) return;                    // an empty group: nobody waits
    int *flags = sync + 1 + (size_t)g * mt;
    if (stop) {                             // as in the real sweep
        if (threadIdx.x == 0) agent_store(&flags[t], 1);
        return;
    }
    const int m = BACK ? mt - 1 - t : t;
    const int mv = plasma_tile_mview(B, m);
    const int lane = threadIdx.x & 63;
    const int wave = dg::uni(threadIdx.x >> 6);
    const int row0 = 16 * wave;
    const bool active = row0 < mv;
    const int col = lane & 7, part = (lane >> 3) & 1;

    // half h of the operand tile of step s: L(m, s) forward,
    // L(mt - 1 - s, m)^H backward; the last one (s == t) is W_mm or W_mm^H
    auto load = [&](ZFrag<R> &f, int s, int h) {
        if (!active) return;
        const int k = BACK ? mt - 1 - s : s;
        if (s == t) {
            load_half<R, !BACK>(f, inv + (size_t)m * A.mb * A.mb, A.mb, row0,
                                mv, mv, h);
        }
        else {
            const CView<R> L = BACK ? lower_cview<R>(A, UPPER, k, m)
                                    : lower_cview<R>(A, UPPER, m, k);
            load_half<R, UL>(f, L.p, UPPER ? L.rs : L.cs, row0, mv,
                             plasma_tile_mview(B, k), h);
        }
    };
    // -Y_k into sy (Y2 negated where X is conjugated); rows and right-hand
    // sides past the end are zero
    auto fetch = [&](int s) {
        const int k = BACK ? mt - 1 - s : s;
        const CView<R> Y = tile_cview<R>(B, k, tn);
        const int kv = plasma_tile_mview(B, k);
        constexpr int IT = ZF_NB * ZF_NC / ZF_NT;
        R re[IT], im[IT];
#pragma unroll
        for (int u = 0; u < IT; u++) {
            const int r = threadIdx.x % ZF_NB;
            const int c = threadIdx.x / ZF_NB + u * (ZF_NT / ZF_NB);
            re[u] = im[u] = R(0);
            if (r < kv && c < nv) {
                const cx<R> *p = Y.p + r + (ptrdiff_t)(c0 + c) * Y.cs;
                re[u] = agent_load(&p->re);
                im[u] = agent_load(&p->im);
            }
        }
#pragma unroll
        for (int u = 0; u < IT; u++) {
            const int r = threadIdx.x % ZF_NB;
            const int c = threadIdx.x / ZF_NB + u * (ZF_NT / ZF_NB);
            R *y = sy + zk_pos(r, kv) * ZF_LD + c;
            y[0] = -re[u];
            y[ZF_NC] = -im[u];
            y[ZF_Y2] = UL ? im[u] : -im[u];
            y[ZF_Y2 + ZF_NC] = UL ? -re[u] : re[u];
        }
    };

    // the block row itself: lanes 0 .. 7 of 16 the real parts of the 8
    // right-hand sides, lanes 8 .. 15 the imaginary parts
    const CView<R> Bm = tile_cview<R>(B, m, tn);
    auto bref = [&](int r) {
        return reinterpret_cast<R *>(Bm.p + r +
                                     (ptrdiff_t)(c0 + col) * Bm.cs) + part;
    };
    acc_t acc;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int r = row0 + Mfma<R>::row(lane, q);
        acc[q] = R(0);
        if (r < mv && col < nv) acc[q] = *bref(r);
    }
    ZFrag<R> f0, f1;
    load(f0, 0, 0);
    load(f1, 0, 1);
    for (int s = 0; s < t; s++) {
        if (threadIdx.x == 0)
            while (agent_load(&flags[s]) == 0) __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
        __syncthreads();
        fetch(s);
        __syncthreads();
        const int kv = plasma_tile_mview(B, BACK ? mt - 1 - s : s);
        const int hi = (kv + 3) / 4;
        acc_t p = {0, 0, 0, 0};
        if (active) p = mul_half<R>(p, f0, sy, 0, 0, hi);
        load(f0, s + 1, 0);
        if (active) p = mul_half<R>(p, f1, sy, 1, 0, hi);
        load(f1, s + 1, 1);
#pragma unroll
        for (int q = 0; q < 4; q++) acc[q] += p[q];
    }
    // Y_m = W_mm (or W_mm^H) times the block row, through LDS
    __syncthreads();
    if (active)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = row0 + Mfma<R>::row(lane, q);
            const R x = r < mv ? acc[q] : R(0);
            R *y = sy + zk_pos(r, mv) * ZF_LD;
            y[lane % 16] = x;
            // W forward, W^H backward
            y[ZF_Y2 + (lane % 16 ^ ZF_NC)] = (part != 0) == BACK ? x : -x;
        }
    __syncthreads();
    if (active) {
        // W is lower triangular: k <= row forward, k >= row backward
        const int all = (mv + 3) / 4;
        const int lo = BACK ? row0 / 4 : 0;
        const int hi = BACK ? all : min(row0 / 4 + 4, all);
        acc_t p = {0, 0, 0, 0};
        p = mul_half<R>(p, f0, sy, 0, lo, hi);
        p = mul_half<R>(p, f1, sy, 1, lo, hi);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = row0 + Mfma<R>::row(lane, q);
            if (r < mv && col < nv) agent_store(bref(r), p[q]);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) agent_store(&flags[t], 1);
}

template <typename R>
int launch_zflow(plasma_enum_t uplo, int backward, plasma_desc_t A,
                 plasma_desc_t B, const void *inv, int *sync,
                 const int *status, hipStream_t s)
{
    const int gpt = (B.nb + ZF_NC - 1) / ZF_NC;
    const dim3 grid((unsigned)B.mt * B.nt * gpt), block(ZF_NT);
    const bool up = uplo == PlasmaUpper;
    const void *fn = backward
        ? (up ? (const void *)zflow_sweep_kernel<R, true, true>
              : (const void *)zflow_sweep_kernel<R, true, false>)
        : (up ? (const void *)zflow_sweep_kernel<R, false, true>
              : (const void *)zflow_sweep_kernel<R, false, false>);
    int gp = gpt;
    const cx<R> *w = (const cx<R> *)inv;
    void *args[] = {&A, &B, &w, &gp, &sync, &status};
    return hipLaunchKernel(fn, grid, block, args, 0, s) == hipSuccess
               ? 0 : PlasmaErrorInternal;
}

}  // namespace

extern "C" int plasma_zflow_sweep_ok(plasma_desc_t A, int nrhs)
{
    return (A.precision == PlasmaComplexDouble ||
            A.precision == PlasmaComplexFloat) &&
           A.mb == A.nb && A.mb <= ZF_NB && nrhs <= ZFLOW_SWEEP_NRHS;
}

extern "C" size_t plasma_zflow_sweep_ints(plasma_desc_t B)
{
    return 1 + (size_t)B.mt * B.nt * ((B.nb + ZF_NC - 1) / ZF_NC);
}

extern "C" int plasma_kern_zflow_sweep(plasma_enum_t uplo, int backward,
                                       plasma_desc_t A, plasma_desc_t B,
                                       const void *inv, int *sync,
                                       const int *status, hipStream_t s)
{
    if (B.mb != A.mb || !plasma_zflow_sweep_ok(A, B.n))
        return PlasmaErrorNotSupported;
    if (B.mt <= 0 || B.nt <= 0) return 0;
    if (A.precision == PlasmaComplexDouble)
        return launch_zflow<double>(uplo, backward, A, B, inv, sync, status,
                                    s);
    return launch_zflow<float>(uplo, backward, A, B, inv, sync, status, s);
}
