// directgemm.hip.h -- the low-latency MFMA block product of the critical
// chain (panel solve, next column's update, short trailing updates):
//     C(block) = [C] -/+ X Y^T
// one workgroup of 4 waves per 32 FW x 32 FW block (FW = 1, 2), each wave
// 16 FW x 16 FW of it.
//
// The blocked kernels with LDS staging (tilegemm.hip.h, update64.hip) need
// 14 us of matrix instructions for one 128 x 128 block with K = 128 in FP64;
// a launch of a few dozen such blocks leaves most CUs idle for that long.
// Smaller blocks spread the same work over the chip.  They read each operand
// more often, but the operands of these launches are small and come from L2,
// and an MFMA occupies its unit long enough (64 cycles in FP64, 32 in FP32)
// that they can go straight from memory to registers: no LDS, no barrier, a
// ring of RING chunks of 4 V k values in flight (V = 16 bytes / element).
//
// Within a chunk the k index of MFMA step v is kc + V (lane / 16) + v, the
// same for both operands, so an operand with contiguous k (upper storage)
// moves by 16-byte loads, one per chunk and row, and one with contiguous
// rows by 128-byte runs of 16 lanes.  Rows past the operand read its last
// row (their results are not stored); a K that is no multiple of the chunk
// ends with a chunk of checked loads.
#pragma once

#include "common.hip.h"
#include "tilegemm.hip.h"

namespace dg {

constexpr int NT = 256;
constexpr int RING = 4;

template <typename T> struct Chunk {
    static constexpr int V = 16 / (int)sizeof(T);
    static constexpr int KC = 4 * V;
};

// A value that is the same in every lane, in scalar registers (tile numbers
// come out of vector arithmetic), so that loads take a scalar base and a
// 32-bit lane offset.
__device__ __forceinline__ int uni(int x)
{
    return __builtin_amdgcn_readfirstlane(x);
}
#define DG_GLOBAL __attribute__((address_space(1)))
template <typename T> __device__ __forceinline__ DG_GLOBAL T *uni(T *p)
{
    const uint64_t v = (uint64_t)p;
    return (DG_GLOBAL T *)((uint64_t)(unsigned)uni((int)(v >> 32)) << 32 |
                           (unsigned)uni((int)v));
}
// The same pointer, opaque: the compiler would otherwise turn every
// (base + lane offset) of a loop into a 64-bit vector pointer of its own.
template <typename P> __device__ __forceinline__ P scalar(P p)
{
    const uint64_t v = (uint64_t)p;
    uint64_t u = (uint64_t)(unsigned)uni((int)(v >> 32)) << 32 |
                 (unsigned)uni((int)v);
    asm("" : "+s"(u));
    return (P)u;
}

// FW operand rows of a lane for one chunk
template <typename T, int FW> struct Regs {
    T v[FW][Chunk<T>::V];
};

// One operand as the wave reads it: rows row0 + 16 i + lane % 16.
template <typename T, int FW, bool UNIT> struct Operand {
    static constexpr int V = Chunk<T>::V;
    typedef T vec_t __attribute__((ext_vector_type(V)));
    const DG_GLOBAL T *p;
    unsigned off[FW];  // byte offset of the lane's first value
    int ld;            // stride of the other index
    bool vec;          // 16-byte loads allowed (contiguous k)

    __device__ __forceinline__ void init(const View<T> &A, int row0, int rows)
    {
        const int lane = threadIdx.x & 63;
        p = uni(A.p);
        ld = uni(UNIT ? A.cs : A.rs);
        vec = !UNIT && (uintptr_t)p % 16 == 0 && ld % V == 0;
#pragma unroll
        for (int i = 0; i < FW; i++) {
            const int r = min(row0 + 16 * i + lane % 16, rows - 1);
            off[i] = (UNIT ? r + V * (lane / 16) * ld
                           : r * ld + V * (lane / 16)) * (int)sizeof(T);
        }
    }
    template <typename U>
    static __device__ __forceinline__ U at(const DG_GLOBAL T *q, unsigned o)
    {
        return *(const DG_GLOBAL U *)((const DG_GLOBAL char *)q + o);
    }
    // the chunk at k = kc, all of it inside K
    __device__ __forceinline__ void load(Regs<T, FW> &g, int kc) const
    {
        const DG_GLOBAL T *q =
            scalar(p + (UNIT ? (ptrdiff_t)kc * ld : (ptrdiff_t)kc));
        if (UNIT) {
#pragma unroll
            for (int v = 0; v < V; v++) {
                const DG_GLOBAL T *qv = scalar(q + (ptrdiff_t)v * ld);
#pragma unroll
                for (int i = 0; i < FW; i++) g.v[i][v] = at<T>(qv, off[i]);
            }
        }
        else if (vec && kc % V == 0) {
#pragma unroll
            for (int i = 0; i < FW; i++) {
                const vec_t x = at<vec_t>(q, off[i]);
#pragma unroll
                for (int v = 0; v < V; v++) g.v[i][v] = x[v];
            }
        }
        else {
#pragma unroll
            for (int i = 0; i < FW; i++)
#pragma unroll
                for (int v = 0; v < V; v++) g.v[i][v] = at<T>(scalar(q + v), off[i]);
        }
    }
    // the last, partial chunk: k values past K read as zero
    __device__ __forceinline__ void load_tail(Regs<T, FW> &g, int kc,
                                              int K) const
    {
        const int h = V * ((threadIdx.x & 63) / 16);
#pragma unroll
        for (int i = 0; i < FW; i++)
#pragma unroll
            for (int v = 0; v < V; v++) {
                const bool in = kc + h + v < K;
                // a lane whose value is outside reads the first one
                const DG_GLOBAL T *q = p + (in ? (UNIT ? (ptrdiff_t)(kc + v) * ld
                                             : (ptrdiff_t)(kc + v))
                                     : (UNIT ? -(ptrdiff_t)h * ld
                                             : -(ptrdiff_t)h));
                const T x = at<T>(q, off[i]);
                g.v[i][v] = in ? x : T(0);
            }
    }
};

// CROW: C has unit row stride (the product is formed as Y X^T, so that 16
// consecutive rows of a C column sit in 16 lanes); ACC: C is read, and the
// product is subtracted from it, with SEGS by segments of k.
template <typename T, int FW, bool CROW, bool ACC, bool XU, bool YU, bool SEGS>
__device__ __forceinline__ void run(tg::Job<T> job)
{
    constexpr int V = Chunk<T>::V, KC = Chunk<T>::KC, WT = 16 * FW;
    typedef typename Mfma<T>::acc_t acc_t;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = (wave >> 1) * WT, wc = (wave & 1) * WT;
    job.xrows = uni(job.xrows);
    job.yrows = uni(job.yrows);
    job.K = uni(job.K);
    DG_GLOBAL T *cp = uni(job.C.p);
    job.C.rs = uni(job.C.rs);
    job.C.cs = uni(job.C.cs);
    job.lower = uni(job.lower);
    if (wr >= job.xrows || wc >= job.yrows) return;

    Operand<T, FW, XU> X;
    Operand<T, FW, YU> Y;
    X.init(job.X, wr, job.xrows);
    Y.init(job.Y, wc, job.yrows);
    const int nk = job.K / KC;          // whole chunks
    auto crow = [&](int i, int q) {
        return wr + 16 * i + (CROW ? lane % 16 : Mfma<T>::row(lane, q));
    };
    auto ccol = [&](int j, int q) {
        return wc + 16 * j + (CROW ? Mfma<T>::row(lane, q) : lane % 16);
    };
    // C element (i, j, q) at a lane offset plus a scalar one
    constexpr int QS = sizeof(T) == 8 ? 4 : 1;      // Mfma<T>::row per q
    const int crs = job.C.rs, ccs = job.C.cs;
    const unsigned clane = sizeof(T) * (CROW
        ? (lane % 16) * crs + Mfma<T>::row(lane, 0) * ccs
        : Mfma<T>::row(lane, 0) * crs + (lane % 16) * ccs);
    auto cref = [&](DG_GLOBAL T *q) -> DG_GLOBAL T & {
        return *(DG_GLOBAL T *)((DG_GLOBAL char *)q + clane);
    };
    auto cptr = [&](int i, int j, int q) {
        return scalar(cp + (ptrdiff_t)(wr + 16 * i) * crs +
                      (ptrdiff_t)(wc + 16 * j) * ccs +
                      (ptrdiff_t)(q * QS) * (CROW ? ccs : crs));
    };
    auto inside = [&](int i, int j, int q) {
        return crow(i, q) < job.xrows && ccol(j, q) < job.yrows;
    };
    const bool full = wr + WT <= job.xrows && wc + WT <= job.yrows;
    acc_t acc[FW][FW];
    T c0[FW][FW][4];
    if (ACC && full) {
#pragma unroll
        for (int i = 0; i < FW; i++)
#pragma unroll
            for (int j = 0; j < FW; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    c0[i][j][q] = cref(cptr(i, j, q));
    }
    else if (ACC) {
#pragma unroll
        for (int i = 0; i < FW; i++)
#pragma unroll
            for (int j = 0; j < FW; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    c0[i][j][q] = T(0);
                    if (inside(i, j, q)) c0[i][j][q] = cref(cptr(i, j, q));
                }
    }
#pragma unroll
    for (int i = 0; i < FW; i++)
#pragma unroll
        for (int j = 0; j < FW; j++) acc[i][j] = acc_t{0, 0, 0, 0};

    auto step = [&](const Regs<T, FW> &x, const Regs<T, FW> &y) {
#pragma unroll
        for (int v = 0; v < V; v++)
#pragma unroll
            for (int i = 0; i < FW; i++)
#pragma unroll
                for (int j = 0; j < FW; j++)
                    acc[i][j] = CROW
                        ? Mfma<T>::mma(y.v[j][v], x.v[i][v], acc[i][j])
                        : Mfma<T>::mma(x.v[i][v], y.v[j][v], acc[i][j]);
    };
    // C's loads go first, so that waiting for a chunk never waits for a later
    // load
    __builtin_amdgcn_sched_barrier(0);
    // The product of SEG chunks (16 k values) is summed by itself and then
    // subtracted from C (SEGS).  One sum over all K rounds K / 4 times at the
    // size of that sum, also where C nearly cancels it, as in the trailing blocks
    // of a kernel (RBF) matrix; one chain that starts from C rounds as often at
    // the size of C, too often where little is subtracted.  Error of the FP64
    // factor against long double, n = 1000: RBF, noise 1e-3, 471 u with one sum,
    // 213 u with a chain, 248 u in segments of 32 and 215 u in segments of 16; for
    // G G^T / n + I 1.6, 4.6, 1.1 and 1.4 u.  The subtraction follows the first
    // chunk of the next segment, so that it does not wait for the matrix unit:
    // dposv n = 2049 takes 1327 us with and without segments.
    constexpr int SEG = 16 / KC;
    auto chunk = [&](int u, const Regs<T, FW> &x, const Regs<T, FW> &y) {
        if (!ACC || !SEGS || u % SEG != 0) {
            step(x, y);
            return;
        }
        acc_t prev[FW][FW];
#pragma unroll
        for (int i = 0; i < FW; i++)
#pragma unroll
            for (int j = 0; j < FW; j++) {
                prev[i][j] = acc[i][j];
                acc[i][j] = acc_t{0, 0, 0, 0};
            }
        step(x, y);
#pragma unroll
        for (int i = 0; i < FW; i++)
#pragma unroll
            for (int j = 0; j < FW; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) c0[i][j][q] -= prev[i][j][q];
    };
    Regs<T, FW> gx[RING], gy[RING];
    static_assert(RING % SEG == 0, "a segment ends inside the ring");
    if (nk >= RING) {
#pragma unroll
        for (int u = 0; u < RING; u++) {
            X.load(gx[u], u * KC);
            Y.load(gy[u], u * KC);
            __builtin_amdgcn_sched_barrier(0);
        }
        int kc = 0;
        for (; kc + 2 * RING <= nk; kc += RING) {
#pragma unroll
            for (int u = 0; u < RING; u++) {
                chunk(u, gx[u], gy[u]);
                X.load(gx[u], (kc + RING + u) * KC);
                Y.load(gy[u], (kc + RING + u) * KC);
                // keep the loads this far ahead of their use
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the ring, and up to RING - 1 chunks still to load
#pragma unroll
        for (int u = 0; u < RING; u++) {
            chunk(u, gx[u], gy[u]);
            if (kc + RING + u < nk) {
                X.load(gx[u], (kc + RING + u) * KC);
                Y.load(gy[u], (kc + RING + u) * KC);
            }
        }
#pragma unroll
        for (int u = 0; u < RING - 1; u++)
            if (kc + RING + u < nk) chunk(u, gx[u], gy[u]);
    }
    else {
        for (int kc = 0; kc < nk; kc++) {
            X.load(gx[0], kc * KC);
            Y.load(gy[0], kc * KC);
            step(gx[0], gy[0]);
        }
    }
    if (job.K % KC != 0) {
        X.load_tail(gx[0], nk * KC, job.K);
        Y.load_tail(gy[0], nk * KC, job.K);
        step(gx[0], gy[0]);
    }

    const bool all = full && !job.lower;
#pragma unroll
    for (int i = 0; i < FW; i++)
#pragma unroll
        for (int j = 0; j < FW; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (all || (inside(i, j, q) &&
                            (!job.lower ||
                             ccol(j, q) + job.diag_off <= crow(i, q))))
                    cref(cptr(i, j, q)) = ACC ? c0[i][j][q] - acc[i][j][q]
                                               : acc[i][j][q];
}

template <typename T, int FW, bool CROW, bool ACC, bool XU, bool YU,
          typename Decode>
__global__ __launch_bounds__(NT, 2) void kernel(Decode dec, int njobs,
                                                const int *status)
{
    if (block_should_stop(status)) return;
    const int padded = tg::xcd_grid(njobs), chunk = padded / tg::NXCD;
    const int b = blockIdx.x;
    const int jb = (b % tg::NXCD) * chunk + b / tg::NXCD;
    tg::Job<T> job;
    if (jb >= njobs || !dec(jb, job)) return;
    run<T, FW, CROW, ACC, XU, YU, Decode::SEGS>(job);
}

// Block width of the direct kernel for a launch of n128
// 128 x 128 blocks, in units of 32; 0: the staged kernels.  Up to W_32 of
// them even 64 x 64 blocks leave most CUs idle; beyond W_64 (two rounds of
// the chip's workgroup slots) the staged kernels' smaller operand traffic
// counts.  FP64 solves (nrhs 64 / 10 / 1): n = 500 512 us with the staged
// kernels alone, 444 with 64 x 64 blocks, 437 with both widths; n = 2049
// 2186, 1762, 1734 us; n = 8192 12.6, 10.1, 10.0 ms.  W_64 = 512: n = 16384
// 40.3 ms, 1024: 40.1, 2048: 40.0 (staged alone 44.0); W_32 = 64: n = 8192
// 10.2 ms.  One launch at n = 8192: panel 28.6 -> 16.8 us beside the bulk
// update, next column's update (K = 128) 27 -> 12 us.
constexpr long W_32 = 24, W_64 = 1024;

inline int width(long n128)
{
    return n128 <= W_32 ? 1 : n128 <= W_64 ? 2 : 0;
}

}  // namespace dg
