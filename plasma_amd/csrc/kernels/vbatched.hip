// vbatched.hip -- many independent SPD systems of uneven order n <= 512, up
// to 16 right-hand sides each (no counterpart in the reference, which factors
// one matrix per call; compute/batched.c holds the entry points).
//
// One workgroup of NW waves per system, NW = 2, 4, 8 for n <= 128, 256, 512,
// so that small systems share a CU (16 waves of at most 128 registers: eight,
// four or two workgroups) and hide each other's latency.  A persistent grid
// per class takes its systems from a ticket.
//
// Left-looking by block columns J of 16, the matrix in place in global memory
// (L2), only the block column in LDS:
//   1. the waves put A(:, J) into LDS by strips of 16 rows and subtract
//      L(:, <J) L(J, <J)^T from it on MFMA, operands straight from L2 (the
//      matrix is read about n / 96 times and written once; a right-looking
//      update would also write it that often);
//   2. every wave eliminates the 16 columns for up to 64 of its rows
//      (panel16.hip.h; each repeats the diagonal block, so the pivots need no
//      exchange) and stores them.
// The right-hand sides ride along as one more strip of rows: [A; b^T] L^{-T}
// gives y^T = (L^{-1} b)^T, kept in the workgroup's slab of workspace, so the
// forward solve costs no pass of its own and B stays untouched until the
// factorization has succeeded.  L^T X = Y then goes backwards by 16 rows for
// all right-hand sides together: one wave solves the diagonal block in
// registers (16 steps), then the waves update the rows above on MFMA.
// Measured: 1024 FP64 systems of 32 to 512 unknowns 2.71 -> 1.80 ms; 4096 FP32
// systems of 8 to 128 unknowns 700 -> 250 us (427 of them before the host
// side ordered by counting and sent its arrays in one copy).  One 512 x 512
// FP64 system: 0.72 ms alone, 0.83 ms with one system per CU, of which the
// products take 0.44 ms (matrix-core floor 0.16; every MFMA needs 1.4 operand
// loads of 512 bytes, most of what a CU's L1 delivers).
#include "common.hip.h"
#include "directgemm.hip.h"
#include "panel16.hip.h"
#include "plasma_kernels.h"

namespace {

using namespace p16;

constexpr int VN_LD = 17;
constexpr int VN_BLK = 16 * VN_LD;
constexpr int VN_RHS = 16;              // right-hand sides at most

// a scalar the compiler does not derive anything from ahead of its use
__device__ __forceinline__ int opaque_s(int x)
{
    x = dg::uni(x);
    asm("" : "+s"(x));
    return x;
}

// (block of strip g in LDS) -= (rows of strip g) (rows of block row J)^T over
// columns 0 .. j0-1, more chunks in flight the fewer strips share a wave's
// registers.
//
// The product of 32 columns at a time is summed by itself and then subtracted
// from the block.  One sum over all columns rounds j0 / 4 times at the size of
// that sum: what is left of A below it is far smaller in a kernel (RBF) matrix
// (noise 1e-3, error of the FP64 factor against long double with one sum and
// with this: n = 128 17 and 12.5 u, 256 61 and 33 u, 512 239 and 91 u); one chain
// that starts from the block rounds as often at the block's size, and that is
// too often where little is subtracted (G G^T / n + I).  It costs the LDS traffic:
// 1024 FP64 systems of 32 to 512 unknowns 1.77 -> 1.80 ms; FP32, which summed 32
// columns apart before but added them up, 4096 systems of 8 to 128 unknowns 251 ->
// 246 us.  Sums of 64 columns: 137 u at n = 512, and slower.  Adding in LDS by its
// FP64 atomics: 1.85 ms.
// The blocks are at `own` and every STRIDE elements after it, the last one at
// `last`.
template <typename T, int CNT, bool UNIT, int STRIDE>
__device__ __forceinline__ void strip_products(
    T *own, T *last, const dg::Operand<T, 1, UNIT> (&op)[4],
    const dg::Operand<T, 1, UNIT> &bop, int j0)
{
    constexpr int KC = dg::Chunk<T>::KC, V = dg::Chunk<T>::V;
    constexpr int R = CNT <= 2 ? 4 : 2;
    constexpr int SEG = 32 / KC;        // chunks summed by themselves
    typename Mfma<T>::acc_t acc[CNT];
    dg::Regs<T, 1> x[R][CNT], b[R];
    // j0 is a multiple of 16, i.e. of KC, and positive; a chunk past the end
    // reads the last one again
    auto load = [&](int u, int i) {
        const int kc = min(i * KC, j0 - KC);
        bop.load(b[u], kc);
#pragma unroll
        for (int g = 0; g < CNT; g++) op[g].load(x[u][g], kc);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto clear = [&]() {
#pragma unroll
        for (int g = 0; g < CNT; g++)
            acc[g] = typename Mfma<T>::acc_t{0, 0, 0, 0};
    };
    auto flush = [&]() {
        const int l = opaque(threadIdx.x & 63);
        const int o = Mfma<T>::row(l, 0) * VN_LD + (l & 15);
        constexpr int QS = (sizeof(T) == 8 ? 4 : 1) * VN_LD;
#pragma unroll
        for (int g = 0; g < CNT; g++) {
            T *blk = (g + 1 < CNT ? own + g * STRIDE : last) + o;
#pragma unroll
            for (int e = 0; e < 4; e++) blk[e * QS] -= acc[g][e];
        }
        clear();
    };
    auto step = [&](int u) {
#pragma unroll
        for (int v = 0; v < V; v++)
#pragma unroll
            for (int g = 0; g < CNT; g++)
                acc[g] = Mfma<T>::mma(b[u].v[0][v], x[u][g].v[0][v], acc[g]);
    };
    const int nk = j0 / KC;
#pragma unroll
    for (int u = 0; u < R; u++) load(u, u);
    clear();
    constexpr int N = R > SEG ? R : SEG;        // chunks per round
    int i = 0;
    for (; i + N <= nk; i += N) {
#pragma unroll
        for (int u = 0; u < N; u++) {
            step(u % R);
            load(u % R, i + R + u);
            if ((u + 1) % SEG == 0) flush();
        }
    }
#pragma unroll
    for (int u = 0; u < N - 1; u++) {
        if (i + u >= nk) break;
        step(u % R);
        if (u + R < N - 1) load(u % R, i + R + u);
        if ((u + 1) % SEG == 0) flush();
    }
    if (nk % SEG != 0) flush();
}

// x in lane i of a 16-lane row: the equations K, K - 1, .. of L^T x = t with
// column i of L in lc (zero up to the diagonal) and 1 / L(i, i) in rd; x * rd
// is the solution afterwards
template <typename T, int K> struct BackSolve {
    static __device__ __forceinline__ void run(T &x, const T (&lc)[16], T rd)
    {
        if constexpr (K > 0) {
            x = __builtin_elementwise_fma(-lc[K], row_bcast<K>(x * rd), x);
            BackSolve<T, K - 1>::run(x, lc, rd);
        }
    }
};

template <typename T, int NW, bool UPPER>
__global__ __launch_bounds__(64 * NW, 4) void vbatched16_kernel(
    int lo, int hi, const int *nvec, T *A, const size_t *aoff, T *W, int nrhs,
    T *B, const size_t *boff, int *info, const int *order, int *ticket)
{
    typedef typename Mfma<T>::acc_t acc_t;
    constexpr int NMAX = 64 * NW;
    constexpr bool UNIT = !UPPER;
    __shared__ T sblk[(4 * NW + 1) * VN_BLK];   // block 0: diagonal
    __shared__ int s_i;
    const int lane = threadIdx.x & 63, r16 = lane & 15;
    const int wave = dg::uni(threadIdx.x >> 6);
    // y^T: element (rhs r, column k), contiguous along r for lower storage,
    // along k for upper (as the rows of the matrix)
    View<T> Y;
    Y.p = W + (size_t)blockIdx.x * VN_RHS * NMAX;
    Y.rs = UPPER ? NMAX : 1;
    Y.cs = UPPER ? 1 : VN_RHS;

    for (;;) {
        if (threadIdx.x == 0) s_i = lo + atomicAdd(ticket, 1);
        __syncthreads();
        const int i = dg::uni(s_i);
        __syncthreads();
        if (i >= hi) break;
        const int sys = dg::uni(order[i]);
        const int n = dg::uni(nvec[sys]);
        // an order outside the class (its argument check aside) or 0 takes
        // the same way through the barriers as any other: no `continue` here,
        // the compiler would send thread 0 and the other threads round the
        // loop on different paths
        const bool ok = n >= 0 && n <= NMAX;
        View<T> L;
        L.p = A + aoff[sys];
        L.rs = UPPER ? n : 1;
        L.cs = UPPER ? 1 : n;
        T *b = nrhs > 0 ? B + boff[sys] : nullptr;
        const int nbk = ok ? (n + 15) / 16 : 0;
        int fail = ok ? 0 : -3;

        for (int J = 0; J < nbk && fail == 0; J++) {
            const int j0 = 16 * J;
            const int ns = nbk - 1 - J;             // strips below J
            const int np = ns + (nrhs > 0);         // and the right-hand sides
            // this wave's strips q = wave, wave + NW, ..; the diagonal block
            // goes to the wave with the fewest
            const int cnt = wave < np ? (np - wave + NW - 1) / NW : 0;
            const bool diag = wave == np % NW;
            auto strip = [&](int g) {               // g == cnt: the diagonal
                return g < cnt ? wave + NW * g : -1;
            };
            const int all = cnt + diag;             // 5 only at J = 0
            // the blocks of A into LDS; padding is zero, on the diagonal one
            // (all loads at clamped addresses before the first use)
            const int l1 = opaque(lane), r1 = l1 & 15, n1 = opaque_s(n);
#pragma unroll
            for (int g0 = 0; g0 < 5; g0 += 3) {
                if (g0 >= all) break;
                T av[3][4];
#pragma unroll
                for (int g = g0; g < g0 + 3 && g < 5; g++) {
                    if (g >= all) break;
                    const int q = strip(g);
                    const bool rhs = q == ns;
                    const DG_GLOBAL T *src = dg::scalar(dg::uni(rhs ? b : L.p));
                    const int row = rhs ? min(r1, nrhs - 1)
                                        : min(j0 + 16 * (q + 1) + r1, n1 - 1);
                    const int rs = UPPER || rhs ? n1 : 1;
                    const int cs = UPPER || rhs ? 1 : n1;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int col = j0 + Mfma<T>::row(l1, e);
                        av[g - g0][e] = dg::Operand<T, 1, UNIT>::template at<T>(
                            src, sizeof(T) * (row * rs + min(col, n1 - 1) * cs));
                    }
            }
#pragma unroll
                for (int g = g0; g < g0 + 3 && g < 5; g++) {
                    if (g >= all) break;
                    const int q = strip(g);
                    const int row = q == ns ? (r1 < nrhs ? n1 : 2 * n1)
                                            : j0 + 16 * (q + 1) + r1;
                    T *blk = sblk + (q + 1) * VN_BLK;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        // inside: a row of the matrix or a right-hand side (row
                        // n1 here), columns up to the diagonal
                        const int c = Mfma<T>::row(l1, e), col = j0 + c;
                        const T pad = (q < 0 && r1 == c) ? T(1) : T(0);
                        const bool in = col < n1 && col <= row &&
                                        row < (q == ns ? n1 + 1 : n1);
                        blk[c * VN_LD + r1] = in ? av[g - g0][e] : pad;
                    }
                }
            }
            // minus the products, each wave in its own blocks
            if (J > 0 && all > 0) {
                dg::Operand<T, 1, UNIT> op[4], bop;
                bop.init(L, j0, n);
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int q = strip(g);
                    if (q == ns)     op[g].init(Y, 0, VN_RHS);
                    else if (q >= 0) op[g].init(L, j0 + 16 + 16 * q, n);
                    else             op[g] = bop;
                }
                constexpr int ST = NW * VN_BLK;
                T *own = sblk + (wave + 1) * VN_BLK;
                T *last = diag ? sblk : own + (all - 1) * ST;
                if (all == 1)
                    strip_products<T, 1, UNIT, ST>(own, last, op, bop, j0);
                else if (all == 2)
                    strip_products<T, 2, UNIT, ST>(own, last, op, bop, j0);
                else if (all == 3)
                    strip_products<T, 3, UNIT, ST>(own, last, op, bop, j0);
                else
                    strip_products<T, 4, UNIT, ST>(own, last, op, bop, j0);
                // the padding of a last, partial block column again
                if (diag && j0 + 16 > n) {
                    const int l0 = opaque(lane), r0 = l0 & 15;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int c = Mfma<T>::row(l0, e);
                        if (j0 + max(r0, c) >= n)
                            sblk[c * VN_LD + r0] = r0 == c ? T(1) : T(0);
                    }
                }
            }
            __syncthreads();

            // the panel: lane group g holds strip wave + NW g
            T dd[16], p[16], piv;
            const int l2 = opaque(lane), r2 = l2 & 15;
            const int pq = wave + NW * (l2 >> 4);
            const T *ps = sblk + (pq < np ? pq + 1 : 0) * VN_BLK + r2;
#pragma unroll
            for (int c = 0; c < 16; c++) {
                dd[c] = sblk[c * VN_LD + r2];
                p[c] = ps[c * VN_LD];
            }
            Rsqrt<T> first;
            first.x = piv = row_bcast<0>(dd[0]);
            first.template step<0>();
            first.rest();
            Columns<T, 0>::run(dd, p, piv, first.y, r2);
            const unsigned long long bad = __ballot(!(piv > T(0)));
            if (bad) fail = j0 + __ffsll((long long)bad);
            else {
                const int l3 = opaque(lane), r3 = l3 & 15;
                const int pq3 = wave + NW * (l3 >> 4);
                const int lcs = UPPER ? 1 : opaque_s(n);
                constexpr int ycs = UPPER ? 1 : VN_RHS;
                const int row = j0 + 16 + 16 * pq3 + r3;
                if (pq3 < ns && row < n) {
                    T *o = &L.at(row, j0);
#pragma unroll
                    for (int c = 0; c < 16; c++)
                        if (j0 + c < n) o[c * lcs] = p[c];
                }
                else if (pq3 == ns && nrhs > 0) {
                    T *o = &Y.at(r3, j0);
#pragma unroll
                    for (int c = 0; c < 16; c++) o[c * ycs] = p[c];
                }
                if (wave == np % NW && l3 < 16 && j0 + r3 < n) {
                    T *o = &L.at(j0 + r3, j0);
#pragma unroll
                    for (int c = 0; c < 16; c++)
                        if (c < r3) o[c * lcs] = dd[c];
                    // the diagonal itself: the correctly rounded root
                    o[r3 * lcs] = sqrt(piv);
                }
            }
            __syncthreads();
        }

        // L^T X = Y, all right-hand sides at once: X(k, rhs) in LDS
        if (fail == 0 && nrhs > 0) {
            T *sX = sblk;                           // n x 17, the panel's
            // (columns from nrhs on hold leftovers, which stay in them)
            for (int r = 0; r < nrhs; r++)
                if ((int)threadIdx.x < 16 * nbk)
                    sX[threadIdx.x * VN_LD + r] = Y.at(r, threadIdx.x);
            for (int J = nbk - 1; J >= 0; J--) {
                const int j0 = 16 * J, kv = min(16, n - j0);
                // this wave's strips I = wave, wave + NW, .. above
                const int cnt = wave < J ? (J - wave + NW - 1) / NW : 0;
                __syncthreads();                    // rows j0 .. are final
                if (wave == J % NW) {
                    // the diagonal block: lane group g takes right-hand
                    // sides g, g + 4, ..; lane i of it row i, with column i
                    // of the block (zero up to the diagonal)
                    const int l4 = opaque(lane), i = l4 & 15;
                    const int n4 = opaque_s(n);
                    T lc[16], dv = T(1);
                    const DG_GLOBAL T *lp = dg::scalar(dg::uni(L.p));
#pragma unroll
                    for (int k = 0; k < 16; k++) {
                        const int row = min(j0 + k, n4 - 1);
                        const int col = min(j0 + i, n4 - 1);
                        lc[k] = dg::Operand<T, 1, UNIT>::template at<T>(
                            lp, sizeof(T) * (UPPER ? row * n4 + col
                                                   : col * n4 + row));
                    }
#pragma unroll
                    for (int k = 0; k < 16; k++) {
                        if (k == i && i < kv) dv = lc[k];
                        if (k <= i || k >= kv) lc[k] = T(0);
                    }
                    const T rd = T(1) / dv;
                    for (int r = l4 >> 4; r < VN_RHS; r += 4) {
                        if (dg::uni(r) >= nrhs) break;
                        T *xp = sX + (j0 + i) * VN_LD + r;
                        T x = i < kv ? *xp : T(0);
                        BackSolve<T, 15>::run(x, lc, rd);
                        *xp = x * rd;
                    }
                }
                // L(J, I)^T (in flight while that wave solves): row c of strip
                // I, k value V (lane / 16) + v of chunk ch, zero past the end
                constexpr int KC = dg::Chunk<T>::KC, V = dg::Chunk<T>::V;
                constexpr int NC = 16 / KC;
                T lt[4][NC][V];
                if (cnt > 0) {
                    const int l5 = opaque(lane), n5 = opaque_s(n);
                    const DG_GLOBAL T *lp = dg::scalar(dg::uni(L.p));
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const int I = wave + NW * min(g, cnt - 1);
                        const int c = 16 * I + l5 % 16;
#pragma unroll
                        for (int ch = 0; ch < NC; ch++)
#pragma unroll
                            for (int v = 0; v < V; v++) {
                                const int k = ch * KC + V * (l5 / 16) + v;
                                const int row = min(j0 + k, n5 - 1);
                                const T x =
                                    dg::Operand<T, 1, UNIT>::template at<T>(
                                        lp, sizeof(T) *
                                                (UPPER ? row * n5 + c
                                                       : c * n5 + row));
                                lt[g][ch][v] = k < kv ? x : T(0);
                            }
                    }
                }
                __syncthreads();
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    if (g >= cnt) break;
                    const int l6 = opaque(lane);
                    T *xp = sX + (16 * (wave + NW * g) +
                                  Mfma<T>::row(l6, 0)) * VN_LD + l6 % 16;
                    const T *xj = sX + (j0 + V * (l6 / 16)) * VN_LD + l6 % 16;
                    constexpr int QS = sizeof(T) == 8 ? 4 : 1;
                    acc_t sum = {0, 0, 0, 0};
#pragma unroll
                    for (int ch = 0; ch < NC; ch++)
#pragma unroll
                        for (int v = 0; v < V; v++)
                            sum = Mfma<T>::mma(lt[g][ch][v],
                                               xj[(ch * KC + v) * VN_LD], sum);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        xp[e * QS * VN_LD] -= sum[e];
                }
            }
            __syncthreads();
            for (int r = 0; r < nrhs; r++)
                if ((int)threadIdx.x < n)
                    b[r * n + threadIdx.x] = sX[threadIdx.x * VN_LD + r];
        }
        if (threadIdx.x == 0) info[sys] = fail;
        __syncthreads();
    }
}

// per class: waves, workgroups per CU
constexpr int VN_NW[3] = {8, 4, 2};

template <typename T, int NW>
void launch_class(int upper, int lo, int hi, const int *n, void *A,
                  const size_t *aoff, void *W, int nrhs, void *B,
                  const size_t *boff, int *info, const int *order,
                  int *ticket, int cus, hipStream_t s)
{
    if (hi <= lo) return;
    const int grid = min(hi - lo, cus * (16 / NW));
    if (upper)
        hipLaunchKernelGGL((vbatched16_kernel<T, NW, true>), dim3(grid),
                           dim3(64 * NW), 0, s, lo, hi, n, (T *)A, aoff,
                           (T *)W, nrhs, (T *)B, boff, info, order, ticket);
    else
        hipLaunchKernelGGL((vbatched16_kernel<T, NW, false>), dim3(grid),
                           dim3(64 * NW), 0, s, lo, hi, n, (T *)A, aoff,
                           (T *)W, nrhs, (T *)B, boff, info, order, ticket);
}

template <typename T>
int launch_vbatched16(int upper, int batch, const int *cls, const int *n,
                      void *A, const size_t *aoff, void *const W[3], int nrhs,
                      void *B, const size_t *boff, int *info,
                      const int *order, int *ticket, int cus,
                      hipStream_t const s[3])
{
    launch_class<T, 8>(upper, 0, cls[0], n, A, aoff, W[0], nrhs, B, boff, info,
                       order, ticket, cus, s[0]);
    launch_class<T, 4>(upper, cls[0], cls[1], n, A, aoff, W[1], nrhs, B, boff,
                       info, order, ticket + 1, cus, s[1]);
    launch_class<T, 2>(upper, cls[1], batch, n, A, aoff, W[2], nrhs, B, boff,
                       info, order, ticket + 2, cus, s[2]);
    return hipGetLastError() == hipSuccess ? 0 : PlasmaErrorInternal;
}

}  // namespace

extern "C" int plasma_vbatched16_ok(int nrhs)
{
    return nrhs <= VN_RHS;
}

extern "C" size_t plasma_vbatched16_bytes(plasma_enum_t precision, int cls,
                                          int count, int cus)
{
    const size_t es = precision == PlasmaRealDouble ? 8 : 4;
    const size_t grid = min(count, cus * (16 / VN_NW[cls]));
    return grid * VN_RHS * 64 * VN_NW[cls] * es;
}

extern "C" int plasma_kern_vbatched16(plasma_enum_t precision, int upper,
                                      int batch, const int cls[2],
                                      const int *n, void *A,
                                      const size_t *aoff, void *const W[3],
                                      int nrhs, void *B, const size_t *boff,
                                      int *info, const int *order,
                                      int *ticket, int cus,
                                      hipStream_t const s[3])
{
    if (nrhs > VN_RHS) return PlasmaErrorNotSupported;
    if (precision == PlasmaRealDouble)
        return launch_vbatched16<double>(upper, batch, cls, n, A, aoff, W,
                                         nrhs, B, boff, info, order, ticket,
                                         cus, s);
    if (precision == PlasmaRealFloat)
        return launch_vbatched16<float>(upper, batch, cls, n, A, aoff, W,
                                        nrhs, B, boff, info, order, ticket,
                                        cus, s);
    return PlasmaErrorNotSupported;
}
