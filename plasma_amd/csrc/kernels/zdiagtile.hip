// zdiagtile.hip -- the diagonal tile of the complex tile Cholesky for tiles of
// order n <= 128: L L^H = A and W = L^{-1} in one pass, the whole tile in LDS.
//
// The complex counterpart of the real diagonal tile (diagtile.hip; reference
// core_zpotrf in compute/pzpotrf.c:41-45): 16-column panels of [A; I], each
// eliminated in the registers of two waves, and the trailing blocks updated by
// the matrix cores.  The identity's rows turn into L^{-H}, so W needs no pass
// of its own.
//
// 36 slots of 16 x 16 complex elements are 147 KB of the 160 KB of LDS: there
// is no room for a separate panel as in the real kernel.  The results of
// panel J stay in the slots of column J (and row J for the identity's rows);
// only two blocks have a place of their own, X0 (the row block J + 1, whose
// slot the block L^{-H}(J, J + 1) takes in the same phase) and X1 (the
// diagonal block).  The blocks L^{-H}(J, c), c > J + 1, are born in the slot
// of the panel block they are made from, after everything else that reads
// it:
//
//   phase A   waves 0, 1: panel J in registers; waves 2 .. 7: the rest of
//             step J - 1 (columns J + 1 .. , stores)
//   phase B   waves 0, 1: panel J to LDS; waves 2 .. 7: the blocks born in
//             step J - 1, one each
//   phase C   column J + 1, one block per wave
//
// Element (r, c) of a slot lies at 16 c + (r ^ c): column reads stay one
// contiguous (permuted) line, row reads (the stores that run along rows) are
// free of bank conflicts as well.
//
// Measured, one 128 x 128 tile in FP64: 63 us (in global memory with 32-column
// blocks, zchol.hip: 322 us); zposv n = 5001, 40 such tiles in a chain: 25.3 ->
// 16.3 ms.  Bound by the panel's chain of multiply-adds: 8 for each of the 120
// column pairs, in two waves.
#include "common.hip.h"
#include "panel16.hip.h"
#include "plasma_kernels.h"
#include "zview.hip.h"

namespace {

using namespace p16;

constexpr int ZD_NT = 512;              // 8 waves
constexpr int ZD_MAXB = 8;              // 16-blocks per tile side
constexpr int ZD_SLOTS = ZD_MAXB * (ZD_MAXB + 1) / 2;
constexpr int ZD_BLK = 256;             // elements of a slot

__host__ __device__ constexpr int ztri(int i, int j)
{
    return i * (i + 1) / 2 + j;
}
constexpr int ztri_row(int b)
{
    int i = 0;
    while (ztri(i + 1, 0) <= b) i++;
    return i;
}

// LDS (elements): slots, X0, X1, an identity block, info
constexpr int ZD_X0 = ZD_SLOTS * ZD_BLK;
constexpr int ZD_X1 = ZD_X0 + ZD_BLK;
constexpr int ZD_ID = ZD_X1 + ZD_BLK;
constexpr int ZD_INFO = ZD_ID + ZD_BLK;
template <typename R> constexpr size_t zd_lds = (ZD_INFO + 1) * sizeof(cx<R>);

__device__ __forceinline__ int at16(int r, int c) { return 16 * c + (r ^ c); }

// ---------------------------------------------------------------------------
// The panel in registers (panel16.hip.h in complex arithmetic): dd the
// diagonal block's rows, p the panel rows.  Column j eliminates column c by
//     s_c -= a_j conj(l_c),  l_c = lane c's element of the scaled column j,
// in sums s that start from zero; the column itself is added when its turn as
// the pivot column comes, and is read from LDS two columns before that (the
// identity's rows from a block of their own).  Eliminated in place the column is
// rounded 2 j times at its own size instead of once: error of the factor of one
// tile against long double 1.07 u instead of 0.67 u, at the same time.
// ---------------------------------------------------------------------------
template <typename R> struct Rows {
    R re[16], im[16];
};

// one column: 0-3 d.re, d.im, p.re, p.im; 4, 5 the scaled column of the
// diagonal block (the DPP source); 6, 7 that of the panel rows
#define Z16_COL(F, dr, di, pr, pi, c)                                          \
    F(dr, "%[lr]", "-%[lr]", c) F(di, "%[lr]", "-%[li]", c)                    \
    F(pr, "%[lr]", "-%[xr]", c) F(pi, "%[lr]", "-%[xi]", c)                    \
    F(dr, "%[li]", "-%[li]", c) F(di, "%[li]", "%[lr]", c)                     \
    F(pr, "%[li]", "-%[xi]", c) F(pi, "%[li]", "%[xr]", c)
#define Z16_F64(d, l, m, c)                                                    \
    "v_fmac_f64_dpp " d ", " l ", " m " row_newbcast:" c                      \
    " row_mask:0xf bank_mask:0xf\n\t"
#define Z16_F32(d, l, m, c)                                                    \
    "v_fmac_f32_dpp " d ", " l ", " m " row_newbcast:" c                      \
    " row_mask:0xf bank_mask:0xf\n\t"

// column C; columns C and C + 1
#define Z16_ELIM(T, F)                                                         \
    template <int C>                                                          \
    __device__ __forceinline__ void zelim1(Rows<T> &d, Rows<T> &p, T lr,      \
                                           T li, T xr, T xi)                  \
    {                                                                         \
        asm volatile("s_nop 1\n\t" Z16_COL(F, "%0", "%1", "%2", "%3", "%[c]") \
                     : "+v"(d.re[C]), "+v"(d.im[C]), "+v"(p.re[C]),           \
                       "+v"(p.im[C])                                          \
                     : [lr] "v"(lr), [li] "v"(li), [xr] "v"(xr),              \
                       [xi] "v"(xi), [c] "i"(C));                             \
    }                                                                         \
    template <int C>                                                          \
    __device__ __forceinline__ void zelim2(Rows<T> &d, Rows<T> &p, T lr,      \
                                           T li, T xr, T xi)                  \
    {                                                                         \
        asm volatile("s_nop 1\n\t" Z16_COL(F, "%0", "%1", "%2", "%3", "%[c]") \
                     Z16_COL(F, "%4", "%5", "%6", "%7", "%[c1]")              \
                     : "+v"(d.re[C]), "+v"(d.im[C]), "+v"(p.re[C]),           \
                       "+v"(p.im[C]), "+v"(d.re[C + 1]), "+v"(d.im[C + 1]),   \
                       "+v"(p.re[C + 1]), "+v"(p.im[C + 1])                   \
                     : [lr] "v"(lr), [li] "v"(li), [xr] "v"(xr),              \
                       [xi] "v"(xi), [c] "i"(C), [c1] "i"(C + 1));            \
    }
Z16_ELIM(double, Z16_F64)
Z16_ELIM(float, Z16_F32)

// columns C.. two at a time, one step of the next pivot's 1/sqrt after each
// group
template <typename R, int C, int S> struct ZElim {
    static __device__ __forceinline__ void run(Rows<R> &d, Rows<R> &p, R lr,
                                               R li, R xr, R xi,
                                               Rsqrt<R> &next)
    {
        constexpr int N = C + 1 < 16 ? 2 : 1;
        if constexpr (C + 1 < 16) zelim2<C>(d, p, lr, li, xr, xi);
        else if constexpr (C == 15) zelim1<C>(d, p, lr, li, xr, xi);
        if constexpr (S < Rsqrt<R>::steps) {
            next.template step<S>();
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (C < 16 || S < Rsqrt<R>::steps)
            ZElim<R, C + N, S + 1>::run(d, p, lr, li, xr, xi, next);
    }
};

// The original columns of the panel, read some columns ahead: the diagonal
// block's and the panel rows' element of this lane.
template <typename R> struct Ahead {
    static constexpr int N = 2;
    const cx<R> *ds, *ps;
    cx<R> d[N], p[N];
    template <int C> __device__ __forceinline__ void read(int r)
    {
        if constexpr (C < 16) {
            d[C % N] = ds[at16(r, C)];
            p[C % N] = ps[at16(r, C)];
        }
    }
};

template <typename R, int J> struct ZColumns {
    static __device__ __forceinline__ void run(Rows<R> &d, Rows<R> &p, R &piv,
                                               R y, int r, Ahead<R> &a)
    {
        const R lr = d.re[J] * y, li = d.im[J] * y;
        const R xr = p.re[J] * y, xi = p.im[J] * y;
        d.re[J] = lr;
        d.im[J] = li;
        p.re[J] = xr;
        p.im[J] = xi;
        if constexpr (J + 1 < 16) {
            Rsqrt<R> next;
            zelim1<J + 1>(d, p, lr, li, xr, xi);
            constexpr int N = (J + 1) % Ahead<R>::N;
            d.re[J + 1] += a.d[N].re;
            next.x = row_bcast<J + 1>(d.re[J + 1]);
            next.template step<0>();
            d.im[J + 1] += a.d[N].im;
            p.re[J + 1] += a.p[N].re;
            p.im[J + 1] += a.p[N].im;
            a.template read<J + 1 + Ahead<R>::N>(r);
            __builtin_amdgcn_sched_barrier(0);
            ZElim<R, J + 2, 1>::run(d, p, lr, li, xr, xi, next);
            piv = (r == J + 1) ? next.x : piv;
            ZColumns<R, J + 1>::run(d, p, piv, next.y, r, a);
        }
    }
};

// ---------------------------------------------------------------------------
// slot(r, c) -= sum_k Pb(r, k) conj(Pc(c, k)); `fresh`: the slot starts from
// zero (it may be Pc itself: all reads come before the writes).  The product
// is formed transposed, so operands and results are lane-linear, and summed
// before it meets the slot: added to the slot term by term it would be
// rounded 16 times at the slot's size.
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ void zslot_update(cx<R> *slot, const cx<R> *Pb,
                                             const cx<R> *Pc, bool fresh)
{
    const int lane = opaque(threadIdx.x & 63);
    const int l16 = lane & 15, lk = lane >> 4;
    cx<R> a[4], b[4], v[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        a[s] = Pc[at16(l16, 4 * s + lk)];
        b[s] = Pb[at16(l16, 4 * s + lk)];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = slot[at16(l16, Mfma<R>::row(lane, q))];
    typename Mfma<R>::acc_t re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++) {
        re = Mfma<R>::mma(a[s].re, b[s].re, re);
        im = Mfma<R>::mma(a[s].re, b[s].im, im);
        re = Mfma<R>::mma(a[s].im, b[s].im, re);
        im = Mfma<R>::mma(-a[s].im, b[s].re, im);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const cx<R> o = fresh ? czero<R>() : v[q];
        slot[at16(l16, Mfma<R>::row(lane, q))] =
            cx<R>{o.re - re[q], o.im - im[q]};
    }
}

// Where the results of panel K lie: row block b of the panel (b < nk: tile
// row block K + 1 + b; else the identity's row block b - nk).
__device__ __forceinline__ int zpanel_at(int K, int nk, int b)
{
    return b == 0 && nk > 0 ? ZD_X0
                            : (b < nk ? ztri(K + 1 + b, K)
                                      : ztri(K, b - nk)) * ZD_BLK;
}

// The results of step J from LDS to the tile and the workspace, by threads
// t of NT (all LDS reads before the first store).
template <typename R, int NT>
__device__ __forceinline__ void zstore_step(const CView<R> &L, int n,
                                            const CView<R> &Wv,
                                            const cx<R> *sm, int J, int nbk,
                                            int t)
{
    constexpr int IT = (ZD_MAXB + 1) * ZD_BLK / NT;
    const int nr = nbk - 1 - J;
    const bool up = L.rs != 1;
    cx<R> v[IT];
    // entry e: block e / 256 (0 .. nbk - 1 the panel's, 8 the diagonal one).
    // L goes out along the tile's contiguous index, W along its columns
    auto place = [&](int e, int &b, int &r, int &c) {
        const int lo = e & 15, hi = (e >> 4) & 15;
        b = e >> 8;
        const bool rfast = !up && (b < nr || b == ZD_MAXB);
        r = rfast ? lo : hi;
        c = rfast ? hi : lo;
    };
#pragma unroll
    for (int u = 0; u < IT; u++) {
        int b, r, c;
        place(t + u * NT, b, r, c);
        const int src = b == ZD_MAXB ? ZD_X1
                                     : zpanel_at(J, nr, min(b, nbk - 1));
        v[u] = sm[src + at16(r, c)];
    }
#pragma unroll
    for (int u = 0; u < IT; u++) {
        int b, r, c;
        place(t + u * NT, b, r, c);
        const int col = 16 * J + c;
        if (b < nr || b == ZD_MAXB) {
            const int row = 16 * (b == ZD_MAXB ? J : J + 1 + b) + r;
            if (row < n && col < n && row >= col) L.put(row, col, v[u]);
        }
        else if (b < nbk) {
            // W(16 J + c, 16 i + r) = conj of L^{-H} block (i, J)'s (r, c)
            const int wc = 16 * (b - nr) + r;
            if (col < n && wc < n)
                Wv.put(col, wc,
                       col < wc ? czero<R>() : cx<R>{v[u].re, -v[u].im});
        }
    }
}

// The tile (lower-equivalent view L, order n <= 128) factored in place, W =
// L^{-1} with zeros above its diagonal into Wv.  Returns 0 or the 1-based
// column of the first pivot that is not positive, the same in every thread;
// does nothing when *status is set (read beside the tile).
template <typename R>
__device__ int factor_zdiag128(const CView<R> &L, const int n,
                               const CView<R> &Wv, const int *status,
                               cx<R> *sm)
{
    int *sinfo = reinterpret_cast<int *>(sm + ZD_INFO);
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nbk = (n + 15) / 16;
    const bool up = L.rs != 1;

    // the tile into its slots, padded with the identity, the diagonal's
    // imaginary part dropped; two blocks per pass, all loads in flight before
    // the first LDS store
    {
        const int e = t & 255, h = __builtin_amdgcn_readfirstlane(t >> 8);
        const int rr = up ? e >> 4 : e & 15, cc = up ? e & 15 : e >> 4;
        cx<R> x[ZD_SLOTS / 2];
#pragma unroll
        for (int s = 0; s < ZD_SLOTS / 2; s++) {
            constexpr auto I = [](int b) constexpr { return ztri_row(b); };
            const int I0 = I(2 * s), I1 = I(2 * s + 1);
            const int bi = h ? I1 : I0;
            const int bj = h ? 2 * s + 1 - ztri(I1, 0) : 2 * s - ztri(I0, 0);
            x[s] = L.raw(min(16 * bi + rr, n - 1), min(16 * bj + cc, n - 1));
        }
#pragma unroll
        for (int s = 0; s < ZD_SLOTS / 2; s++) {
            constexpr auto I = [](int b) constexpr { return ztri_row(b); };
            const int I0 = I(2 * s), I1 = I(2 * s + 1);
            const int bi = h ? I1 : I0;
            const int bj = h ? 2 * s + 1 - ztri(I1, 0) : 2 * s - ztri(I0, 0);
            const int r = 16 * bi + rr, c = 16 * bj + cc;
            cx<R> v{r == c ? R(1) : R(0), R(0)};
            if (r < n && c < n && c <= r) {
                v = x[s];
                if (c == r) v.im = R(0);
            }
            sm[(2 * s + h) * ZD_BLK + at16(rr, cc)] = v;
        }
    }
    if (t < ZD_BLK)
        sm[ZD_ID + at16(t & 15, t >> 4)] =
            cx<R>{(t & 15) == t >> 4 ? R(1) : R(0), R(0)};
    if (t == 0) *sinfo = seq_failed(status) ? 1 : 0;
    __syncthreads();
    if (*sinfo) return 0;

    for (int J = 0; J < nbk; J++) {
        const int nr = nbk - 1 - J;         // tile row blocks below J
        const int K = J - 1, nk = nr + 1;   // the step before
        Rows<R> dd, p;
        R piv = R(1);
        const int r16 = lane & 15, b = 4 * wave + (lane >> 4);
        // phase A
        if (wave < 2) {
            const int rp = opaque(r16);
            const int i = b - nr;           // identity row block
            Ahead<R> a;
            a.ds = sm + ztri(J, J) * ZD_BLK;
            a.ps = sm + (b < nr  ? ztri(J + 1 + b, J) * ZD_BLK
                         : i < J ? ztri(J, i) * ZD_BLK : ZD_ID);
            a.template read<0>(rp);
#pragma unroll
            for (int c = 1; c < 16; c++)
                dd.re[c] = dd.im[c] = p.re[c] = p.im[c] = R(0);
            dd.re[0] = a.d[0].re;
            dd.im[0] = a.d[0].im;
            p.re[0] = a.p[0].re;
            p.im[0] = a.p[0].im;
            a.template read<1>(rp);
            a.template read<2>(rp);
            Rsqrt<R> first;
            first.x = piv = row_bcast<0>(dd.re[0]);
            first.template step<0>();
            first.rest();
            ZColumns<R, 0>::run(dd, p, piv, first.y, rp, a);
        }
        else if (J > 0) {
            // step K beside the panel: its columns c from J + 1 on (row
            // blocks c - J .. nbk - 2 of the panel each; block nbk - 1, the
            // identity's row block K, is born in phase B), and its stores
            int c = K + 2, bb = 1 + wave - 2;
            for (;;) {
                while (c < nbk && bb >= nbk - 1) {
                    bb += c - K - (nbk - 1);
                    c++;
                }
                if (c >= nbk) break;
                zslot_update<R>(sm + (bb < nk ? ztri(K + 1 + bb, c)
                                              : ztri(c, bb - nk)) * ZD_BLK,
                                sm + zpanel_at(K, nk, bb),
                                sm + zpanel_at(K, nk, c - K - 1), false);
                bb += ZD_NT / 64 - 2;
            }
            zstore_step<R, ZD_NT - 128>(L, n, Wv, sm, K, nbk,
                                        opaque(t - 128));
        }
        else {
            // zeros above the diagonal blocks of W
            for (int c = 16 + wave - 2; c < n; c += ZD_NT / 64 - 2)
                for (int r = lane; r < (c & ~15); r += 64)
                    Wv.put(r, c, czero<R>());
        }
        __syncthreads();
        // phase B
        if (wave < 2) {
            if (b < nbk) {
                const int rw = opaque(r16);
                cx<R> *pb = sm + zpanel_at(J, nr, b);
#pragma unroll
                for (int c = 0; c < 16; c++)
                    pb[at16(rw, c)] = cx<R>{p.re[c], p.im[c]};
            }
            if (wave == 0) {
                if (lane < 16) {
                    const int rw = opaque(r16);
                    cx<R> *pd = sm + ZD_X1;
#pragma unroll
                    for (int c = 0; c < 16; c++)
                        pd[at16(rw, c)] = cx<R>{dd.re[c], dd.im[c]};
                    // the diagonal itself: the correctly rounded root
                    pd[at16(rw, rw)] = cx<R>{(R)sqrt(piv), R(0)};
                }
                const unsigned long long bad = __ballot(!(piv > R(0)));
                if (lane == 0)
                    *sinfo = bad ? 16 * J + __ffsll(bad) : 0;
            }
        }
        else if (J > 0 && K + wave < nbk) {
            // L^{-H}(K, c), c = K + wave >= K + 2
            cx<R> *slot = sm + ztri(K + wave, K) * ZD_BLK;
            zslot_update<R>(slot, sm + ztri(K, K) * ZD_BLK, slot, true);
        }
        __syncthreads();
        const int info = *sinfo;
        if (info) return info;
        // phase C: column J + 1, one row block per wave
        if (J + 1 < nbk && wave < nbk)
            zslot_update<R>(sm + (wave < nr ? ztri(J + 1 + wave, J + 1)
                                            : ztri(J + 1, wave - nr)) *
                                     ZD_BLK,
                            sm + zpanel_at(J, nr, wave), sm + ZD_X0,
                            wave - nr == J);
        __syncthreads();
    }
    // six of the eight waves: 2304 entries are not a multiple of 512 threads
    if (t < 384)
        zstore_step<R, ZD_NT - 128>(L, n, Wv, sm, nbk - 1, nbk, t);
    return 0;
}

template <typename R>
__global__ __launch_bounds__(ZD_NT, 2) void zdiag128_kernel(
    plasma_desc_t A, int upper, int k, cx<R> *inv, int *status)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const CView<R> Wv = buf_cview(inv + (size_t)k * A.mb * A.mb, A.mb);
    const int info = factor_zdiag128<R>(lower_cview<R>(A, upper != 0, k, k),
                                        plasma_tile_mview(A, k), Wv, status,
                                        reinterpret_cast<cx<R> *>(smem_raw));
    if (info && threadIdx.x == 0) atomicCAS(status, 0, A.nb * k + info);
}

template <typename R>
int launch_zdiag128(plasma_enum_t uplo, plasma_desc_t A, int k, void *inv,
                    int *status, hipStream_t s)
{
    constexpr size_t lds = zd_lds<R>;
    if (lds > 65536) {
        static unsigned long long done = 0;     // a bit per device
        int dev = 0;
        (void)hipGetDevice(&dev);
        const unsigned long long bit = 1ull << (dev & 63);
        if (!(__atomic_load_n(&done, __ATOMIC_RELAXED) & bit)) {
            (void)hipFuncSetAttribute((const void *)zdiag128_kernel<R>,
                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            __atomic_fetch_or(&done, bit, __ATOMIC_RELAXED);
        }
    }
    hipLaunchKernelGGL(zdiag128_kernel<R>, dim3(1), dim3(ZD_NT), lds, s, A,
                       uplo == PlasmaUpper, k, (cx<R> *)inv, status);
    return hipGetLastError() == hipSuccess ? 0 : PlasmaErrorInternal;
}

}  // namespace

// Tiles that fit LDS; larger ones are factored in global memory (zchol.hip).
extern "C" int plasma_zdiag128_ok(plasma_desc_t A)
{
    return A.mb <= 16 * ZD_MAXB && A.mb == A.nb &&
           (A.precision == PlasmaComplexDouble ||
            A.precision == PlasmaComplexFloat);
}

extern "C" int plasma_kern_zdiag128(plasma_enum_t uplo, plasma_desc_t A,
                                    int k, void *inv, int *status,
                                    hipStream_t s)
{
    if (!plasma_zdiag128_ok(A)) return PlasmaErrorNotSupported;
    if (A.precision == PlasmaComplexDouble)
        return launch_zdiag128<double>(uplo, A, k, inv, status, s);
    return launch_zdiag128<float>(uplo, A, k, inv, status, s);
}
