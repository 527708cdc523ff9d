// diagtile.hip -- the diagonal tile of the tile Cholesky for tiles of order
// n <= 128: L L^T = A and W = L^{-1} in one pass, the whole tile in LDS.
//
// Replaces the potrf task of the reference's right-looking tile Cholesky
// (compute/pzpotrf.c:41-45).  It sits on the factorization's critical chain
// (diagonal tile, panel, next column), one workgroup on an otherwise busy
// chip, so what counts is its latency, not its rate.
//
// Algorithm: 16-column panels of the matrix [A; I].  Eliminating the columns
// of A from the identity's rows as well turns those rows into L^{-T}, so the
// inverse needs no pass of its own: at step J the rows still active are the
// tile's row blocks below J and the identity's row blocks 0..J, always
// nbk = ceil(n / 16) blocks.  The block L^{-T}(i, c), i < c, is born at step
// i, when the tile's block (c, i) has just been consumed, and takes its LDS
// slot: 36 slots of 16 x 16 hold everything (FP64 73.7 KB + a 20 KB panel).
//
//   panel J    two waves, no barrier and no LDS inside: every 16-lane row of
//              a wave holds the 16 rows of the diagonal block (dd, the same
//              in each row) and 16 panel rows (p); column j of L reaches the
//              lanes as the DPP operand (row_newbcast) of the multiply-adds.
//              The next pivot's 1/sqrt (the hardware estimate with one
//              third-order correction in FP64) runs between the
//              eliminations of the column before.
//   column J+1 one 16 x 16 MFMA block per wave (K = 16), then the panel
//              waves go on to panel J + 1
//   the rest   of the trailing update and the stores of step J run on the
//              other six waves beside panel J + 1.
//
// All LDS blocks are column major, so MFMA operands and results are
// lane-linear reads and writes (the product is formed transposed).
// Measured, one 128 x 128 tile: 29.5 us in FP64 and 23.5 us in FP32 (the tile
// in global memory with 32-column blocks, kernels/potrf.hip: 100 and 57 us).
// A step takes about 7000 cycles in FP64: panel 4400, panel to LDS 1000,
// column J + 1 1100.  Spills cost more than their instructions: with 22
// spilled registers (a kernel with scratch memory) the launch took 7 us
// longer, hence opaque() below.
#include "common.hip.h"
#include "panel16.hip.h"
#include "plasma_kernels.h"

namespace {

using namespace p16;

constexpr int DT_NT = 512;              // 8 waves
constexpr int DT_MAXB = 8;              // 16-blocks per tile side
constexpr int DT_SLOTS = DT_MAXB * (DT_MAXB + 1) / 2;
constexpr int DT_BLK = 256;             // elements of a slot
constexpr int DT_PLD = 17;              // panel block: column stride
constexpr int DT_PBLK = 16 * DT_PLD;

__host__ __device__ constexpr int tri(int i, int j)
{
    return i * (i + 1) / 2 + j;
}
constexpr int tri_row(int b)
{
    int i = 0;
    while (tri(i + 1, 0) <= b) i++;
    return i;
}

// LDS of one tile (elements): slots, panel (nbk row blocks + the diagonal
// block), info
template <typename T> struct DiagLds {
    static constexpr int S = 0;
    static constexpr int P = DT_SLOTS * DT_BLK;
    static constexpr int INFO = P + (DT_MAXB + 1) * DT_PBLK;
    static constexpr size_t bytes = (INFO + 2) * sizeof(T);
};

// slot (column major 16 x 16, element (r, c) at 16 c + r) -= Pb Pc^T with
// panel blocks Pb (the slot's rows) and Pc (its columns); `fresh`: the slot
// starts from zero.  The product is summed by itself: added to the slot term by
// term it rounds 16 times at the slot's size (error of the factor of one tile of
// order 128 against long double 1.90 u instead of 0.93 u in FP64, 1.89 u instead
// of 0.88 u in FP32).
template <typename T>
__device__ __forceinline__ void slot_update(T *slot, const T *Pb, const T *Pc,
                                            bool fresh)
{
    const int lane = opaque(threadIdx.x & 63);
    const int ro = (lane / 16) * DT_PLD + lane % 16;
    T a[4], b[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        a[s] = Pc[4 * s * DT_PLD + ro];
        b[s] = Pb[4 * s * DT_PLD + ro];
    }
    T v[4];
#pragma unroll
    for (int q = 0; q < 4; q++)
        v[q] = slot[16 * Mfma<T>::row(lane, q) + lane % 16];
    typename Mfma<T>::acc_t acc = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++) acc = Mfma<T>::mma(a[s], b[s], acc);
#pragma unroll
    for (int q = 0; q < 4; q++)
        slot[16 * Mfma<T>::row(lane, q) + lane % 16] =
            (fresh ? T(0) : v[q]) - acc[q];
}

// two independent blocks, their LDS reads and products interleaved
template <typename T>
__device__ __forceinline__ void slot_update2(T *s0, const T *Pb0,
                                             const T *Pc0, bool f0, T *s1,
                                             const T *Pb1, const T *Pc1,
                                             bool f1)
{
    const int lane = opaque(threadIdx.x & 63);
    const int ro = (lane / 16) * DT_PLD + lane % 16;
    T a0[4], b0[4], a1[4], b1[4], v0[4], v1[4];
    typename Mfma<T>::acc_t acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++) {
        a0[s] = Pc0[4 * s * DT_PLD + ro];
        b0[s] = Pb0[4 * s * DT_PLD + ro];
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
        v0[q] = s0[16 * Mfma<T>::row(lane, q) + lane % 16];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        a1[s] = Pc1[4 * s * DT_PLD + ro];
        b1[s] = Pb1[4 * s * DT_PLD + ro];
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
        v1[q] = s1[16 * Mfma<T>::row(lane, q) + lane % 16];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        acc0 = Mfma<T>::mma(a0[s], b0[s], acc0);
        acc1 = Mfma<T>::mma(a1[s], b1[s], acc1);
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
        s0[16 * Mfma<T>::row(lane, q) + lane % 16] =
            (f0 ? T(0) : v0[q]) - acc0[q];
#pragma unroll
    for (int q = 0; q < 4; q++)
        s1[16 * Mfma<T>::row(lane, q) + lane % 16] =
            (f1 ? T(0) : v1[q]) - acc1[q];
}

// The results of step J from the panel to the tile and the workspace, by
// threads t of NT (all LDS reads before the first store).
template <typename T, int NT>
__device__ __forceinline__ void store_step(const View<T> &L, int n,
                                           const View<T> &Wv, const T *sm,
                                           int J, int nbk, int t)
{
    constexpr int IT = (DT_MAXB + 1) * DT_BLK / NT;
    const T *P = sm + DiagLds<T>::P;
    const int nr = nbk - 1 - J;
    const bool up = L.rs != 1;
    T v[IT];
    // entry e: block e / 256 (0 .. nbk - 1 the panel's, 8 the diagonal one).
    // L goes out along the tile's contiguous index, W along its columns
    auto place = [&](int e, int &b, int &r, int &c) {
        const int lo = e & 15, hi = (e >> 4) & 15;
        b = e >> 8;
        const bool rfast = !up && (b < nr || b == DT_MAXB);
        r = rfast ? lo : hi;
        c = rfast ? hi : lo;
    };
#pragma unroll
    for (int u = 0; u < IT; u++) {
        int b, r, c;
        place(t + u * NT, b, r, c);
        v[u] = P[b * DT_PBLK + c * DT_PLD + r];
    }
#pragma unroll
    for (int u = 0; u < IT; u++) {
        int b, r, c;
        place(t + u * NT, b, r, c);
        const int col = 16 * J + c;
        if (b < nr || b == DT_MAXB) {
            const int row = 16 * (b == DT_MAXB ? J : J + 1 + b) + r;
            if (row < n && col < n && row >= col) L.at(row, col) = v[u];
        }
        else if (b < nbk) {
            // W(16 J + c, 16 i + r) = L^{-T} block (i, J), element (r, c)
            const int wc = 16 * (b - nr) + r;
            if (col < n && wc < n) Wv.at(col, wc) = col < wc ? T(0) : v[u];
        }
    }
}

// The tile (lower-equivalent view L, order n <= 128) factored in place, W =
// L^{-1} with zeros above its diagonal into Wv.  Returns 0 or the 1-based
// column of the first pivot that is not positive, the same in every thread;
// does nothing when *status is set (read beside the tile).
template <typename T>
__device__ int factor_diag128(const View<T> &L, const int n,
                              const View<T> &Wv, const int *status, T *sm)
{
    T *S = sm + DiagLds<T>::S, *P = sm + DiagLds<T>::P;
    int *sinfo = reinterpret_cast<int *>(sm + DiagLds<T>::INFO);
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nbk = (n + 15) / 16;
    const bool up = L.rs != 1;

    // the tile into its slots, padded with the identity; two blocks per
    // pass, all loads in flight before the first LDS store
    {
        const int e = t & 255, h = __builtin_amdgcn_readfirstlane(t >> 8);
        const int rr = up ? e >> 4 : e & 15, cc = up ? e & 15 : e >> 4;
        T x[DT_SLOTS / 2];
#pragma unroll
        for (int s = 0; s < DT_SLOTS / 2; s++) {
            constexpr auto I = [](int b) constexpr { return tri_row(b); };
            const int I0 = I(2 * s), I1 = I(2 * s + 1);
            const int bi = h ? I1 : I0;
            const int bj = h ? 2 * s + 1 - tri(I1, 0) : 2 * s - tri(I0, 0);
            x[s] = L.at(min(16 * bi + rr, n - 1), min(16 * bj + cc, n - 1));
        }
#pragma unroll
        for (int s = 0; s < DT_SLOTS / 2; s++) {
            constexpr auto I = [](int b) constexpr { return tri_row(b); };
            const int I0 = I(2 * s), I1 = I(2 * s + 1);
            const int bi = h ? I1 : I0;
            const int bj = h ? 2 * s + 1 - tri(I1, 0) : 2 * s - tri(I0, 0);
            const int r = 16 * bi + rr, c = 16 * bj + cc;
            T v = r == c ? T(1) : T(0);
            if (r < n && c < n && c <= r) v = x[s];
            S[(2 * s + h) * DT_BLK + 16 * cc + rr] = v;
        }
    }
    if (t == 0) *sinfo = seq_failed(status) ? 1 : 0;
    __syncthreads();
    if (*sinfo) return 0;

    for (int J = 0; J < nbk; J++) {
        const int nr = nbk - 1 - J;         // tile row blocks below J
        T dd[16], p[16], piv = T(1);
        const int r16 = lane & 15, b = 4 * wave + (lane >> 4);
        if (wave < 2) {
            const int rp = opaque(r16);
            const T *ds = S + tri(J, J) * DT_BLK + r16;
            const int i = b - nr;           // identity row block
            const T *ps = S + (b < nr ? tri(J + 1 + b, J)
                                      : tri(J, min(i, J))) * DT_BLK + r16;
#pragma unroll
            for (int c = 0; c < 16; c++) {
                dd[c] = ds[16 * c];
                p[c] = ps[16 * c];
            }
            if (i >= J)
#pragma unroll
                for (int c = 0; c < 16; c++)
                    p[c] = (i == J && c == rp) ? T(1) : T(0);
            Rsqrt<T> first;
            first.x = piv = row_bcast<0>(dd[0]);
            first.template step<0>();
            first.rest();
            Columns<T, 0>::run(dd, p, piv, first.y, rp);
        }
        else if (J > 0) {
            // step J - 1 beside the panel: its columns c from J + 1 on
            // (row blocks c - J .. nbk - 1 of the panel each), two blocks
            // per pass, and its stores
            const int K = J - 1, nk = nbk - 1 - K;
            int c = K + 2, bb = 1 + wave - 2;
            auto next = [&](int step) {
                bb += step;
                while (bb >= nbk && c < nbk) {
                    bb += c - K - nbk;
                    c++;
                }
            };
            auto slot_of = [&](int c_, int b_) {
                return S + (b_ < nk ? tri(K + 1 + b_, c_)
                                    : tri(c_, b_ - nk)) * DT_BLK;
            };
            next(0);
            while (c < nbk) {
                const int c0 = c, b0 = bb;
                next(DT_NT / 64 - 2);
                if (c < nbk) {
                    slot_update2<T>(slot_of(c0, b0), P + b0 * DT_PBLK,
                                    P + (c0 - K - 1) * DT_PBLK, b0 - nk == K,
                                    slot_of(c, bb), P + bb * DT_PBLK,
                                    P + (c - K - 1) * DT_PBLK, bb - nk == K);
                    next(DT_NT / 64 - 2);
                }
                else {
                    slot_update<T>(slot_of(c0, b0), P + b0 * DT_PBLK,
                                   P + (c0 - K - 1) * DT_PBLK, b0 - nk == K);
                }
            }
            store_step<T, DT_NT - 128>(L, n, Wv, sm, K, nbk,
                                       opaque(t - 128));
        }
        else {
            // zeros above the diagonal blocks of W
            for (int c = 16 + wave - 2; c < n; c += DT_NT / 64 - 2)
                for (int r = lane; r < (c & ~15); r += 64)
                    Wv.at(r, c) = T(0);
        }
        __syncthreads();                    // panel J - 1 consumed
        if (wave < 2) {
            if (b < nbk)
#pragma unroll
                for (int c = 0; c < 16; c++)
                    P[b * DT_PBLK + c * DT_PLD + r16] = p[c];
            if (wave == 0) {
                if (lane < 16) {
                    const int rw = opaque(r16);
                    T *pd = P + DT_MAXB * DT_PBLK + rw;
#pragma unroll
                    for (int c = 0; c < 16; c++) pd[c * DT_PLD] = dd[c];
                    // the diagonal itself: the correctly rounded root
                    pd[rw * DT_PLD] = sqrt(piv);
                }
                const unsigned long long bad = __ballot(!(piv > T(0)));
                if (lane == 0)
                    *sinfo = bad ? 16 * J + __ffsll(bad) : 0;
            }
        }
        __syncthreads();
        const int info = *sinfo;
        if (info) return info;
        // column J + 1: one row block per wave
        if (J + 1 < nbk && wave < nbk) {
            T *slot = S + (wave < nr ? tri(J + 1 + wave, J + 1)
                                     : tri(J + 1, wave - nr)) * DT_BLK;
            slot_update<T>(slot, P + wave * DT_PBLK, P, wave - nr == J);
        }
        __syncthreads();
    }
    // all eight waves: 2304 entries are not a multiple of 512 threads
    if (t < 384)
        store_step<T, DT_NT - 128>(L, n, Wv, sm, nbk - 1, nbk, t);
    return 0;
}

template <typename T>
__global__ __launch_bounds__(DT_NT, 4) void diag128_kernel(
    plasma_desc_t A, int upper, int k, T *inv, int *status)
{
    View<T> Wv;
    Wv.p = inv + (size_t)k * A.mb * A.mb;
    Wv.rs = 1;
    Wv.cs = A.mb;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int info = factor_diag128<T>(lower_view<T>(A, upper != 0, k, k),
                                       plasma_tile_mview(A, k), Wv, status,
                                       reinterpret_cast<T *>(smem_raw));
    if (info && threadIdx.x == 0) atomicCAS(status, 0, A.nb * k + info);
}

template <typename T>
int launch_diag128(plasma_enum_t uplo, plasma_desc_t A, int k, void *inv,
                   int *status, hipStream_t s)
{
    constexpr size_t lds = DiagLds<T>::bytes;
    if (lds > 65536) {
        static unsigned long long done = 0;     // a bit per device
        int dev = 0;
        (void)hipGetDevice(&dev);
        const unsigned long long bit = 1ull << (dev & 63);
        if (!(__atomic_load_n(&done, __ATOMIC_RELAXED) & bit)) {
            (void)hipFuncSetAttribute((const void *)diag128_kernel<T>,
                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            __atomic_fetch_or(&done, bit, __ATOMIC_RELAXED);
        }
    }
    hipLaunchKernelGGL(diag128_kernel<T>, dim3(1), dim3(DT_NT), lds, s, A,
                       uplo == PlasmaUpper, k, (T *)inv, status);
    return hipGetLastError() == hipSuccess ? 0 : PlasmaErrorInternal;
}

}  // namespace

extern "C" int plasma_diag128_ok(plasma_desc_t A)
{
    return A.mb <= 16 * DT_MAXB && A.mb == A.nb &&
           (A.precision == PlasmaRealDouble || A.precision == PlasmaRealFloat);
}

extern "C" int plasma_kern_diag128(plasma_enum_t uplo, plasma_desc_t A, int k,
                                   void *inv, int *status, hipStream_t s)
{
    if (!plasma_diag128_ok(A)) return PlasmaErrorNotSupported;
    if (A.precision == PlasmaRealDouble)
        return launch_diag128<double>(uplo, A, k, inv, status, s);
    return launch_diag128<float>(uplo, A, k, inv, status, s);
}
