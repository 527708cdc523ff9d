// substpanel.hip -- the FP32 panel solve P(m) = A(m,k) L_kk^{-T} for tiles of
// order <= 128, by substitution over 16-column blocks (the trsm tasks of the
// reference's pzpotrf.c:47-57; upper: :90-99).
//
// Why not the product A(m,k) W_kk^T with the inverse of the whole tile: its
// rounding grows with the condition of the tile, substitution by blocks with
// that of the 16 x 16 diagonal blocks.  On a kernel (RBF) matrix, where a tile
// is about as ill-conditioned as the matrix, the product loses digits of the
// factor: 1-D points, n = 512, condition 2e6, backward error of the factor
// 4.0e-7 against 1.4e-7 here, and the refinement of a mixed solve takes 23
// steps against 5; at 1e7 the FP32 factorization breaks down, here it takes 11.
// With 32-column blocks the counts are the same there, but 16 to 29 against 6
// or 7 for 2-D points (n = 2048, condition 7e6).
//
// One workgroup per 64 rows of a panel tile, 16 rows per wave, in two phases:
//   1. every wave loads 9 of the 36 lower 16 x 16 blocks of L_kk (the diagonal
//      ones: W_kk's, whose diagonal blocks are the inverses of L's) and its own
//      rows of A(m,k), all loads in flight; the blocks go to LDS in the order in
//      which the MFMA operand reads them;
//   2. after the one barrier each wave solves its rows alone.  It forms
//      X^T (panel columns on the MFMA rows):
//          T   = A_J^T - sum_{I < J} L_JI X_I^T,     X_J^T = W_JJ T.
//      The result of v_mfma_f32_16x16x4_f32 has k value 4 g + q of row block
//      in element q of lane group g, so element q of all lanes is the operand
//      of a later product over k = {q, 4 + q, 8 + q, 12 + q}: X never leaves
//      the registers.
// Bound by latency: one round trip to memory for the blocks, which another XCD
// has just written, and 144 dependent matrix instructions (1.9 us) per wave.
// Measured per launch: 6.6 us (n = 6000, upper) and 6.5 us (n = 4000, lower);
// the product with W_kk took 7.0 and 6.2 us, substitution by 32 columns with a
// barrier per step about 20 us.  With the descriptor's tile arithmetic in the
// kernel the same took 9.2 us: 1200 instructions, 4 us, before the barrier.
#include "common.hip.h"
#include "directgemm.hip.h"
#include "paneltiles.h"
#include "plasma_kernels.h"

namespace {

constexpr int SP_NT = 256;
constexpr int SP_ROWS = 64;             // rows of a panel tile per workgroup
constexpr int SP_MAXB = 8;              // 16-column blocks of a tile

__host__ __device__ constexpr int sp_tri(int i, int j)
{
    return i * (i + 1) / 2 + j;
}

// What the kernel needs to know of the descriptor, worked out on the host
// (paneltiles.h).
struct Panel {
    const float *A;             // the matrix
    const float *L, *W;         // L_kk, W_kk
    plasma_panel_tiles_t tiles; // A(m,k), m > k
    float *P;                   // solved panel of tile k + 1
    ptrdiff_t pstep;            // from one tile's panel to the next
    int ldl, ldp, nb;           // nb: tile order
    const int *status;
};

// BLKS: 16-column blocks of a tile at most (4 or 8).  FULL: a tile of order
// 16 BLKS; else loads are clamped and what lies outside becomes zero.  VEC: 16-
// byte loads of four columns (upper storage, FULL, aligned).
template <bool UPPER, int BLKS, bool FULL, bool VEC>
__global__ __launch_bounds__(SP_NT, 2) void panel_subst_kernel(Panel g)
{
    // fragment order: lane's row lane % 16, columns 4 (lane / 16) + 0 .. 3
    __shared__ float4_t sB[sp_tri(BLKS, 0) * 64];
    __shared__ int s_stop;
    const int t = threadIdx.x, lane = t & 63, l16 = lane & 15;
    const int g4 = 4 * (lane >> 4);
    const int wave = dg::uni(t >> 6);
    const int m = blockIdx.x;
    const bool last = m == g.tiles.ntiles - 1;
    const int nb = FULL ? 16 * BLKS : g.nb;
    const int mv = last ? g.tiles.rows_last : nb;
    const int row0 = blockIdx.y * SP_ROWS;
    if (row0 >= mv) return;
    // read beside the blocks: set, nothing is solved
    const int stop = t == 0 ? __atomic_load_n(g.status, __ATOMIC_RELAXED) : 0;
    const int row = row0 + 16 * wave + l16;
    const DG_GLOBAL float *ap =
        (const DG_GLOBAL float *)(g.A + plasma_panel_tile(&g.tiles, m));
    const int lda = last ? g.tiles.ld_last : g.tiles.ld;

    // Rows r0 + lane % 16, columns c0 + 4 (lane / 16) + 0 .. 3 of a window of
    // `rows` rows and nb columns; element (r, c) at p[r + c ld] (UNIT) or
    // p[r ld + c].  off: the lane's offsets for r0 = c0 = 0 (FULL).
    struct Off {
        unsigned o[4];
    };
    auto offsets = [&](bool unit, int r, int ld) {
        Off f;
#pragma unroll
        for (int q = 0; q < 4; q++)
            f.o[q] = 4u * (unsigned)(unit ? r + (g4 + q) * ld
                                          : r * ld + g4 + q);
        return f;
    };
    auto fetch = [&](const DG_GLOBAL float *p, bool unit, int ld, int r0,
                     int rmax, int c0, const Off &f) {
        float4_t x;
        if constexpr (FULL) {
            const DG_GLOBAL char *b = (const DG_GLOBAL char *)dg::scalar(
                p + (unit ? r0 + (ptrdiff_t)c0 * ld
                          : (ptrdiff_t)r0 * ld + c0));
            if (VEC && !unit) {
                x = *(const DG_GLOBAL float4_t *)(b + f.o[0]);
            }
            else {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    x[q] = *(const DG_GLOBAL float *)(b + f.o[q]);
            }
        }
        else {
            const int r = min(r0 + l16, rmax - 1);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int c = min(c0 + g4 + q, nb - 1);
                x[q] = p[unit ? r + (ptrdiff_t)c * ld
                              : (ptrdiff_t)r * ld + c];
            }
        }
        return x;
    };

    // A wave's blocks (J, I), without a branch: the diagonal ones of block rows
    // wave (and wave + 4), and of the pairs of diagonals J - I = d and BLKS - d,
    // which have BLKS blocks together, those numbered wave (and wave + 4).
    constexpr int ND = BLKS / 4, NB = BLKS == 8 ? 7 : 2;
    auto block = [&](int u, int &J, int &I) {
        if constexpr (BLKS == 8) {
            const int d = u / 2 + 1;            // u == 6: d = 4, four blocks
            const bool up = u % 2 == 0 || wave < 4 - d;
            I = u % 2 == 0 ? wave : up ? wave + 4 : wave + d - 4;
            J = up ? I + d : wave + 4;
        }
        else if (u == 0) {
            I = wave < 3 ? wave : 0;
            J = wave < 3 ? wave + 1 : 3;
        }
        else {
            I = wave % 2;                       // (2, 0) and (3, 1), twice
            J = I + 2;
        }
    };
    float4_t dia[ND], b[NB], x[BLKS];
    {
        const DG_GLOBAL float *lp = (const DG_GLOBAL float *)g.L;
        const DG_GLOBAL float *wp = (const DG_GLOBAL float *)g.W;
        const Off lo = offsets(!UPPER, l16, g.ldl);
        const Off wo = offsets(true, l16, g.ldp);
        // rows past the tile's read its last one, their results stay here
        const Off ao = offsets(!UPPER, min(row, mv - 1), lda);
#pragma unroll
        for (int u = 0; u < ND; u++) {
            const int J = wave + 4 * u;
            dia[u] = fetch(wp, true, g.ldp, 16 * J, nb, 16 * J, wo);
        }
#pragma unroll
        for (int u = 0; u < NB; u++) {
            int J, I;
            block(u, J, I);
            b[u] = fetch(lp, !UPPER, g.ldl, 16 * J, nb, 16 * I, lo);
        }
#pragma unroll
        for (int J = 0; J < BLKS; J++)
            x[J] = fetch(ap, !UPPER, lda, FULL ? 0 : row - l16, mv, 16 * J,
                         ao);
    }
    auto put = [&](int J, int I, float4_t v) {
        if (!FULL)
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (16 * J + l16 >= nb || 16 * I + g4 + q >= nb) v[q] = 0;
        sB[sp_tri(J, I) * 64 + lane] = v;
    };
    if (t == 0) s_stop = stop;
#pragma unroll
    for (int u = 0; u < ND; u++) put(wave + 4 * u, wave + 4 * u, dia[u]);
#pragma unroll
    for (int u = 0; u < NB; u++) {
        int J, I;
        block(u, J, I);
        put(J, I, b[u]);
    }
    __syncthreads();
    if (s_stop || row0 + 16 * wave >= mv) return;

#pragma unroll
    for (int J = 0; J < BLKS; J++) {
        float4_t s = {0, 0, 0, 0}, y = {0, 0, 0, 0}, d;
#pragma unroll
        for (int I = 0; I < J; I++) {
            d = sB[sp_tri(J, I) * 64 + lane];
#pragma unroll
            for (int q = 0; q < 4; q++)
                s = Mfma<float>::mma(d[q], x[I][q], s);
        }
        d = sB[sp_tri(J, J) * 64 + lane];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const bool in = FULL || 16 * J + g4 + q < nb;
            y = Mfma<float>::mma(d[q], in ? x[J][q] - s[q] : 0.0f, y);
        }
        x[J] = y;
    }
    if (row >= mv) return;
    DG_GLOBAL float *P = (DG_GLOBAL float *)(g.P + m * g.pstep);
    const Off po = offsets(true, row, g.ldp);
#pragma unroll
    for (int J = 0; J < BLKS; J++) {
        DG_GLOBAL char *c =
            (DG_GLOBAL char *)dg::scalar(P + (ptrdiff_t)16 * J * g.ldp);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (FULL || 16 * J + g4 + q < nb)
                *(DG_GLOBAL float *)(c + po.o[q]) = x[J][q];
    }
}

template <bool UPPER, int BLKS>
const void *kernel_of(bool full, bool vec)
{
    if (!full) return (const void *)panel_subst_kernel<UPPER, BLKS, false,
                                                       false>;
    if (UPPER && vec)
        return (const void *)panel_subst_kernel<UPPER, BLKS, true, UPPER>;
    return (const void *)panel_subst_kernel<UPPER, BLKS, true, false>;
}

}  // namespace

extern "C" int plasma_panel_subst_ok(plasma_desc_t A)
{
    return A.precision == PlasmaRealFloat && A.mb == A.nb &&
           A.mb <= 16 * SP_MAXB;
}

extern "C" int plasma_kern_panel_subst(plasma_enum_t uplo, plasma_desc_t A,
                                       int k, const void *inv, void *panel,
                                       int pbase, int pcols, int pcol,
                                       const int *status, hipStream_t s)
{
    if (!plasma_panel_subst_ok(A)) return PlasmaErrorNotSupported;
    if (A.mt - k - 1 <= 0) return 0;
    const bool up = uplo == PlasmaUpper, small = A.mb <= 64;
    const size_t mb = A.mb;
    Panel g;
    g.A = (const float *)A.matrix;
    g.tiles = plasma_panel_tiles(A, up, k);
    g.L = (const float *)plasma_tile_addr(A, k, k);
    g.W = (const float *)inv + k * mb * mb;
    g.P = (float *)panel + (size_t)(k - pbase) * mb * pcols +
          (size_t)pcol * mb;
    g.pstep = (ptrdiff_t)mb * pcols;
    g.ldl = plasma_tile_mmain(A, k);
    g.ldp = A.mb;
    g.nb = A.mb;                        // tile k is not the last one
    g.status = status;
    const plasma_panel_tiles_t &t = g.tiles;
    const bool full = A.mb == (small ? 64 : 128);
    const bool vec = ((uintptr_t)g.A | (uintptr_t)g.L) % 16 == 0 &&
                     (t.first | t.last) % 4 == 0 &&
                     (t.step | t.step2) % 4 == 0 &&
                     (g.ldl | t.ld | t.ld_last) % 4 == 0;
    const void *fn = up ? (small ? kernel_of<true, 4>(full, vec)
                                 : kernel_of<true, 8>(full, vec))
                        : (small ? kernel_of<false, 4>(full, vec)
                                 : kernel_of<false, 8>(full, vec));
    const dim3 grid(t.ntiles, (A.mb + SP_ROWS - 1) / SP_ROWS);
    void *args[] = {&g};
    return hipLaunchKernel(fn, grid, dim3(SP_NT), args, 0, s) == hipSuccess
               ? 0 : PlasmaErrorInternal;
}
