// panel16.hip.h -- one wave eliminates 16 columns of a Cholesky panel in
// registers: every 16-lane row of the wave holds the 16 rows of the diagonal
// block (dd, the same in each row) and 16 panel rows (p), one row of each per
// lane.  No LDS and no barrier.
#pragma once

#include "common.hip.h"

namespace p16 {

// lane C's value of each 16-lane row, in every lane of the row
template <int C> __device__ __forceinline__ double row_bcast(double x)
{
    return __longlong_as_double(__builtin_amdgcn_update_dpp(
        0LL, __double_as_longlong(x), 0x150 + C, 0xf, 0xf, true));
}
template <int C> __device__ __forceinline__ float row_bcast(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(
        0, __float_as_int(x), 0x150 + C, 0xf, 0xf, true));
}

// x, hidden from the compiler: it would otherwise compute addresses and lane
// masks of every phase before the step loop and spill them
__device__ __forceinline__ int opaque(int x)
{
    asm("" : "+v"(x));
    return x;
}

// 1 / sqrt(x) of a pivot, one step at a time (Rsqrt::step<S>, S = 0 ..
// steps - 1), so that the steps can be placed between the eliminations of
// the column before: 0 for +inf, NaN for x < 0 or NaN.
//
// FP32: the FP64 estimate (measured on 10^6 FP32 arguments: 0.88 2^-24 at
// most), rounded.  The FP32 estimate takes a subnormal pivot for zero (infinite,
// and NaN once corrected); with one correction step its rms error is the same
// (0.50 and 0.49 2^-24), at twice the instructions.  A correction in FP64
// as well (0.46) made the FP32 batched solver 1.2 % and sposv n = 6000 1 %
// slower without a smaller error in either.
//
// FP64: the estimate y0 and one correction with e = 1 - x y0^2 to third order,
// (1 - e)^{-1/2}.  The clamp keeps x y0 = 0 (not NaN) for an infinite pivot.
template <typename T> struct Rsqrt;
template <> struct Rsqrt<float> {
    static constexpr int steps = 2;
    float x, y;
    double z;
    template <int S> __device__ __forceinline__ void step()
    {
        if constexpr (S == 0) z = __builtin_amdgcn_rsq((double)x);
        if constexpr (S == 1) y = (float)z;
    }
    __device__ __forceinline__ void rest() { step<1>(); }
};
template <> struct Rsqrt<double> {
    static constexpr int steps = 5;
    double x, y, t, e, q;
    template <int S> __device__ __forceinline__ void step()
    {
        if constexpr (S == 0) {
            y = __builtin_amdgcn_rsq(x);
            t = __builtin_fmin(x, 0x1.fffffffffffffp+1023);
        }
        if constexpr (S == 1) t = t * y;
        if constexpr (S == 2) e = __builtin_fma(-t, y, 1.0);
        if constexpr (S == 3) {
            q = __builtin_fma(e, 0.375, 0.5);
            e = y * e;
        }
        if constexpr (S == 4) y = __builtin_fma(e, q, y);
    }
    __device__ __forceinline__ void rest()
    {
        step<1>();
        step<2>();
        step<3>();
        step<4>();
    }
};

// v -= bcast_C(l) * m in one instruction: lane C of each 16-lane row of l,
// the DPP operand of a multiply-add.  A DPP source must not have been written
// in the two instructions before (s_nop 1 opens every group: the compiler
// does not look for that hazard inside inline assembly).
#define P16_FMAC64(d, l, m, c)                                                 \
    "v_fmac_f64_dpp " d ", " l ", -" m " row_newbcast:" c                     \
    " row_mask:0xf bank_mask:0xf\n\t"
#define P16_FMAC32(d, l, m, c)                                                 \
    "v_fmac_f32_dpp " d ", " l ", -" m " row_newbcast:" c                     \
    " row_mask:0xf bank_mask:0xf\n\t"

// columns C and C + 1 of the block's rows (d) and of the panel rows (p)
template <int C>
__device__ __forceinline__ void elim2(double &d0, double &p0, double &d1,
                                      double &p1, double dj, double pj)
{
    asm volatile("s_nop 1\n\t"
                 P16_FMAC64("%0", "%4", "%4", "%6")
                 P16_FMAC64("%1", "%4", "%5", "%6")
                 P16_FMAC64("%2", "%4", "%4", "%7")
                 P16_FMAC64("%3", "%4", "%5", "%7")
                 : "+v"(d0), "+v"(p0), "+v"(d1), "+v"(p1)
                 : "v"(dj), "v"(pj), "i"(C), "i"(C + 1));
}
template <int C>
__device__ __forceinline__ void elim2(float &d0, float &p0, float &d1,
                                      float &p1, float dj, float pj)
{
    asm volatile("s_nop 1\n\t"
                 P16_FMAC32("%0", "%4", "%4", "%6")
                 P16_FMAC32("%1", "%4", "%5", "%6")
                 P16_FMAC32("%2", "%4", "%4", "%7")
                 P16_FMAC32("%3", "%4", "%5", "%7")
                 : "+v"(d0), "+v"(p0), "+v"(d1), "+v"(p1)
                 : "v"(dj), "v"(pj), "i"(C), "i"(C + 1));
}
// columns C .. C + 3
#define P16_ELIM4(T, F)                                                        \
    template <int C>                                                          \
    __device__ __forceinline__ void elim4(T (&d)[16], T (&p)[16], T dj, T pj) \
    {                                                                         \
        asm volatile("s_nop 1\n\t"                                            \
                     F("%0", "%8", "%8", "%10") F("%1", "%8", "%9", "%10")    \
                     F("%2", "%8", "%8", "%11") F("%3", "%8", "%9", "%11")    \
                     F("%4", "%8", "%8", "%12") F("%5", "%8", "%9", "%12")    \
                     F("%6", "%8", "%8", "%13") F("%7", "%8", "%9", "%13")    \
                     : "+v"(d[C]), "+v"(p[C]), "+v"(d[C + 1]),                \
                       "+v"(p[C + 1]), "+v"(d[C + 2]), "+v"(p[C + 2]),        \
                       "+v"(d[C + 3]), "+v"(p[C + 3])                         \
                     : "v"(dj), "v"(pj), "i"(C), "i"(C + 1), "i"(C + 2),      \
                       "i"(C + 3));                                           \
    }
P16_ELIM4(double, P16_FMAC64)
P16_ELIM4(float, P16_FMAC32)
// column C alone, and its pivot x = bcast_C(d) for the next step
template <int C>
__device__ __forceinline__ void elim1(double &d, double &p, double &x,
                                      double dj, double pj)
{
    asm volatile("s_nop 1\n\t"
                 P16_FMAC64("%0", "%3", "%3", "%5")
                 P16_FMAC64("%1", "%3", "%4", "%5")
                 "s_nop 1\n\t"
                 "v_mov_b64_dpp %2, %0 row_newbcast:%5 row_mask:0xf "
                 "bank_mask:0xf\n\t"
                 : "+v"(d), "+v"(p), "=&v"(x)
                 : "v"(dj), "v"(pj), "i"(C));
}
template <int C>
__device__ __forceinline__ void elim1(float &d, float &p, float &x, float dj,
                                      float pj)
{
    asm volatile("s_nop 1\n\t"
                 P16_FMAC32("%0", "%3", "%3", "%5")
                 P16_FMAC32("%1", "%3", "%4", "%5")
                 "s_nop 1\n\t"
                 "v_mov_b32_dpp %2, %0 row_newbcast:%5 row_mask:0xf "
                 "bank_mask:0xf\n\t"
                 : "+v"(d), "+v"(p), "=&v"(x)
                 : "v"(dj), "v"(pj), "i"(C));
}

// Columns C.. eliminated four at a time, one step of the next pivot's 1/sqrt
// after each group.
template <typename T, int C, int S> struct Elim {
    static __device__ __forceinline__ void run(T (&dd)[16], T (&p)[16], T dj,
                                               T pj, Rsqrt<T> &next)
    {
        constexpr int N = C + 3 < 16 ? 4 : C + 1 < 16 ? 2 : 1;
        if constexpr (C + 3 < 16) elim4<C>(dd, p, dj, pj);
        else if constexpr (C + 1 < 16)
            elim2<C>(dd[C], p[C], dd[C + 1], p[C + 1], dj, pj);
        else if constexpr (C == 15) {
            T x;
            elim1<C>(dd[C], p[C], x, dj, pj);
        }
        if constexpr (S < Rsqrt<T>::steps) {
            next.template step<S>();
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (C < 16 || S < Rsqrt<T>::steps)
            Elim<T, C + N, S + 1>::run(dd, p, dj, pj, next);
    }
};

// The columns J.. of a panel: dd the diagonal block's rows, p the panel
// rows, one of each per lane; y: 1 / sqrt of pivot J; piv: lane r % 16 == j
// keeps pivot j.  The next pivot's chain starts as soon as its column is
// updated.
template <typename T, int J> struct Columns {
    static __device__ __forceinline__ void run(T (&dd)[16], T (&p)[16],
                                               T &piv, T y, int r)
    {
        const T dj = dd[J] * y, pj = p[J] * y;
        dd[J] = dj;
        p[J] = pj;
        if constexpr (J + 1 < 16) {
            Rsqrt<T> next;
            elim1<J + 1>(dd[J + 1], p[J + 1], next.x, dj, pj);
            next.template step<0>();
            __builtin_amdgcn_sched_barrier(0);
            Elim<T, J + 2, 1>::run(dd, p, dj, pj, next);
            piv = (r == J + 1) ? next.x : piv;
            Columns<T, J + 1>::run(dd, p, piv, next.y, r);
        }
    }
};

}  // namespace p16
