// zview.hip.h -- complex elements and strided complex windows of tiles and
// buffers, shared by the complex (Hermitian) kernels.
#pragma once

#include "common.hip.h"
#include "plasma_kernels.h"

namespace {

template <typename R> struct alignas(2 * sizeof(R)) cx {
    R re, im;
};

template <typename R> __device__ __forceinline__ cx<R> czero()
{
    return cx<R>{R(0), R(0)};
}

// a * b and a * conj(b)
template <typename R>
__device__ __forceinline__ cx<R> cmul(cx<R> a, cx<R> b)
{
    return cx<R>{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename R>
__device__ __forceinline__ cx<R> cmulc(cx<R> a, cx<R> b)
{
    return cx<R>{a.re * b.re + a.im * b.im, a.im * b.re - a.re * b.im};
}

// A strided complex window: element (r, c) at p[r rs + c cs], conjugated
// on read and write when `conj`.  With `herm` the window is the Hermitian
// matrix whose lower triangle (r >= c) is stored: r < c reads the conjugate
// of (c, r) and the diagonal reads as real (LAPACK ignores the imaginary
// part of a Hermitian diagonal).
template <typename R> struct CView {
    cx<R> *p;
    int rs, cs;
    int conj;
    int herm;

    __device__ __forceinline__ cx<R> raw(int r, int c) const
    {
        cx<R> v = p[(ptrdiff_t)r * rs + (ptrdiff_t)c * cs];
        if (conj) v.im = -v.im;
        return v;
    }
    __device__ __forceinline__ cx<R> get(int r, int c) const
    {
        if (herm) {
            if (r == c) {
                cx<R> v = raw(r, r);
                v.im = R(0);
                return v;
            }
            if (r < c) {
                cx<R> v = raw(c, r);
                v.im = -v.im;
                return v;
            }
        }
        return raw(r, c);
    }
    __device__ __forceinline__ void put(int r, int c, cx<R> v) const
    {
        if (conj) v.im = -v.im;
        p[(ptrdiff_t)r * rs + (ptrdiff_t)c * cs] = v;
    }
    // the window moved to start at (r, c) (plain windows only)
    __device__ __forceinline__ CView at(int r, int c) const
    {
        CView v = *this;
        v.p = p + (ptrdiff_t)r * rs + (ptrdiff_t)c * cs;
        return v;
    }
};

// Conjugate transpose of a window (a Hermitian window is its own).
template <typename R>
__device__ __forceinline__ CView<R> herm_of(CView<R> v)
{
    if (v.herm) return v;
    CView<R> h = v;
    h.rs = v.cs;
    h.cs = v.rs;
    h.conj = !v.conj;
    return h;
}

// Tile (m, n), m >= n, of the lower-equivalent factor L.
template <typename R>
__device__ __forceinline__ CView<R> lower_cview(const plasma_desc_t &A,
                                                bool upper, int m, int n)
{
    CView<R> v;
    v.herm = 0;
    if (!upper) {
        v.p = (cx<R> *)plasma_tile_addr(A, m, n);
        v.rs = 1;
        v.cs = plasma_tile_mmain(A, m);
        v.conj = 0;
    }
    else {
        v.p = (cx<R> *)plasma_tile_addr(A, n, m);
        v.rs = plasma_tile_mmain(A, n);
        v.cs = 1;
        v.conj = 1;
    }
    return v;
}

template <typename R>
__device__ __forceinline__ CView<R> tile_cview(const plasma_desc_t &A, int m,
                                               int n)
{
    CView<R> v;
    v.p = (cx<R> *)plasma_tile_addr(A, m, n);
    v.rs = 1;
    v.cs = plasma_tile_mmain(A, m);
    v.conj = 0;
    v.herm = 0;
    return v;
}

// A column-major buffer with leading dimension ld.
template <typename R>
__device__ __forceinline__ CView<R> buf_cview(cx<R> *p, int ld)
{
    CView<R> v;
    v.p = p;
    v.rs = 1;
    v.cs = ld;
    v.conj = 0;
    v.herm = 0;
    return v;
}

}  // namespace
