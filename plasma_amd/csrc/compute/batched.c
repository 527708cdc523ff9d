/*
 * batched.c -- SPD solves of many independent systems of uneven order
 * (plasma_{d,s}posv_vbatched, plasma_{d,s}potrf_vbatched): a persistent
 * launch per class of orders, or one for all with many right-hand sides.  No
 * counterpart in the reference, which factors one matrix per call
 * (compute/zposv.c); each system follows the same algorithm as the
 * reference's tile factorization of a single tile (core_zpotrf.c) and its
 * triangular solves, with LAPACK's info per system.
 *
 * Layout: system i of order n[i] (0 <= n[i] <= 512) is stored column major
 * at A + aoff[i] with leading dimension n[i]; its right-hand sides at
 * B + boff[i], n[i] x nrhs, leading dimension n[i].  A and B are device
 * memory; n, aoff, boff and info may be host or device arrays.
 */
#include <stdlib.h>
#include <string.h>

#include "internal.h"

#define VBATCH_NMAX 512

/* Argument checks of the batched drivers, in the order of their codes:
 * returns -i for an illegal argument i, 1 for the quick return (batch 0),
 * 0 to proceed. */
static int vbatched_args(plasma_enum_t uplo, int batch, const int *n,
                         const void *A, const size_t *aoff, int nrhs,
                         const void *B, const size_t *boff, const int *info)
{
    if (uplo != PlasmaUpper && uplo != PlasmaLower) {
        plasma_error("illegal value of uplo");
        return -1;
    }
    if (batch < 0) {
        plasma_error("illegal value of batch");
        return -2;
    }
    if (batch == 0)
        return 1;
    if (n == NULL) {
        plasma_error("NULL n");
        return -3;
    }
    if (A == NULL || !plasma_is_device_ptr(A)) {
        plasma_error("A must be device memory");
        return -4;
    }
    if (aoff == NULL) {
        plasma_error("NULL aoff");
        return -5;
    }
    if (nrhs < 0) {
        plasma_error("illegal value of nrhs");
        return -6;
    }
    if (nrhs > 0 && (B == NULL || !plasma_is_device_ptr(B))) {
        plasma_error("B must be device memory");
        return -7;
    }
    if (nrhs > 0 && boff == NULL) {
        plasma_error("NULL boff");
        return -8;
    }
    if (info == NULL) {
        plasma_error("NULL info");
        return -9;
    }
    return 0;
}

/* Workgroups of the persistent grid: as many as the LDS lets the CUs hold,
 * at most one per system. */
static int vbatched_grid(plasma_context_t *ctx, plasma_enum_t precision,
                         int batch)
{
    const size_t lds = plasma_kern_vbatched_lds(precision);
    int per_cu = (int)((160 * 1024) / lds);
    if (per_cu < 1)
        per_cu = 1;
    int grid = ctx->num_cus * per_cu;
    return grid > batch ? batch : grid;
}

/* Class of a system's order: 0 above 256, 1 above 128, 2 */
static int order_class(int n)
{
    return n > 256 ? 0 : n > 128 ? 1 : 2;
}

/* The class launches of up to 16 right-hand sides: the largest class on the
 * main stream, the others beside it on the panel stream (their workgroups
 * fill the CUs its last systems leave idle), joined on return. */
static int vbatched16(plasma_context_t *ctx, plasma_enum_t precision,
                      int upper, int batch, const int count[3], const int *n,
                      void *A, const size_t *aoff, void *W, int nrhs, void *B,
                      const size_t *boff, int *info, const int *order,
                      int *ticket)
{
    const int cls[2] = {count[0], count[0] + count[1]};
    void *w[3];
    char *p = W;
    for (int k = 0; k < 3; k++) {
        w[k] = p;
        if (p != NULL && count[k] > 0)
            p += plasma_vbatched16_bytes(precision, k, count[k],
                                         ctx->num_cus);
    }
    const int fork = (count[0] > 0) && (count[1] + count[2] > 0);
    hipStream_t s0 = ctx->stream, s1 = fork ? ctx->panel_stream : s0;
    hipStream_t const s[3] = {s0, s1, s1};
    hipEvent_t ev[2] = {NULL, NULL};
    int err = 0;
    if (fork) {
        for (int k = 0; k < 2 && !err; k++)
            err = plasma_hip_check(hipEventCreateWithFlags(
                                       &ev[k], hipEventDisableTiming),
                                   "hipEventCreate");
        /* the panel stream's launches read what the main stream is still
         * copying: without the fork they must not start */
        if (!err)
            err = plasma_hip_check(hipEventRecord(ev[0], s0),
                                   "hipEventRecord") ||
                  plasma_hip_check(hipStreamWaitEvent(s1, ev[0], 0),
                                   "hipStreamWaitEvent");
    }
    if (!err) {
        err = plasma_kern_vbatched16(precision, upper, batch, cls, n, A, aoff,
                                     w, nrhs, B, boff, info, order, ticket,
                                     ctx->num_cus, s);
        /* without the join the main stream's copy of info would come too
         * early: an error, which the caller returns after waiting for both
         * streams */
        if (fork && (plasma_hip_check(hipEventRecord(ev[1], s1),
                                      "hipEventRecord") ||
                     plasma_hip_check(hipStreamWaitEvent(s0, ev[1], 0),
                                      "hipStreamWaitEvent")))
            err = 1;
    }
    for (int k = 0; k < 2; k++)
        if (ev[k] != NULL)
            hipEventDestroy(ev[k]);
    return err ? PlasmaErrorInternal : 0;
}

/* Systems by order, largest first, equal orders by index. */
static void order_systems(const int *n, int batch, int *order)
{
    int start[VBATCH_NMAX + 2] = {0};
    for (int i = 0; i < batch; i++)
        start[VBATCH_NMAX - n[i] + 1]++;
    for (int v = 0; v <= VBATCH_NMAX; v++)
        start[v + 1] += start[v];
    for (int i = 0; i < batch; i++)
        order[start[VBATCH_NMAX - n[i]]++] = i;
}

static int vbatched(plasma_enum_t precision, plasma_enum_t uplo, int batch,
                    const int *n, void *A, const size_t *aoff, int nrhs,
                    void *B, const size_t *boff, int *info)
{
    plasma_context_t *ctx = plasma_context_self();
    if (ctx == NULL) {
        plasma_error("PLASMA not initialized");
        return PlasmaErrorNotInitialized;
    }
    const int args = vbatched_args(uplo, batch, n, A, aoff, nrhs, B, boff,
                                   info);
    if (args != 0)
        return args < 0 ? args : PlasmaSuccess;

    /* Host view of n (the argument check and the order), and the host
     * arrays that go to the device, packed for one copy: aoff, boff, n,
     * order, tickets.  A copy on another stream than the context's could
     * overwrite a pool block that earlier kernels still read. */
    const size_t nbytes = (size_t)batch * sizeof(int);
    const size_t obytes = (size_t)batch * sizeof(size_t);
    const int dev_n = plasma_is_device_ptr(n);
    const int dev_off = plasma_is_device_ptr(aoff);
    const int dev_boff = nrhs > 0 && plasma_is_device_ptr(boff);
    const int dev_info = plasma_is_device_ptr(info);
    const size_t mbytes = 2 * obytes + 2 * nbytes + 3 * sizeof(int);
    int retval = PlasmaSuccess;
    char *meta = NULL;
    void *W = NULL, *dinfo = NULL;
    char *host = malloc(mbytes);
    if (host == NULL) {
        retval = PlasmaErrorOutOfMemory;
        goto done;
    }
    int *hn = (int *)(host + 2 * obytes), *hord = hn + batch;
    if (dev_n) {
        /* a caller's device array may have been written by work queued on
         * the library's streams (non-blocking, so the copy below would not
         * wait for it) */
        hipStreamSynchronize(ctx->panel_stream);
        hipStreamSynchronize(ctx->stream);
        if (plasma_hip_check(hipMemcpy(hn, n, nbytes, hipMemcpyDefault),
                             "hipMemcpy(n)")) {
            retval = PlasmaErrorInternal;
            goto done;
        }
    }
    else {
        memcpy(hn, n, nbytes);
    }
    int count[3] = {0, 0, 0};
    for (int i = 0; i < batch; i++) {
        if (hn[i] < 0 || hn[i] > VBATCH_NMAX) {
            plasma_error("illegal order of a system");
            retval = -3;
            goto done;
        }
        count[order_class(hn[i])]++;
    }
    order_systems(hn, batch, hord);
    if (!dev_off)
        memcpy(host, aoff, obytes);
    if (nrhs > 0 && !dev_boff)
        memcpy(host + obytes, boff, obytes);
    memset(hord + batch, 0, 3 * sizeof(int));

    /* resident grids, each workgroup with its own slab of W */
    const int grid = vbatched_grid(ctx, precision, batch);
    const int classes = plasma_vbatched16_ok(nrhs);
    size_t wbytes = (size_t)grid * plasma_kern_vbatched_wslab(precision);
    if (classes) {
        wbytes = 0;
        for (int k = 0; k < 3; k++)
            wbytes += plasma_vbatched16_bytes(precision, k, count[k],
                                              ctx->num_cus);
    }
    W = plasma_dev_alloc(wbytes);
    meta = plasma_dev_alloc(mbytes);
    if (!dev_info)
        dinfo = plasma_dev_alloc(nbytes);
    if (W == NULL || meta == NULL || (!dev_info && dinfo == NULL)) {
        retval = PlasmaErrorOutOfMemory;
        goto done;
    }
    hipStream_t s = ctx->stream;
    if (plasma_hip_check(hipMemcpyAsync(meta, host, mbytes,
                                        hipMemcpyHostToDevice, s),
                         "hipMemcpyAsync")) {
        retval = PlasmaErrorInternal;
        goto done;
    }
    const size_t *doff = dev_off ? aoff : (const size_t *)meta;
    const size_t *dboff = nrhs <= 0  ? NULL
                          : dev_boff ? boff
                                     : (const size_t *)(meta + obytes);
    const int *dn = dev_n ? n : (const int *)(meta + 2 * obytes);
    int *dord = (int *)(meta + 2 * obytes + nbytes);
    int *dticket = dord + batch;
    int *di = dev_info ? info : dinfo;
    if (classes
            ? vbatched16(ctx, precision, uplo == PlasmaUpper, batch, count, dn,
                         A, doff, W, nrhs, B, dboff, di, dord, dticket)
            : plasma_kern_vbatched_posv(precision, uplo == PlasmaUpper, batch,
                                        dn, A, doff, W, nrhs, B, dboff, di,
                                        dord, dticket, grid, s)) {
        retval = PlasmaErrorInternal;
        goto done;
    }
    if (!dev_info &&
        plasma_hip_check(hipMemcpyAsync(info, dinfo, nbytes,
                                        hipMemcpyDeviceToHost, s),
                         "hipMemcpy(info)")) {
        retval = PlasmaErrorInternal;
        goto done;
    }
    if (plasma_hip_check(hipStreamSynchronize(s), "hipStreamSynchronize"))
        retval = PlasmaErrorInternal;

done:
    /* the host arrays below are freed only after the copies that read them
     * (also on the error paths) */
    hipStreamSynchronize(ctx->panel_stream);
    hipStreamSynchronize(ctx->stream);
    plasma_dev_free(dinfo);
    plasma_dev_free(meta);
    plasma_dev_free(W);
    free(host);
    return retval;
}

int plasma_dposv_vbatched(plasma_enum_t uplo, int batch, const int *n,
                          double *A, const size_t *aoff, int nrhs, double *B,
                          const size_t *boff, int *info)
{
    return vbatched(PlasmaRealDouble, uplo, batch, n, A, aoff, nrhs, B, boff,
                    info);
}

int plasma_sposv_vbatched(plasma_enum_t uplo, int batch, const int *n,
                          float *A, const size_t *aoff, int nrhs, float *B,
                          const size_t *boff, int *info)
{
    return vbatched(PlasmaRealFloat, uplo, batch, n, A, aoff, nrhs, B, boff,
                    info);
}

int plasma_dpotrf_vbatched(plasma_enum_t uplo, int batch, const int *n,
                           double *A, const size_t *aoff, int *info)
{
    return vbatched(PlasmaRealDouble, uplo, batch, n, A, aoff, 0, NULL, NULL,
                    info);
}

int plasma_spotrf_vbatched(plasma_enum_t uplo, int batch, const int *n,
                           float *A, const size_t *aoff, int *info)
{
    return vbatched(PlasmaRealFloat, uplo, batch, n, A, aoff, 0, NULL, NULL,
                    info);
}

/* The allocation-free variant: every device buffer beyond the caller's
 * inputs and outputs is a region of the per-device scratch array of
 * kernels/noalloc.hip (its address looked up once per device), and no host
 * buffer is allocated either.  Host metadata arrays are copied into the
 * scratch; the systems are ordered on the device. */
int plasma_dposv_vbatched_noalloc(plasma_enum_t uplo, int batch,
                                  const int *n, double *A,
                                  const size_t *aoff, int nrhs, double *B,
                                  const size_t *boff, int *info)
{
    plasma_context_t *ctx = plasma_context_self();
    if (ctx == NULL) {
        plasma_error("PLASMA not initialized");
        return PlasmaErrorNotInitialized;
    }
    const int args = vbatched_args(uplo, batch, n, A, aoff, nrhs, B, boff,
                                   info);
    if (args != 0)
        return args < 0 ? args : PlasmaSuccess;
    if (batch > PLASMA_VBATCH_NOALLOC_MAX) {
        plasma_error("batch above PLASMA_VBATCH_NOALLOC_MAX, the number of "
                     "systems the allocation-free scratch holds");
        return -2;
    }
    plasma_noalloc_t r;
    if (plasma_noalloc_setup(ctx->device) != 0 ||
        plasma_noalloc_regions(ctx->device, &r) != 0 ||
        plasma_kern_vbatched_wslab(PlasmaRealDouble) > r.wslab_bytes) {
        plasma_error("allocation-free scratch unavailable");
        return PlasmaErrorInternal;
    }
    hipStream_t s = ctx->stream;
    const size_t nbytes = (size_t)batch * sizeof(int);
    const size_t obytes = (size_t)batch * sizeof(size_t);
    const int host_n = !plasma_is_device_ptr(n);
    const int *dn = n;
    int count[3] = {0, 0, 0};
    if (host_n) {
        /* checked here, like plasma_dposv_vbatched, before any launch */
        for (int i = 0; i < batch; i++)
            if (n[i] < 0 || n[i] > VBATCH_NMAX) {
                plasma_error("illegal order of a system");
                return -3;
            }
        for (int i = 0; i < batch; i++)
            count[order_class(n[i])]++;
        if (plasma_hip_check(hipMemcpyAsync(r.n, n, nbytes,
                                            hipMemcpyHostToDevice, s),
                             "hipMemcpyAsync(n)"))
            return PlasmaErrorInternal;
        dn = r.n;
    }
    const size_t *daoff = aoff, *dboff = boff;
    if (!plasma_is_device_ptr(aoff)) {
        if (plasma_hip_check(hipMemcpyAsync(r.aoff, aoff, obytes,
                                            hipMemcpyHostToDevice, s),
                             "hipMemcpyAsync(aoff)"))
            return PlasmaErrorInternal;
        daoff = r.aoff;
    }
    if (nrhs > 0 && !plasma_is_device_ptr(boff)) {
        if (plasma_hip_check(hipMemcpyAsync(r.boff, boff, obytes,
                                            hipMemcpyHostToDevice, s),
                             "hipMemcpyAsync(boff)"))
            return PlasmaErrorInternal;
        dboff = r.boff;
    }
    const int host_info = !plasma_is_device_ptr(info);
    int *dinfo = host_info ? r.info : info;
    if (plasma_kern_vbatched_order(dn, batch, r.order, r.ctrl, s) != 0)
        return PlasmaErrorInternal;
    if (!host_n) {
        /* orders in device memory: checked by the order kernel */
        int ctrl[4] = {0, 0, 0, 0};
        if (plasma_hip_check(hipMemcpyAsync(ctrl, r.ctrl, sizeof(ctrl),
                                            hipMemcpyDeviceToHost, s),
                             "hipMemcpyAsync(flag)") ||
            plasma_hip_check(hipStreamSynchronize(s), "hipStreamSynchronize"))
            return PlasmaErrorInternal;
        if (ctrl[1] != 0) {
            plasma_error("illegal order of a system");
            return -3;
        }
        count[0] = ctrl[2];
        count[1] = ctrl[3] - ctrl[2];
        count[2] = batch - ctrl[3];
    }
    /* the class launches, when the slab area holds their workspace (they
     * run one after the other and share it); a workgroup's results do not
     * depend on the launch that holds it */
    size_t wmax = 0;
    for (int k = 0; k < 3; k++) {
        const size_t w = plasma_vbatched16_bytes(PlasmaRealDouble, k, count[k],
                                                 ctx->num_cus);
        if (w > wmax)
            wmax = w;
    }
    if (plasma_vbatched16_ok(nrhs) &&
        wmax <= r.wslab_bytes * (size_t)r.grid_max) {
        const int cls[2] = {count[0], count[0] + count[1]};
        void *const w[3] = {r.W, r.W, r.W};
        hipStream_t const ss[3] = {s, s, s};
        if (plasma_kern_vbatched16(PlasmaRealDouble, uplo == PlasmaUpper,
                                   batch, cls, dn, A, daoff, w, nrhs, B,
                                   dboff, dinfo, r.order, r.ctrl + 4,
                                   ctx->num_cus, ss) != 0)
            return PlasmaErrorInternal;
        goto copy_info;
    }
    int grid = vbatched_grid(ctx, PlasmaRealDouble, batch);
    if (grid > r.grid_max)
        grid = r.grid_max;
    if (plasma_kern_vbatched_posv(PlasmaRealDouble, uplo == PlasmaUpper,
                                  batch, dn, A, daoff, r.W, nrhs, B, dboff,
                                  dinfo, r.order, r.ctrl, grid, s) != 0)
        return PlasmaErrorInternal;
copy_info:
    if (host_info &&
        plasma_hip_check(hipMemcpyAsync(info, r.info, nbytes,
                                        hipMemcpyDeviceToHost, s),
                         "hipMemcpyAsync(info)"))
        return PlasmaErrorInternal;
    return plasma_hip_check(hipStreamSynchronize(s), "hipStreamSynchronize")
               ? PlasmaErrorInternal : PlasmaSuccess;
}
