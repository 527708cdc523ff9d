"""CPU tests of the batched driver's host side (compute/batched.c), compiled
against a stand-in for the HIP calls and kernels it uses: the class launches run
on two streams, and a failing fork or join of these streams is an error, never
kernels on arrays still being copied or an info read too early.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "plasma_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

STAND_IN = r'''
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "internal.h"

/* which call fails: its name and, from 0, its number among those of the name */
static const char *fail_name;
static int fail_number, calls[3];
static hipError_t result(int k, const char *name)
{
    const int number = calls[k]++;
    printf("%s ", name);
    return strcmp(name, fail_name) == 0 && number == fail_number
               ? hipErrorUnknown : hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags)
{
    *e = (hipEvent_t)malloc(1);
    return result(0, "create");
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    return result(1, "record");
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned flags)
{
    return result(2, "wait");
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    free(e);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k,
                          hipStream_t t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    printf("sync%d ", (int)(size_t)s);
    return hipSuccess;
}

static plasma_context_t context;
static double A[1], B[1];
plasma_context_t *plasma_context_self(void) { return &context; }
int plasma_is_device_ptr(const void *p) { return p == A || p == B; }
void *plasma_dev_alloc(size_t bytes) { return malloc(bytes); }
void plasma_dev_free(void *p) { free(p); }
int plasma_hip_check(hipError_t e, const char *what) { return e != 0; }
int plasma_vbatched16_ok(int nrhs) { return nrhs <= 16; }
size_t plasma_vbatched16_bytes(plasma_enum_t p, int c, int n, int cus)
{
    return 8;
}
int plasma_kern_vbatched16(plasma_enum_t p, int up, int batch,
                           const int cls[2], const int *n, void *a,
                           const size_t *aoff, void *const W[3], int nrhs,
                           void *b, const size_t *boff, int *info,
                           const int *order, int *ticket, int cus,
                           hipStream_t const s[3])
{
    printf("launch ");
    memset(info, 0, batch * sizeof(int));
    return 0;
}
size_t plasma_kern_vbatched_lds(plasma_enum_t p) { return 65536; }
size_t plasma_kern_vbatched_wslab(plasma_enum_t p) { return 8; }
int plasma_kern_vbatched_posv(plasma_enum_t p, int up, int batch,
                              const int *n, void *a, const size_t *aoff,
                              void *W, int nrhs, void *b, const size_t *boff,
                              int *info, const int *order, int *ticket,
                              int grid, hipStream_t s)
{
    return 0;
}
int plasma_kern_vbatched_order(const int *n, int batch, int *order, int *c,
                               hipStream_t s)
{
    return 0;
}
int plasma_noalloc_setup(int device) { return 0; }
int plasma_noalloc_regions(int device, plasma_noalloc_t *r) { return 0; }

int main(int argc, char **argv)
{
    fail_name = argv[1];
    fail_number = atoi(argv[2]);
    context.num_cus = 256;
    context.stream = (hipStream_t)0;
    context.panel_stream = (hipStream_t)1;
    int n[3] = {300, 20, 200}, info[3] = {7, 7, 7};
    size_t off[3] = {0, 0, 0};
    const int rc = plasma_dposv_vbatched(PlasmaLower, 3, n, A, off, 1, B, off,
                                         info);
    printf("return %d\n", rc);
    return 0;
}
'''


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("batched")
    src = d / "stand_in.c"
    src.write_text(STAND_IN)
    exe = d / "driver"
    subprocess.run(["gcc", "-std=c11", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROCM, "include"),
                    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    "-I", os.path.join(CSRC, "kernels"), str(src),
                    os.path.join(CSRC, "compute", "batched.c"),
                    "-o", str(exe)], check=True)

    def run(name, number):
        return subprocess.run([str(exe), name, str(number)], check=True,
                              capture_output=True, text=True).stdout.split()
    return run


INTERNAL = "-106"                       # PlasmaErrorInternal


def test_fork_and_join(driver):
    assert driver("none", 0) == ["create", "create", "record", "wait",
                                 "launch", "record", "wait", "sync0",
                                 "sync1", "sync0", "return", "0"]


@pytest.mark.parametrize("name,number", [("create", 0), ("create", 1),
                                         ("record", 0), ("wait", 0)])
def test_no_launch_without_the_fork(driver, name, number):
    out = driver(name, number)
    assert "launch" not in out
    assert out[-4:] == ["sync1", "sync0", "return", INTERNAL]


@pytest.mark.parametrize("name", ["record", "wait"])
def test_a_failing_join_is_an_error(driver, name):
    out = driver(name, 1)
    assert out.count("launch") == 1
    assert out[-4:] == ["sync1", "sync0", "return", INTERNAL]
