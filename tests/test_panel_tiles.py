"""CPU test of the polynomial by which a kernel finds the tiles of a column
(csrc/kernels/paneltiles.h) against the descriptor's own tile arithmetic: every
storage type, both triangles, views, ragged orders.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r'''
#include <stdio.h>
#include "plasma.h"
#include "paneltiles.h"

static int check(plasma_desc_t A, int upper)
{
    int bad = 0;
    for (int k = 0; k < A.mt - 1; k++) {
        const plasma_panel_tiles_t t = plasma_panel_tiles(A, upper, k);
        for (int m = k + 1; m < A.mt; m++) {
            const int last = m == A.mt - 1;
            const size_t o = upper ? plasma_tile_offset(A, k, m)
                                   : plasma_tile_offset(A, m, k);
            bad += plasma_panel_tile(&t, m - k - 1) != o ||
                   (last ? t.ld_last : t.ld) !=
                       plasma_tile_mmain(A, upper ? k : m) ||
                   (last ? t.rows_last : A.mb) != plasma_tile_mview(A, m);
        }
        bad += t.ntiles != A.mt - k - 1;
    }
    return bad;
}

int main(void)
{
    int bad = 0, count = 0;
    for (int mb = 3; mb <= 16; mb += 13)
        for (int n = 1; n < 9 * mb; n++)
            for (int before = 0; before < 2; before++)
                for (int after = 0; after < 3; after++) {
                    /* a view that starts `before` tiles into the matrix and
                     * ends before its last rows */
                    const int at = before * mb, N = at + n + after * 2;
                    plasma_desc_t A;
                    plasma_desc_general_init(PlasmaRealFloat, NULL, mb, mb, N,
                                             N, at, at, n, n, &A);
                    bad += check(A, 0) + check(A, 1);
                    plasma_desc_triangular_init(PlasmaRealFloat, PlasmaLower,
                                                NULL, mb, mb, N, N, at, at, n,
                                                n, &A);
                    bad += check(A, 0);
                    plasma_desc_triangular_init(PlasmaRealFloat, PlasmaUpper,
                                                NULL, mb, mb, N, N, at, at, n,
                                                n, &A);
                    bad += check(A, 1);
                    plasma_desc_general_band_init(PlasmaRealFloat,
                                                  PlasmaGeneral, NULL, mb, mb,
                                                  N, N, at, at, n, n, n - 1,
                                                  n - 1, &A);
                    bad += check(A, 0) + check(A, 1);
                    count++;
                }
    printf("%d %d\n", count, bad);
    return 0;
}
'''


def test_offsets(tmp_path):
    import plasma_amd as pa
    src, exe = tmp_path / "t.c", tmp_path / "t"
    src.write_text(SOURCE)
    lib = os.path.dirname(pa.LIB_PATH)
    subprocess.run(["gcc", "-std=c11", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "plasma_amd", "csrc", "kernels"),
                    str(src), "-o", str(exe), "-L", lib, "-lplasma_amd",
                    "-Wl,-rpath," + lib], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True,
                         text=True).stdout.split()
    assert int(out[0]) > 900 and int(out[1]) == 0, out
