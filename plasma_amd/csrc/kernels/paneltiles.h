/*
 * paneltiles.h -- where the tiles (m, k), m > k, of the lower-equivalent
 * factor lie, as a polynomial in m.
 *
 * A kernel that works the address of its tile out of the descriptor spends
 * more instructions on that than on what precedes its first load; from these
 * numbers, computed once on the host, it takes a few.
 */
#ifndef PLASMA_PANELTILES_H
#define PLASMA_PANELTILES_H

#include <stddef.h>
#include "plasma_descriptor.h"

typedef struct {
    size_t first, last;     /* element offsets of tiles k + 1 and mt - 1 */
    ptrdiff_t step, step2;  /* first and second difference of the offsets of
                             * tiles k + 1 .. mt - 2, which are whole: of degree
                             * 1 in m, or 2 where upper tiles are packed column
                             * by column */
    int ntiles;             /* mt - k - 1 */
    int ld, ld_last;        /* leading dimensions */
    int rows_last;          /* rows of the last tile */
} plasma_panel_tiles_t;

/* Offset of tile k + 1 + m. */
static inline PLASMA_HD size_t plasma_panel_tile(const plasma_panel_tiles_t *t,
                                                 int m)
{
    if (m == t->ntiles - 1)
        return t->last;
    return t->first + (size_t)(m * t->step +
                               m * (ptrdiff_t)(m - 1) / 2 * t->step2);
}

/* upper: the factor is stored as U = L^T, tile (m, k) of it at (k, m). */
static inline plasma_panel_tiles_t plasma_panel_tiles(plasma_desc_t A,
                                                      int upper, int k)
{
    plasma_panel_tiles_t t;
    size_t o[4];
    t.ntiles = A.mt - k - 1;
    for (int i = 0; i < 4; i++) {
        const int m = k + 1 + (i < t.ntiles ? i : t.ntiles - 1);
        o[i] = upper ? plasma_tile_offset(A, k, m)
                     : plasma_tile_offset(A, m, k);
    }
    t.first = o[0];
    t.last = upper ? plasma_tile_offset(A, k, A.mt - 1)
                   : plasma_tile_offset(A, A.mt - 1, k);
    t.step = t.ntiles > 2 ? (ptrdiff_t)(o[1] - o[0]) : 0;
    t.step2 = t.ntiles > 3 ? (ptrdiff_t)(o[2] - o[1]) - t.step : 0;
    t.ld = plasma_tile_mmain(A, upper ? k : k + 1);
    t.ld_last = plasma_tile_mmain(A, upper ? k : A.mt - 1);
    t.rows_last = plasma_tile_mview(A, A.mt - 1);
    return t;
}

#endif
