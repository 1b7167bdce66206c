/* Host check of the pixels that the tile painters store (p2m_dev.h): for
 * every nside 1..8192 and every tile size they take, the tiles of tile_shape
 * as k_tile_desc describes and stage_row stages them.
 *  - A row's pixels first + sector_start(k) .. + width - 1 lie inside their
 *    ring and the map, start where the row of the sector before ended, and the
 *    rings follow one another from 0 to 12 nside^2: every map pixel is stored
 *    by exactly one tile.
 *  - A row is at most 2^log2c pixels wide and a tile at most 16 rows, so that
 *    the in-tile pixel (row << log2c) + column is below 2^log2w and the
 *    wave's offsets fit the 16 bits they are kept in.
 *  - The tiles are numbered band by band below 2^24. */
#include "p2m_dev.h"
#include <cstdio>

int main()
{
    long bad = 0, rows = 0;
    for (int32_t nside = 1; nside <= 8192; nside *= 2)
        for (int log2w = 6; log2w <= 11; ++log2w) {
            const TileShape g = tile_shape(nside, log2w);
            const int64_t npix = 12LL * nside * nside;
            int64_t next = 0, tiles = 0;
            bool ok = g.nside == nside && g.log2r >= 0 && g.log2r <= 4 && g.log2c >= 2 && g.log2c <= 7 && g.log2r + g.log2c <= log2w;
            int32_t ring = 1;
            for (int32_t b = 0; b < n_bands(g); ++b) {
                int32_t r0, r1;
                const int32_t K = band_sectors(g, b, r0, r1);
                ok &= r0 == ring && r1 >= r0 && r1 - r0 < (1 << g.log2r) && r1 <= 4 * nside - 1;
                ring = r1 + 1;
                tiles += K;
                for (int32_t r = r0; r <= r1; ++r) {
                    int32_t npr, ks;
                    int64_t first;
                    ring_info(nside, r, npr, ks, first);
                    ok &= first == next;
                    int32_t at = 0;
                    for (int32_t k = 0; k < K; ++k, ++rows) {
                        const int32_t i0 = sector_start(npr, K, k), w = sector_start(npr, K, k + 1) - i0;
                        ok &= i0 == at && w >= 0 && w <= (1 << g.log2c) && i0 + w <= npr && first + i0 + w <= npix;
                        at += w;
                    }
                    ok &= at == npr;
                    next = first + npr;
                }
            }
            ok &= ring == 4 * nside && next == npix && tiles < (1 << 24);
            if (!ok && ++bad < 10) printf("nside %d tile %d\n", nside, 1 << log2w);
        }
    printf("checked %ld rows, %ld mismatches\n", rows, bad);
    return bad != 0;
}
