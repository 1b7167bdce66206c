/* Host check of the tile geometry and the binning's bounds (p2m_dev.h):
 *  - the tiles of every nside 1..8192 and several shapes cover each ring
 *    exactly once, in sectors at most C wide and at most a quarter of the ring;
 *  - for random discs (radius 1e-7..2 rad, poles included) every pixel run of
 *    the FP64 disc query lies on a ring that disc_rings keeps and in tiles that
 *    halo_tiles lists, each once, with that ring among its rows;
 *  - disc_ring_run_chord gives the run of disc_ring_run_z, or says that the
 *    exact evaluation has to decide (counted) within a widened run;
 *  - ring_gaps counts the empty rings between rings with pixels. */
#include "p2m_dev.h"
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <set>
#include <vector>

struct H { double cosang, zz0, a, phi0; };

static long bad = 0, all_gaps = 0, asked = 0;
static void fail(const char *what, int nside, int ring, double rad)
{
    if (++bad < 10) printf("%s: nside %d ring %d rad %.3e\n", what, nside, ring, rad);
}

int main()
{
    long rings = 0, undecided = 0, tiles = 0;
    const int shapes[][2] = {{2, 4}, {3, 5}, {4, 6}, {4, 7}, {0, 6}, {1, 4}};
    for (int32_t nside = 1; nside <= 8192; nside *= 2)
        for (auto &sh : shapes) {
            const TileShape g = {nside, sh[0], sh[1]};
            int32_t next = 1;
            for (int32_t b = 0; b < n_bands(g); ++b) {
                int32_t r0, r1;
                const int32_t K = band_sectors(g, b, r0, r1);
                if (r0 != next || r1 < r0 || r1 - r0 >= (1 << g.log2r)) fail("band", nside, r0, 0);
                next = r1 + 1;
                /* every ring of the smaller maps, a band's end rings of the others */
                for (int32_t r = r0; r <= r1; r += nside <= 64 || r == r1 ? 1 : r1 - r0) {
                    int32_t npr, ks;
                    int64_t first;
                    ring_info(nside, r, npr, ks, first);
                    if (sector_start(npr, K, 0) != 0 || sector_start(npr, K, K) != npr) fail("ends", nside, r, 0);
                    for (int32_t k = 0; k < K; ++k, ++tiles) {
                        const int32_t w = sector_start(npr, K, k + 1) - sector_start(npr, K, k);
                        if (w < 0 || w > (1 << g.log2c) || 4 * w > npr) fail("width", nside, r, 0);
                    }
                }
            }
            if (next != 4 * nside) fail("cover", nside, next, 0);
        }
    std::mt19937_64 rng(77);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    for (int d = 0; d < 2000000; ++d) {
        const int32_t nside = 1 << (int)(U(rng) * 14);
        const TileShape g = {nside, shapes[d % 6][0], shapes[d % 6][1]};
        double z0 = 2.0 * U(rng) - 1.0;
        if (d % 40 == 0) z0 = d % 80 == 0 ? 1.0 : -1.0;
        if (d % 40 == 1) z0 = std::cos(1e-3 * U(rng)) * (d % 80 == 1 ? 1.0 : -1.0);
        const double ph = 2.0 * M_PI * U(rng) - M_PI, st = std::sqrt(std::max(0.0, 1.0 - z0 * z0));
        /* every third disc a few ring spacings across, the others over the whole range */
        const double rad = d >= 200000 ? (0.3 + 1.2 * U(rng)) / nside : d % 3 == 0 ? (0.2 + 4.0 * U(rng)) / nside
                                      : std::exp(std::log(1e-7) + U(rng) * (std::log(2.0) - std::log(1e-7)));
        H h;
        h.cosang = p2m_cos(rad);
        const double x0 = st * std::cos(ph), y0 = st * std::sin(ph), nrm = p2m_sqrt((x0 * x0 + y0 * y0) + z0 * z0);
        h.zz0 = z0 / nrm;
        const double xn = x0 / nrm, yn = y0 / nrm;
        h.a = xn * xn + yn * yn;
        h.phi0 = xn != 0.0 || yn != 0.0 ? p2m_atan2(yn, xn) : 0.0;
        const double s0 = p2m_sqrt(h.a), sh = p2m_sin(0.5 * rad), thr = 4.0 * (sh * sh);
        const double rl0 = p2m_asin(h.zz0);
        const double zmax = rl0 + rad >= HPX_HALFPI ? 1.0 : p2m_sin(rl0 + rad);
        const double zmin = rl0 - rad <= -HPX_HALFPI ? -1.0 : p2m_sin(rl0 - rad);
        const int32_t irmin = std::max(1, ring_num(nside, zmax) - 1), irmax = std::min(4 * nside - 1, ring_num(nside, zmin) + 1);
        const uint32_t kept = disc_rings(nside, zmax, zmin, irmin, irmax);
        const int32_t ka = kept & 0xffff, kb = kept >> 16;
        const float turn = (float)(h.phi0 / HPX_TWOPI), half = disc_half_turn(thr, s0);
        /* the listed tiles: (band, sector) -> rows */
        struct T { int32_t band, k, r0, r1; };
        std::vector<T> list;
        std::set<std::pair<int32_t, int32_t>> seen;
        if (irmax - irmin < 200 && d < 200000)
            halo_tiles(g, turn, half, kept, [&](int32_t band, int32_t k, int32_t row, int32_t n) {
                if (!seen.insert({band, k}).second) fail("twice", nside, band, rad);
                const int32_t f = (band << g.log2r) + 1 + row;
                if (row < 0 || n < 1 || row + n > (1 << g.log2r)) fail("rows", nside, f, rad);
                list.push_back({band, k, f, f + n - 1});
            });
        if (irmax - irmin < 400) {
            /* gaps over every ring of the query, as an empty ring with pixels before and after */
            std::vector<int32_t> runs;
            for (int32_t ring = irmin; ring <= irmax; ++ring) runs.push_back(ring_run_of(h, nside, ring));
            int32_t gaps = 0;
            for (size_t k = 1; k + 1 < runs.size(); ++k)
                if (runs[k] == 0 && runs[k - 1] > 0)
                    for (size_t j = k + 1; j < runs.size(); ++j) if (runs[j] > 0) { ++gaps; break; }
            const int32_t got = gaps_possible(nside, zmax, zmin, h.a, half, kept) ? ring_gaps(h, nside, kept) : 0;
            all_gaps += gaps;
            asked += gaps_possible(nside, zmax, zmin, h.a, half, kept);
            if (got != gaps) fail("gaps", nside, irmin, rad);
        }
        if (d >= 200000) continue;      /* the rest: small discs, for the gaps alone */
        for (int32_t ring = irmin; ring <= irmax; ring += 1 + (irmax - irmin) / 150) {
            int32_t npr, ks;
            int64_t first;
            ring_info(nside, ring, npr, ks, first);
            int32_t lo_e = -1, lo_c = -1;
            const int32_t np = disc_ring_run_z(h, ring2z(nside, ring), npr, ks, lo_e);
            ++rings;
            double zr, sth, off, den;
            ring_zsth(nside, ring, zr, sth);
            ring_phi_param(nside, ring, off, den);
            const double kphi = HPX_HALFPI / den, ik = den * (2.0 / HPX_PI);
            double ipc = __builtin_rint(h.phi0 * ik - off);
            if (ipc < 0.0) ipc += (double)npr;
            if (ipc >= (double)npr) ipc -= (double)npr;
            double xc = 0.5 * ((ipc + off) * kphi - h.phi0);
            xc -= HPX_PI * __builtin_rint(xc * (1.0 / HPX_PI));
            const double dz = zr - h.zz0, ds = sth - s0;
            int32_t np_max;
            const int32_t nc = disc_ring_run_chord(thr, dz * dz + ds * ds, (float)((4.0 * sth) * s0),
                                                   (float)(2e-15 / (sth * sth)), (float)xc, (float)(2.0 * ik), (int32_t)ipc,
                                                   npr, lo_c, np_max);
            if (nc < 0) {
                ++undecided;
                /* the run is among the np_max pixels from lo */
                if (np > 0) {
                    const int32_t rel = ((lo_e - lo_c) % npr + npr) % npr;
                    if (np_max < npr && rel + np > np_max) fail("run outside the widened run", nside, ring, rad);
                }
            } else if (nc != np || (np > 0 && lo_c != lo_e)) fail("chord run", nside, ring, rad);
            if (np == 0) continue;
            if (ring < ka || ring > kb) { fail("ring dropped", nside, ring, rad); continue; }
            if (irmax - irmin >= 200) continue;
            /* both ends and a few pixels between */
            int32_t r0, r1;
            const int32_t band = (ring - 1) >> g.log2r, K = band_sectors(g, band, r0, r1);
            for (int j = 0; j < 9; ++j) {
                const int32_t ip = (int32_t)((lo_e + (int64_t)(np - 1) * j / 8) % npr);
                int32_t k = (int32_t)(((int64_t)ip * K) / npr);
                while (sector_start(npr, K, k + 1) <= ip) ++k;
                while (sector_start(npr, K, k) > ip) --k;
                bool ok = false;
                if (seen.count({band, k}))
                    for (auto &t : list) ok |= t.band == band && t.k == k && ring >= t.r0 && ring <= t.r1;
                if (!ok) { fail("tile missed", nside, ring, rad); break; }
            }
        }
    }
    printf("checked %ld tiles, %ld rings, %ld undecided, %ld gaps (%ld discs asked), %ld mismatches\n", tiles, rings, undecided, all_gaps, asked, bad);
    return bad != 0;
}
