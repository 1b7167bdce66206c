/*
 * p2m_dev.h -- device-side data layout and FP64 routines of the painter.
 *
 * Every FP64 routine here reproduces the arithmetic of the reference path
 * operation for operation (same operands, same association, same elementary
 * functions from p2m_math.h), so pixel membership, profile-table cells and
 * FP64 contributions agree bit for bit with a faithful CPU evaluation.
 * Reference: src/pks2map_src/{pks2map,haloproject,maptable,cosmology}.f90 and
 * the vendored HEALPix 3.10 (src/modules/External/pix_tools.F90,
 * pixel_routines.F90).
 */
#ifndef P2M_DEV_H
#define P2M_DEV_H

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "p2m_math.h"

#define P2M_MAXMAPS 6
#define P2M_DEV __device__ static inline

/* healpix_types.F90:65-73 */
#define HPX_PI      3.141592653589793238462643383279502884197
#define HPX_HALFPI  1.570796326794896619231321691639751442099
#define HPX_TWOPI   6.283185307179586476925286766559005768394
#define HPX_TWOTHIRD 0.6666666666666666666666666666666666666666
/* cosmology.f90:8-9: double parameter from a real(4) literal */
#define COSMO_PI ((double)3.14159265359f)

/* Distance tables (cosmology.f90:40-43), FP64, built on the host. */
struct CosmoDev {
    const double *rofz;
    const double *zofr;
    double drofz, dzofr, rofz_min, zofr_min;
    int32_t nrofz, nzofr;
    double omegam, omegal, rho_0, rhocrit_0, mypi;
};

/* Profile-table grid shared by all map slots (maptable.f90:9-21, 166-168). */
struct TabGeom {
    int32_t nchit, nmht, nrt;
    double chimint, chimaxt, mhmint, mhmaxt, rmint, rmaxt;
    double drt, dchit, dmht;
    double lr0, lc0, lm0;        /* log of the lower bounds */
};

/* One painted halo after decode: the per-halo constants of both painters
 * and of interpolate_table.  Struct of doubles first for alignment. */
struct HaloRec {
    double hx, hy, hz;       /* hpvec1 = (z,y,x)/chi (haloproject.f90:51-53) */
    double dtheta;           /* rmax*asin(rh/chi) (haloproject.f90:47) */
    double zz0, phi0, a;     /* discphirange_at_z: z0, atan2(y0,x0), x0^2+y0^2 */
    double cosang;           /* cos(radius) */
    double s0;               /* sqrt(a): sin of the centre colatitude */
    double thr;              /* (2 sin(dtheta/2))^2: chord^2 of the disc edge */
    double chi_r;            /* rofz(z) of interpolate_table (maptable.f90:184) */
    double fc, fm;           /* per-halo table fractions (maptable.f90:201-202) */
    double vh;               /* velocity factor (1 for tSZ) */
    double th, ph;           /* flat sky: asin(x/chi), asin(y/chi) (haloproject.f90:105-106) */
    int64_t cat;             /* catalogue index */
    int32_t ichi, imh;       /* per-halo table cells (maptable.f90:197-198) */
    int32_t irmin, irmax;    /* ring range of query_disc */
    int32_t chi_out;         /* chi > chimaxt: every value is 0 */
    int32_t flat;            /* 1 if the flat-sky painter covers this halo */
    int32_t jmin, jmax, kmin, kmax;  /* flat-sky index box (haloproject.f90:124-128) */
};

/* The fields of a painted halo that the FP32 tile painter stages per
 * (halo, ring) segment, packed into one 64-B line. */
struct __attribute__((aligned(64))) TileHalo {
    double zz0, s0, phi0, thr;   /* as in HaloRec */
    float thr_hi;                /* outer edge of the deferral band: thr (1 + CHORD_BAND) */
    float chi2;                  /* (float)(chi_r * chi_r) */
    float w00, w10, w01, w11;    /* weights of the table cell's corners times the velocity factor, from
                                    the table fractions rounded to float; 0 when chi > chimaxt */
    int32_t colbase;             /* nrt * ((imh - 1) + nmht * (ichi - 1)); 0 when chi > chimaxt */
    uint32_t pad;
};

/* Half-width of the band around the disc edge, relative in chord^2, that the
 * FP32 painter leaves to the FP64 decision. */
#define CHORD_BAND 4e-6

/* What the binning needs of a painted halo: its centre's azimuth and the
 * disc's azimuth half-width, both in turns, and the rings the disc itself
 * reaches (disc_rings), first | last << 16 (no ring: first > last), with
 * the top bit set if it may have a ring gap. */
struct PairHalo {
    float turn, half;
    uint32_t rings;
};
#define RINGS_ASK_GAPS 0x80000000u

/* ------------------------------------------------------------ cosmology */
P2M_DEV double tab_lookup(const double *t, int n, double tmin, double dt, double x)
{
    if (x != x) return x;
    double u = (x - tmin) / dt + 1.0;
    if (u < 1.0) return t[0];
    if (u >= (double)n) return t[n - 1];
    int itab = (int)u;
    double fint = ((x - (double)(itab - 1) * dt) - tmin) / dt;
    return (1.0 - fint) * t[itab - 1] + fint * t[itab];
}

P2M_DEV double cube(double x) { return (x * x) * x; }

/* cosmology.f90:185-195 */
P2M_DEV double rhocrit_z(const CosmoDev &c, double z)
{
    double z3 = cube(1.0 + z);
    return (c.rhocrit_0 * (c.omegam * z3 + c.omegal)) / z3;
}

/* cosmology.f90:199-214 */
P2M_DEV double deltacrit_z(const CosmoDev &c, double z)
{
    double z3 = cube(1.0 + z);
    double omegaz = (c.omegam * z3) / ((c.omegam * z3 + 1.0) - c.omegam);
    double x = omegaz - 1.0;
    return (18.0 * (COSMO_PI * COSMO_PI) + 82.0 * x) - 39.0 * (x * x);
}

/* ------------------------------------------------------------ HEALPix */
/* ring_num, pix_tools.F90:490-533 */
P2M_HD int32_t ring_num(int32_t nside, double z)
{
    int32_t iring = (int32_t)p2m_nint((double)nside * (2.0 - 1.5 * z));
    if (z > HPX_TWOTHIRD) {
        iring = (int32_t)p2m_nint((double)nside * p2m_sqrt(3.0 * (1.0 - z)));
        if (iring == 0) iring = 1;
    }
    if (z < -HPX_TWOTHIRD) {
        iring = (int32_t)p2m_nint((double)nside * p2m_sqrt(3.0 * (1.0 + z)));
        if (iring == 0) iring = 1;
        iring = 4 * nside - iring;
    }
    return iring;
}

/* ring2z, pix_tools.F90:535-560 */
P2M_HD double ring2z(int32_t nside, int32_t ir)
{
    double fn = (double)nside;
    if (ir < nside) {
        double tmp = (double)ir;
        return 1.0 - (tmp * tmp) / ((3.0 * fn) * fn);
    } else if (ir < 3 * nside) {
        return ((double)(2 * nside - ir) * 2.0) / (3.0 * fn);
    }
    double tmp = (double)(4 * nside - ir);
    return -1.0 + (tmp * tmp) / ((3.0 * fn) * fn);
}

/* pixels_per_ring, pix_tools.F90:802-836: npr, kshift, first pixel of ring */
P2M_HD void ring_info(int32_t nside, int32_t ring, int32_t &npr, int32_t &kshift, int64_t &first)
{
    int32_t m = nside < ring ? nside : ring;
    if (4 * nside - ring < m) m = 4 * nside - ring;
    npr = 4 * m;
    kshift = (ring + 1) & 1;
    if (nside == 1) kshift = 1 - kshift;
    if (npr < 4 * nside) kshift = 1;
    int64_t npnorth;
    if (ring <= nside) {
        npnorth = (int64_t)ring * (ring + 1LL) * 2LL;
    } else if (ring <= 3 * nside) {
        npnorth = (int64_t)nside * (nside + 1LL) * 2LL + 4LL * nside * (int64_t)(ring - nside);
    } else {
        int64_t irs = 4LL * nside - ring - 1;
        npnorth = 12LL * nside * nside - irs * (irs + 1LL) * 2LL;
    }
    first = npnorth - npr;
}

/* Ring tiles: ring `ring` is cut into ceil(npr / W) tiles of W = 2^log2w
 * consecutive RING pixels, the last one narrower.  Tile `col` starts at
 * in-ring pixel ip0 = col W, holds `width` pixels, and its first map pixel is
 * first + ip0 (first: the ring's first pixel).  Host checks of the ring
 * geometry use them; the painters' tiles are bands of rings by sectors, below. */
P2M_HD int32_t ring_tiles(int32_t nside, int32_t ring, int32_t log2w)
{
    int32_t npr, kshift;
    int64_t first;
    ring_info(nside, ring, npr, kshift, first);
    return (npr + (1 << log2w) - 1) >> log2w;
}

P2M_HD void tile_span(int32_t nside, int32_t ring, int32_t col, int32_t log2w, int64_t &first, int32_t &ip0,
                      int32_t &width)
{
    int32_t npr, kshift;
    ring_info(nside, ring, npr, kshift, first);
    ip0 = col << log2w;
    width = npr - ip0 < (1 << log2w) ? npr - ip0 : (1 << log2w);
}

/* ------------------------------------------------------------ tiles */
/* The map is painted in tiles of R = 2^log2r consecutive rings (a band; the
 * last one may hold fewer) by one sector of azimuth.  A band's rings are
 * each cut into the same number K of sectors, sector k of a ring of npr
 * pixels being [floor(k npr / K), floor((k + 1) npr / K)): K is large
 * enough that no sector is wider than C = 2^log2c pixels, nor (K >= 4, npr
 * a multiple of 4) than a quarter of its ring.  Tiles are numbered sector
 * by sector, band by band. */
struct TileShape {
    int32_t nside, log2r, log2c;
};

/* Rows and columns of a tile of up to 2^log2w pixels: at most 16 rings, 64
 * pixels along each at the default 1024.  A map of few tiles (nside 128 and
 * below at that size) takes fewer rings per tile, so that there are tiles for
 * the CUs. */
P2M_HD TileShape tile_shape(int32_t nside, int log2w)
{
    TileShape g = {nside, log2w / 2 - 1 < 4 ? log2w / 2 - 1 : 4, 0};
    g.log2c = log2w - g.log2r;
    while (g.log2r > 0 && (12LL * nside * nside) >> (g.log2r + g.log2c) < 2048) --g.log2r;
    return g;
}

P2M_HD int32_t n_bands(const TileShape &g) { return ((4 * g.nside - 1) + (1 << g.log2r) - 1) >> g.log2r; }

/* first and last ring of band `band` and its number of sectors */
P2M_HD int32_t band_sectors(const TileShape &g, int32_t band, int32_t &r0, int32_t &r1)
{
    r0 = (band << g.log2r) + 1;
    r1 = r0 + (1 << g.log2r) - 1;
    if (r1 > 4 * g.nside - 1) r1 = 4 * g.nside - 1;
    /* the longest ring of the band: 4 min(nside, the larger distance to a pole of its ends) */
    int32_t m = r1 < 4 * g.nside - r0 ? r1 : 4 * g.nside - r0;
    if (m > g.nside) m = g.nside;
    const int32_t k = (4 * m + (1 << g.log2c) - 1) >> g.log2c;
    return k < 4 ? 4 : k;
}

/* k npr < 2^31: K is at most 4 or npr / 2^log2c rounded up, npr at most 32768 */
P2M_HD int32_t sector_start(int32_t npr, int32_t K, int32_t k) { return (int32_t)(((uint32_t)k * (uint32_t)npr) / (uint32_t)K); }

/* Rings whose circle meets the disc, within the ring range [irmin, irmax] of
 * query_disc (which adds a ring on either side): lat0 -+ dtheta as sines,
 * 1 and -1 where a pole is inside.  The ring coordinate of a height is the
 * one that ring_num rounds; it is taken 1e-4 of a ring wider, which is far
 * above its rounding.  first > last if the disc lies between two rings. */
P2M_HD double ring_coord(int32_t nside, double z)
{
    if (z > HPX_TWOTHIRD) return (double)nside * p2m_sqrt(3.0 * (1.0 - z));
    if (z < -HPX_TWOTHIRD) return 4.0 * (double)nside - (double)nside * p2m_sqrt(3.0 * (1.0 + z));
    return (double)nside * (2.0 - 1.5 * z);
}

P2M_HD uint32_t disc_rings(int32_t nside, double ztop, double zbot, int32_t irmin, int32_t irmax)
{
    int32_t a = (int32_t)p2m_ceil(ring_coord(nside, ztop) - 1e-4);
    int32_t b = (int32_t)p2m_floor(ring_coord(nside, zbot) + 1e-4);
    if (a < irmin) a = irmin;
    if (b > irmax) b = irmax;
    if (a > b) return 1u;        /* first 1, last 0 */
    return (uint32_t)a | ((uint32_t)b << 16);
}

/* Azimuth half-width of a disc in turns, from its edge's chord^2 thr and the
 * sine s0 of its centre's colatitude: sin(dphi) = sin(dtheta) / s0 where the
 * disc holds no pole and is smaller than a hemisphere, else half a turn.
 * FP32, widened by more than its error (asin's slope is below 8 for
 * arguments up to 0.99). */
P2M_HD float disc_half_turn(double thr, double s0)
{
    const float c2 = (float)thr, s = (float)s0;
    const float sd = sqrtf(c2 * (1.0f - 0.25f * c2));          /* sin(dtheta) below a right angle */
    if (!(c2 < 1.9f) || !(sd < 0.99f * s)) return 0.5f;
    return asinf(sd / s) * (1.00001f / 6.2831853f) + 1e-6f;
}

/* The tiles of a band that a halo's disc may reach: n of its K sectors from
 * k0 (past the last one comes the first), `rows` rows from `row`. */
struct BandTiles { int32_t K, k0, n, row, rows; };
P2M_HD BandTiles band_tiles(const TileShape &g, int32_t band, float turn, float half, int32_t ra, int32_t rb)
{
    int32_t r0, r1;
    const int32_t K = band_sectors(g, band, r0, r1);
    const int32_t first = ra > r0 ? ra : r0, last = rb < r1 ? rb : r1;
    int32_t n = K, k0 = 0;
    if (half < 0.5f) {
        /* a pixel ip of a ring lies at (ip + off) / npr turns, off 0 or
         * 1/2, in the sector ceil((ip + 1) K / npr) - 1: not below the
         * floor of its turn times K, at most a pixel's K / npr above */
        const int32_t m0 = r0 < 4 * g.nside - r1 ? r0 : 4 * g.nside - r1;
        const int32_t nmin = 4 * (m0 < g.nside ? m0 : g.nside);
        const float fk = (float)K;
        const double lo = ((double)turn - (double)half) * fk, hi = ((double)turn + (double)half) * fk + (double)(fk / (float)nmin);
        k0 = (int32_t)p2m_floor(lo);
        n = (int32_t)p2m_floor(hi + 1e-6) - k0 + 1;
        if (n >= K) { n = K; k0 = 0; }
        else if (k0 < 0) k0 += K;
    }
    return {K, k0, n, first - r0, last - first + 1};
}

/* the bands [b0, b1] of the rings of a PairHalo; none: b0 > b1 */
P2M_HD void halo_bands(const TileShape &g, uint32_t rings, int32_t &ra, int32_t &rb, int32_t &b0, int32_t &b1)
{
    ra = (int32_t)(rings & 0xffffu);
    rb = (int32_t)((rings >> 16) & 0x7fffu);
    b0 = (ra - 1) >> g.log2r;
    b1 = ra > rb ? b0 - 1 : (rb - 1) >> g.log2r;
}

/* The tiles a halo's disc may reach, in band order: f(band, sector, first
 * row, rows), every tile once. */
template <typename F>
P2M_HD void halo_tiles(const TileShape &g, float turn, float half, uint32_t rings, F f)
{
    int32_t ra, rb, b0, b1;
    halo_bands(g, rings, ra, rb, b0, b1);
    for (int32_t band = b0; band <= b1; ++band) {
        const BandTiles t = band_tiles(g, band, turn, half, ra, rb);
        for (int32_t j = 0; j < t.n; ++j) f(band, t.k0 + j < t.K ? t.k0 + j : t.k0 + j - t.K, t.row, t.rows);
    }
}

/* how many */
P2M_HD uint32_t halo_tile_count(const TileShape &g, float turn, float half, uint32_t rings)
{
    int32_t ra, rb, b0, b1;
    halo_bands(g, rings, ra, rb, b0, b1);
    uint32_t n = 0;
    for (int32_t band = b0; band <= b1; ++band) n += (uint32_t)band_tiles(g, band, turn, half, ra, rb).n;
    return n;
}

/* Pixel-centre z and sin(theta) of ring `ring`, exactly as pix2vec_ring
 * computes them for any pixel of that ring (pixel_routines.F90:229-311). */
P2M_HD void ring_zsth(int32_t nside, int32_t ring, double &z, double &sth)
{
    if (ring < nside) {
        double fact2 = (3.0 * nside) * nside;
        double ir = (double)ring;
        z = 1.0 - (ir / fact2) * ir;
        sth = ir * p2m_sqrt((1.0 + z) / fact2);
    } else if (ring <= 3 * nside) {
        double fact1 = 1.5 * nside;
        z = (double)(2 * nside - ring) / fact1;
        sth = p2m_sqrt((1.0 - z) * (1.0 + z));
    } else {
        double fact2 = (3.0 * nside) * nside;
        double ir = (double)(4 * nside - ring);
        z = -1.0 + (ir / fact2) * ir;
        sth = ir * p2m_sqrt((1.0 - z) / fact2);
    }
}

/* phi of pixel ip of ring `ring`: phi = (iphi + off) * HALFPI / den with the
 * association of pix2vec_ring. */
P2M_HD void ring_phi_param(int32_t nside, int32_t ring, double &off, double &den)
{
    if (ring < nside) { off = 0.5; den = (double)ring; }
    else if (ring <= 3 * nside) { off = 0.5 * (double)((ring + nside + 1) & 1); den = (double)nside; }
    else { off = 0.5; den = (double)(4 * nside - ring); }
}

P2M_DEV double ring_phi(double ip, double off, double den) { return ((ip + off) * HPX_HALFPI) / den; }

/* pix2vec_ring from the pixel index (pixel_routines.F90:167-359, I4B path). */
P2M_DEV void pix2vec_ring(int32_t nside, int64_t ipix, double v[3])
{
    int64_t npix = 12LL * nside * nside;
    int64_t nl2 = 2LL * nside;
    int64_t ncap = nl2 * (nside - 1LL);
    double z, sth, phi;
    if (ipix < ncap) {
        int64_t iring = ((int64_t)p2m_floor(p2m_sqrt((double)(2 * ipix + 2))) + 1) / 2;
        int64_t iphi = ipix - 2 * iring * (iring - 1);
        double fact2 = (3.0 * nside) * nside;
        z = 1.0 - ((double)iring / fact2) * (double)iring;
        sth = (double)iring * p2m_sqrt((1.0 + z) / fact2);
        phi = (((double)iphi + 0.5) * HPX_HALFPI) / (double)iring;
    } else if (ipix < npix - ncap) {
        int64_t nl4 = 4LL * nside;
        int64_t ip = ipix - ncap;
        int64_t iring = ip / nl4 + nside;
        int64_t iphi = ip & (nl4 - 1);
        double fact1 = 1.5 * nside;
        double fodd = 0.5 * (double)((iring + nside + 1) & 1);
        z = (double)(nl2 - iring) / fact1;
        sth = p2m_sqrt((1.0 - z) * (1.0 + z));
        phi = (((double)iphi + fodd) * HPX_HALFPI) / (double)nside;
    } else {
        int64_t ip = npix - ipix;
        int64_t iring = ((int64_t)p2m_floor(p2m_sqrt((double)(2 * ip))) + 1) / 2;
        int64_t iphi = 2 * iring * (iring + 1) - ip;
        double fact2 = (3.0 * nside) * nside;
        z = -1.0 + ((double)iring / fact2) * (double)iring;
        sth = (double)iring * p2m_sqrt((1.0 - z) / fact2);
        phi = (((double)iphi + 0.5) * HPX_HALFPI) / (double)iring;
    }
    double s, c;
    p2m_sincos(phi, &s, &c);
    v[0] = sth * c;
    v[1] = sth * s;
    v[2] = z;
}

/* angdist + vect_prod (pix_tools.F90:2015-2055) */
P2M_DEV double angdist(double ax, double ay, double az, double bx, double by, double bz)
{
    double sprod = (ax * bx + ay * by) + az * bz;
    double v0 = ay * bz - az * by;
    double v1 = az * bx - ax * bz;
    double v2 = ax * by - ay * bx;
    double vprod = p2m_sqrt((v0 * v0 + v1 * v1) + v2 * v2);
    return p2m_atan2(vprod, sprod);
}

/* phi half-width of the disc on a ring at height z (discphirange_at_z,
 * pix_tools.F90:712-760); -1000 = no intersection. */
template <typename H>
P2M_HD double disc_dphi(const H &h, double z)
{
    double dphi = -1000.0;
    double b = h.cosang - z * h.zz0;
    if (h.a == 0.0) {
        if (b <= 0.0) dphi = HPX_PI;
    } else {
        double cc = 1.0 - z * z;
        if (cc < 1.0e-12) cc = 1.0e-12;
        double cosdphi = b / p2m_sqrt(h.a * cc);
        if (cosdphi < -1.0) dphi = HPX_PI;
        if (p2m_fabs(cosdphi) <= 1.0) dphi = p2m_acos(cosdphi);
    }
    return dphi;
}

/* x mod n in [0, n) (modulo of pixels_on_edge); the disc edges lie within a
 * ring's length or two of zero, so the 64-bit division is rarely needed */
P2M_HD int64_t mod_ring(int64_t x, int64_t n)
{
    if (x >= 0 && x < n) return x;
    if (x < 0 && x >= -n) return x + n;
    if (x >= n && x < 2 * n) return x - n;
    const int64_t r = x % n;
    return r < 0 ? r + n : r;
}

/* Pixel range of the disc on ring `ring` (pixels_on_edge, pix_tools.F90:762-800,
 * and discedge2fulldisc, pixel_routines.F90:1823-1879).  Returns the number
 * of pixels np (0 if none) and the first in-ring index lo (pixels lo..lo+np-1
 * modulo npr). */
template <typename H>
P2M_HD int32_t disc_ring_run_z(const H &h, double z, int32_t npr, int32_t kshift, int32_t &lo);

template <typename H>
P2M_DEV int32_t disc_ring_run(const H &h, int32_t nside, int32_t ring, int32_t npr, int32_t kshift, int32_t &lo)
{
    return disc_ring_run_z(h, ring2z(nside, ring), npr, kshift, lo);
}

/* the same, with the ring's z (ring2z) given */
template <typename H>
P2M_HD int32_t disc_ring_run_z(const H &h, double z, int32_t npr, int32_t kshift, int32_t &lo)
{
    double dphi = disc_dphi(h, z);
    if (dphi >= HPX_PI) { lo = 0; return npr; }
    if (!(dphi >= 0.0)) return 0;
    double shift = (double)kshift * 0.5;
    int64_t il = (int64_t)p2m_ceil(((double)npr * (h.phi0 - dphi)) / HPX_TWOPI - shift);
    int64_t ih = (int64_t)p2m_floor(((double)npr * (h.phi0 + dphi)) / HPX_TWOPI - shift);
    if (ih < il) return 0;
    const int64_t l = mod_ring(il, npr);
    const int64_t hh = mod_ring(ih, npr);
    int64_t np = mod_ring(hh - l, npr);
    np += 1;
    if (np > npr) np = npr;
    lo = (int32_t)l;
    return (int32_t)np;
}

/* The run of disc_ring_run_z with the arc half-width dphi = acos(cosdphi)
 * taken as 2 asin(sqrt((1 - cosdphi)/2)) in FP32 (cosdphi itself, and
 * 1 - cosdphi, in FP64 as the reference forms them).  The ends
 * npr (phi0 -+ dphi) / 2pi - shift are formed in FP64 with the FP32 dphi;
 * when either lies within the bound of that dphi's error (1e-6 relative,
 * against a few ulp of the FP32 asin and sqrt) of an integer, where ceil or
 * floor could differ from the reference's, or the arc nearly closes the ring,
 * the exact FP64 evaluation decides.  So the returned run is the exact one
 * for every disc and ring. */
template <typename H>
P2M_HD int32_t disc_ring_run_fast(const H &h, double z, int32_t npr, int32_t kshift, int32_t &lo)
{
    if (h.a == 0.0) return disc_ring_run_z(h, z, npr, kshift, lo);      /* no acos on this branch */
    const double b = h.cosang - z * h.zz0;
    double cc = 1.0 - z * z;
    if (cc < 1.0e-12) cc = 1.0e-12;
    const double cosdphi = b / p2m_sqrt(h.a * cc);
    if (cosdphi < -1.0) { lo = 0; return npr; }
    if (!(p2m_fabs(cosdphi) <= 1.0)) return 0;
    if (1.0 + cosdphi < 1e-5) return disc_ring_run_z(h, z, npr, kshift, lo);   /* dphi near pi */
    const float sh = sqrtf((float)(0.5 * (1.0 - cosdphi)));
    const double dphi = (double)(2.0f * asinf(sh));
    const double shift = (double)kshift * 0.5;
    const double k = (double)npr * (1.0 / HPX_TWOPI);
    const double tl = (h.phi0 - dphi) * k - shift;
    const double th = (h.phi0 + dphi) * k - shift;
    const double eps = k * (1e-6 * dphi + 1e-12) + 1e-9;
    const double fl = tl - p2m_floor(tl), fh = th - p2m_floor(th);
    if (fl < eps || fl > 1.0 - eps || fh < eps || fh > 1.0 - eps) return disc_ring_run_z(h, z, npr, kshift, lo);
    const int64_t il = (int64_t)p2m_ceil(tl);
    const int64_t ih = (int64_t)p2m_floor(th);
    if (ih < il) return 0;
    const int64_t l = mod_ring(il, npr);
    const int64_t hh = mod_ring(ih, npr);
    int64_t np = mod_ring(hh - l, npr);
    np += 1;
    if (np > npr) np = npr;
    lo = (int32_t)l;
    return (int32_t)np;
}

/* asin(sqrt(h)) for h in [0, 1] to 3e-7 relative: the angle is halved twice
 * (sin^2(x/2) = h / (2 + 2 sqrt(1 - h))) and the series of asin(sqrt(y)) /
 * sqrt(y) summed to y^6 for y <= 0.147; c is cos = sqrt(1 - h). */
P2M_HD float asin_sqrt(float h, float c)
{
#if defined(__HIP_DEVICE_COMPILE__)
#define P2M_RCPF(x) __builtin_amdgcn_rcpf(x)
#define P2M_SQRTF(x) __builtin_amdgcn_sqrtf(x)
#else
#define P2M_RCPF(x) (1.0f / (x))
#define P2M_SQRTF(x) sqrtf(x)
#endif
    const float y1 = h * P2M_RCPF(__builtin_fmaf(2.0f, c, 2.0f));
    const float y = y1 * P2M_RCPF(__builtin_fmaf(2.0f, P2M_SQRTF(1.0f - y1), 2.0f));
    float p = __builtin_fmaf(y, 0.01735276f, 0.02237216f);
    p = __builtin_fmaf(y, p, 0.03038195f);
    p = __builtin_fmaf(y, p, 0.04464286f);
    p = __builtin_fmaf(y, p, 0.075f);
    p = __builtin_fmaf(y, p, 0.16666667f);
    p = __builtin_fmaf(y, p, 1.0f);
    return 4.0f * P2M_SQRTF(y) * p;
}

/* The same run from the chord relation, for a ring whose pixels lie at
 * azimuth (ip + off) kphi: the disc edge is where A + B sin^2(dphi / 2) = thr,
 * A = (z - z0)^2 + (sth - s0)^2 and B = 4 sth s0 in FP64 as the painter forms
 * them, the rest in FP32 relative to the ring pixel ipc nearest the centre,
 * x_c = ((ipc + off) kphi - phi0) / 2 (|x_c| <= kphi / 4): the run is
 * ceil((-dphi/2 - x_c) / (kphi/2)) .. floor((dphi/2 - x_c) / (kphi/2)) from
 * ipc.  Returns the number of pixels and lo in [0, npr), or -1 where the
 * exact evaluation has to decide: an end lies within the error of a pixel
 * centre, the ring only touches the disc or the arc nearly closes the ring
 * (sin^2(dphi/2) within 0.02 of 1).  Every pixel of the run is then among the
 * np_max pixels from lo (the whole ring where that is not cheap to say).
 *
 * The error of sin^2(dphi/2) against the exact evaluation's is
 * e = 4e-15 / B + 2e-15 / sth^2 (e_row: the second term), several times the
 * FP64 rounding of either form (cosang, the product z z0 and 1 - z^2, over
 * s0 sth); 2e-6 of dphi covers the FP32 quotient, roots and arc sine (the
 * slope 1 / cos is at most 7), 3e-7 of a pixel x_c. */
P2M_HD int32_t disc_ring_run_chord(double thr, double A, float B, float e_row, float xc, float ihphi, int32_t ipc,
                                   int32_t npr, int32_t &lo, int32_t &np_max)
{
    const float rB = P2M_RCPF(B);
    const float h2 = (float)(thr - A) * rB;
    const float e = __builtin_fmaf(4e-15f, rB, e_row);
    lo = 0;
    np_max = npr;
    if (h2 < -2.0f * e) return 0;
    if (h2 > 1.00001f + 2.0f * e) return npr;
    const float c = P2M_SQRTF(1.0f - h2);
    const float X = asin_sqrt(h2, c);
    const float t = X * ihphi, o = xc * ihphi;
    const float fl = -t - o, fh = t - o;
    const float eps = ihphi * e * 0.6f * P2M_RCPF(P2M_SQRTF(h2) * c) + __builtin_fmaf(t, 2e-6f, 3e-7f);
    const bool range = h2 > 2.0f * e && h2 < 0.98f && eps < 0.25f;
    const bool far = __builtin_fabsf(fl - __builtin_rintf(fl)) > eps && __builtin_fabsf(fh - __builtin_rintf(fh)) > eps;
    if (!range) return -1;
    /* undecided ends: the run with the pixels that may belong to it */
    const int32_t nl = (int32_t)__builtin_ceilf(far ? fl : fl - eps), nh = (int32_t)__builtin_floorf(far ? fh : fh + eps);
    int32_t l = ipc + nl;
    if (l < 0) l += npr;
    if (l >= npr) l -= npr;
    lo = l;
    const int32_t np = nh - nl + 1;
    np_max = np < npr ? np : npr;
    return far ? (np > 0 ? np_max : 0) : -1;
}

/* Rings of a disc without a pixel between rings with pixels (the row
 * misalignment of discedge2fulldisc, quirk Q15), counted once per gap: an empty
 * ring whose ring before holds a pixel and some ring after it too.
 *
 * A ring one ring spacing or more inside the disc's top or bottom is crossed
 * over at least 2 sqrt(2 R - 1) ring spacings, R the disc's radius in them, and
 * a pixel is at most 2.36 ring spacings wide (at the equator; 1.3 to 1.6 in
 * the caps), so an interior ring can only be empty if R < 1.2: discs that meet
 * three rings.  Asked exactly for the small ones of those, and, where the rings are short
 * (within 16 of a pole) or the disc is wide (half a turn: a pole inside or
 * near), of the two rings inside either end and of every short ring. */
template <typename H>
P2M_HD int32_t ring_run_of(const H &h, int32_t nside, int32_t ring)
{
    int32_t npr, kshift, lo = 0;
    int64_t first;
    ring_info(nside, ring, npr, kshift, first);
    return disc_ring_run_fast(h, ring2z(nside, ring), npr, kshift, lo);
}

P2M_HD bool gaps_possible(int32_t nside, double ztop, double zbot, double a, float half, uint32_t rings)
{
    const int32_t ra = (int32_t)(rings & 0xffffu), rb = (int32_t)(rings >> 16);
    if (rb - ra < 2) return false;
    if (half >= 0.5f || ra < 16 || rb > 4 * nside - 16) return true;
    if (rb - ra > 2) return false;
    /* the middle of three rings: crossed over 2 sqrt(dt db) ring spacings, dt
     * and db its distances from the top and bottom; a pixel there is 2.356
     * sin^2(theta) of them wide at most (1.58 in the caps).  Empty only if
     * that is shorter than 1.15 pixels. */
    const double dt = (double)(ra + 1) - ring_coord(nside, ztop), db = ring_coord(nside, zbot) - (double)(ra + 1);
    const double w2 = (2.356 * 1.15 * a) * (2.356 * 1.15 * a);
    return 4.0 * dt * db < (w2 > 3.3 ? w2 : 3.3);
}

template <typename H>
P2M_HD int32_t ring_gaps(const H &h, int32_t nside, uint32_t rings)
{
    const int32_t ra = (int32_t)(rings & 0xffffu), rb = (int32_t)(rings >> 16);
    int32_t gaps = 0, asked = 0, before = 0;      /* `before`: the run of ring `asked` */
    for (int32_t r = ra + 1; r < rb; ++r) {
        if (r > ra + 2 && r < rb - 2 && r >= 16 && r <= 4 * nside - 16) {
            r = rb - 3 < 4 * nside - 16 ? rb - 3 : 4 * nside - 16;      /* the next one is asked */
            continue;
        }
        const int32_t run = ring_run_of(h, nside, r);
        if (run <= 0) {
            if (asked != r - 1) before = ring_run_of(h, nside, r - 1);
            if (before > 0)
                for (int32_t k = r + 1; k <= rb; ++k)
                    if (ring_run_of(h, nside, k) > 0) { ++gaps; break; }
        }
        asked = r;
        before = run;
    }
    return gaps;
}

/* ------------------------------------------------------------ profile */
/* Table element table(p, ir, imh, ichi) through the flat column-major index,
 * addressed past the declared bounds as the reference does (quirk Q6). */
P2M_DEV double tab_flat(const float *t, int64_t nt, const TabGeom &g, int p, int ir, int imh, int ichi)
{
    int64_t idx = (int64_t)(p - 1) + 2 * ((int64_t)(ir - 1) + (int64_t)g.nrt * ((int64_t)(imh - 1) + (int64_t)g.nmht * (int64_t)(ichi - 1)));
    if (idx < 0 || idx >= nt) return 0.0;
    return (double)t[idx];
}

/* interpolate_table (maptable.f90:176-216) for a halo whose per-halo part
 * (chi, clamps, ichi/imh, fc/fm) is precomputed in h. */
P2M_DEV double interp_exact(const HaloRec &h, const TabGeom &g, const float *t, int64_t nt, int profile, double theta)
{
    if (h.chi_out) return 0.0;
    double r = h.chi_r * p2m_tan(theta);
    if (r > g.rmaxt) return 0.0;
    if (r < g.rmint) r = g.rmint + 1e-5;
    double lr = p2m_log(r);
    int ir = (int)((lr - g.lr0) / g.drt) + 1;
    double fr = lr - (g.lr0 + (double)(ir - 1) * g.drt);
    double fc = h.fc, fm = h.fm;
    int imh = h.imh, ichi = h.ichi;
    double v = tab_flat(t, nt, g, profile, ir, imh, ichi) * (1.0 - fr) * (1.0 - fc) * (1.0 - fm);
    v = v + tab_flat(t, nt, g, profile, ir + 1, imh, ichi) * (fr) * (1.0 - fc) * (1.0 - fm);
    v = v + tab_flat(t, nt, g, profile, ir, imh + 1, ichi) * (1.0 - fr) * (fc) * (1.0 - fm);
    v = v + tab_flat(t, nt, g, profile, ir + 1, imh + 1, ichi) * (fr) * (fc) * (1.0 - fm);
    v = v + tab_flat(t, nt, g, profile, ir, imh, ichi + 1) * (1.0 - fr) * (1.0 - fc) * (fm);
    v = v + tab_flat(t, nt, g, profile, ir + 1, imh, ichi + 1) * (fr) * (1.0 - fc) * (fm);
    v = v + tab_flat(t, nt, g, profile, ir, imh + 1, ichi + 1) * (1.0 - fr) * (fc) * (fm);
    v = v + tab_flat(t, nt, g, profile, ir + 1, imh + 1, ichi + 1) * (fr) * (fc) * (fm);
    return v;
}

P2M_DEV uint64_t halo_hash(int64_t i)
{
    uint64_t z = (uint64_t)i + 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

#endif
