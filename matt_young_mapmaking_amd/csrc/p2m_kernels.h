/*
 * p2m_kernels.h -- launch interface between the host runtime (p2m_api.hip)
 * and the gfx950 kernels (p2m_kernels.hip).
 */
#ifndef P2M_KERNELS_H
#define P2M_KERNELS_H

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "p2m_dev.h"

/* Statistics counters are sharded: shard k of counter c lives at
 * c + k * P2M_CTR_STRIDE, and workgroups add into shard (block % P2M_SHARDS),
 * so no address takes more than 1/64 of the atomics (same-address device
 * atomics serialise beyond the L2).  The host sums the shards.  Append
 * counters (whose value kernels read back) use shard 0 only. */
#define P2M_SHARDS 64
#define P2M_CTR_STRIDE 16

struct DecodeArgs {
    const float *halos;          /* 7 float32 per halo */
    int64_t n, index_base;
    int32_t first;               /* the call's first chunk */
    CosmoDev c;
    TabGeom g;
    double cut_low, cut_high, chihview, mmin, dmodel;
    int32_t precut;
    int32_t profile, nside, npix_fs;
    double fov, dpix;
    uint32_t *cand;              /* chunk indices that passed both cuts, all chunks */
    unsigned long long *n_cand;  /* append counter over all chunks of a call */
    unsigned long long *n_cand0; /* its value before this chunk's cull */
    HaloRec *out;                /* record k of candidate k (all chunks) */
    int64_t cap;
    uint32_t *flat_idx;          /* slots of halos the flat-sky painter covers */
    unsigned long long *n_flat_out;
    TileHalo *hot;               /* the FP32 painter's records (or NULL) */
    PairHalo *pair_halo;         /* the binning's records (tiled painters, or NULL) */
    uint32_t *n_pairs;           /* tiles each of them reaches, at shape */
    TileShape shape;
    int32_t flat_tiles;          /* count the flat-sky painter's pairs */
    unsigned long long *counters;/* sharded: [0] passed radial cut, [2] radius errors, [3] (halo, tile) pairs,
                                    [9] the flat-sky painter's, [10] halos that may have a ring gap, [14] pixels of the discs, about */
};

struct PaintArgs {
    const HaloRec *halos;
    int64_t n_halo;
    int32_t nside, npix_fs, n_maps, profile;
    double fov, dpix;
    TabGeom g;
    const float *tab_flat[P2M_MAXMAPS];
    int64_t n_flat;
    double *map64[P2M_MAXMAPS];
    double *fs64[P2M_MAXMAPS];
    uint32_t *count;
    unsigned long long *hash;
    uint32_t *fs_count;
    unsigned long long *fs_hash;
    unsigned long long *counters; /* [0] listed, [1] hp updates, [2] fs updates, [3] ring gaps */
};

struct BinArgs {
    const PairHalo *halos;
    int64_t n_halo;
    TileShape shape;
    const int32_t *band_tile;     /* first tile of each band */
    uint32_t *n_pairs;            /* tiles per halo (n_halo + 1 entries, last 0) */
    const unsigned long long *pair_off;  /* exclusive scan of n_pairs */
    uint32_t *keys, *vals;        /* the pairs, see k_pair_count */
    unsigned long long pair_cap;
    const HaloRec *recs;          /* the full records */
    uint32_t *n_split;            /* SplitArgs::n, cleared here */
    unsigned long long *counters; /* [3] ring gaps */
};

/* Geometry of a ring: the pixel-centre z and sin(theta), its phi parameters
 * (phi = (ip + off) pi/2 / den, den = npr / 4, kphi = pi/2 / den), its first
 * map pixel and pixels; e_row: see disc_ring_run_chord. */
struct __attribute__((aligned(16))) RingDesc {
    double zr, sth, off, kphi;
    int64_t first;
    int32_t npr;
    float e_row;
    int64_t pad;
};

/* A tile: its first ring, its rings, its sector k of K. */
struct __attribute__((aligned(16))) TileDesc {
    int32_t ring0, rows, k, K;
};

#define P2M_TQ_STRIDE 32           /* tile-queue counters one 128-byte line apart */
#define P2M_TQ_MAX 8192            /* of them, and workgroups of a tile painter */

/* Tiles of more than split_above pairs are painted in slices by several
 * workgroups, see k_tile_bounds: each slice adds its pixels to the tile's
 * part, the one that is done last writes the tile.  Parts and states are 0
 * between calls. */
struct __attribute__((aligned(16))) SplitUnit {
    uint32_t tile, part, from, cnt;        /* its pairs, counted from the tile's first */
    uint32_t slices, pad[3];
};
struct __attribute__((aligned(64))) SplitState {
    uint32_t arrived, lost;        /* slices done; one of them lost deferred pixels */
    unsigned long long stat[4];    /* the FP32 painter's counts: listed, updates, segments, deferrals */
};
struct SplitArgs {
    uint32_t above;                /* pairs of a tile above which it is split; 0: never */
    uint32_t unit_cap, part_cap;
    uint32_t *n;                   /* [0] units, [1] split tiles (0 before k_tile_bounds) */
    SplitUnit *units;
    SplitState *state;             /* per split tile */
    unsigned char *part;           /* per split tile, as the LDS tile: n_maps W doubles, then the membership hashes and counts */
};

struct TileArgs {
    const HaloRec *halos;
    const TileHalo *hot;          /* the same halos, packed for the FP32 painter */
    TileShape shape;
    int32_t nside, log2w, n_maps, profile, accumulate;
    int64_t n_tiles;
    const TileDesc *desc;
    const RingDesc *ring;         /* of every ring */
    const unsigned long long *tile_off;
    const uint32_t *keys, *vals;  /* the sorted pairs */
    TabGeom g;
    const float *tab_flat[P2M_MAXMAPS];
    const float *tab_q;           /* corner-quad table (k_build_quad): a pixel's nodes ir-1, ir of its
                                     cell, 4 corners of every map, are 8 n_maps contiguous floats */
    int64_t n_quad;               /* floats in tab_q */
    int64_t n_flat;
    const float *inv_node2f;      /* exp(-2 (lr0 + k drt)), k = 0..nrt */
    float u_k1, u_k0, u_max, band, fr_clamp;
    double inv_drt, u_max64, band64, fr_clamp64;     /* the FP64 painter's: 1/drt, nrt - 1, the band around cell
                                                        boundaries (in cells) that takes the exact arithmetic */
    int32_t ir_clamp;             /* cell and fraction of r = rmint + 1e-5 (maptable.f90:190, 196, 200) */
    float band_c;                 /* CHORD_BAND */
    double *map64[P2M_MAXMAPS];
    float *map32[P2M_MAXMAPS];
    uint32_t *count;
    unsigned long long *hash;
    uint4 *fb;                    /* deferred FP64 pixels: (row, in-row pixel, halo, tile), P2M_SHARDS sub-lists */
    unsigned long long *fb_count; /* sharded: sub-list k's length at fb_count[k * P2M_CTR_STRIDE] */
    int64_t fb_cap;               /* total; each sub-list holds fb_cap / P2M_SHARDS */
    uint8_t *lost;                /* per tile: set when its deferred pixels did not all fit in fb;
                                     such a tile writes nothing (it is painted again) */
    int32_t redo;                 /* paint only the tiles marked lost, clearing the mark of each
                                     that now fits */
    int64_t n_halo;               /* records in hot / halos */
    unsigned int *tile_next;      /* the tile queues: one counter per XCD or workgroup, P2M_TQ_STRIDE
                                     apart (zeroed by p2m_launch_tile_paint) */
    SplitArgs split;
    int32_t wide;                 /* pairs are mostly the insides of wide discs (paint_exact) */
    int32_t vectors;              /* the FP64 painter keeps pixel vectors (p2m_exact_vectors) */
    unsigned long long *counters; /* [0] listed, [1] hp updates, [4] segments, [5] FP64 fallbacks */
    unsigned long long *err;      /* sharded: pairs whose halo or rows are out of bounds */
    unsigned long long *n_lost;   /* sharded: tiles marked lost */
};

/* the flat-sky painter's (halo, tile) pairs and maps; its tables are TileArgs' */
struct FlatArgs {
    const HaloRec *halos;
    const uint32_t *list;         /* halos to paint */
    int64_t n_list;
    int32_t first;                /* the first part of a call's list: the count starts anew */
    int32_t npix, nj;             /* the map's pixels a side, its tiles in a row of tiles */
    int64_t n_tiles;
    int32_t slices;               /* lists per tile: list k of tile t is k n_tiles + t */
    double fov, dpix;
    uint32_t *cnt;                /* pairs per list while they are listed, 0 before and after; one more 0 */
    unsigned long long *off;      /* their exclusive scan */
    uint2 *pairs;                 /* by list: first row << 4 | rows - 1, halo */
    unsigned long long pair_cap;
    double *map[P2M_MAXMAPS];
    uint32_t *count;
    unsigned long long *hash;
    unsigned long long *counters; /* [2] updates */
};

struct FallbackArgs {
    const HaloRec *halos;
    const uint4 *fb;
    const unsigned long long *fb_count;
    int64_t fb_cap;
    int32_t nside, n_maps, profile;
    TabGeom g;
    const float *tab_flat[P2M_MAXMAPS];
    int64_t n_flat;
    float *map32[P2M_MAXMAPS];
    uint32_t *count;
    unsigned long long *hash;
    const uint8_t *lost;          /* per tile: entries of a lost tile are skipped (it is painted again) */
    const TileDesc *desc;
    int64_t n_tiles;
    int64_t n_halo;
    unsigned long long *counters; /* [0] listed, [1] hp updates */
    unsigned long long *err;      /* sharded: entries whose halo is out of range */
};

void p2m_launch_fill_u32(uint32_t *p, int64_t n, uint32_t v, hipStream_t s);
void p2m_launch_fill_u64(unsigned long long *p, int64_t n, hipStream_t s);
void p2m_launch_fill_f64(double *p, int64_t n, hipStream_t s);
void p2m_launch_fill_f32(float *p, int64_t n, hipStream_t s);
void p2m_launch_clear_ctr(unsigned long long *ctr, int first, int count, hipStream_t s);
void p2m_launch_decode(const DecodeArgs &a, hipStream_t s);
void p2m_launch_paint_plain_hp(const PaintArgs &a, hipStream_t s);
void p2m_launch_paint_fs(const PaintArgs &a, hipStream_t s);
int64_t p2m_flat_tiles(int32_t npix, int32_t *nj);
int p2m_flat_slices(int64_t n_tiles, int64_t n_pairs);
void p2m_launch_flat_pairs(const FlatArgs &f, int emit, hipStream_t s);
int p2m_launch_flat_paint(const TileArgs &a, const FlatArgs &f, hipStream_t s);
void p2m_launch_pair_count(const BinArgs &b, hipStream_t s);
void p2m_launch_ring_gaps(const BinArgs &b, hipStream_t s);
void p2m_launch_pair_emit(const BinArgs &b, hipStream_t s);
void p2m_launch_tile_bounds(const uint32_t *keys, unsigned long long n, int64_t n_tiles, unsigned long long *tile_off,
                            const SplitArgs &split, unsigned long long *err, hipStream_t s);
int p2m_sort_pairs(uint32_t *keys, uint32_t *vals, unsigned long long n, int64_t n_tiles, void *tmp, size_t *tmp_bytes,
                   hipStream_t s);
void p2m_launch_ring_desc(int32_t nside, RingDesc *out, hipStream_t s);
void p2m_launch_tile_desc(const TileShape &g, const int32_t *band_tile, TileDesc *desc, hipStream_t s);
int p2m_scan_u32(const uint32_t *cnt, unsigned long long *off, int64_t n, void *tmp, size_t *tmp_bytes, hipStream_t s);
int p2m_tile_max_log2w(void);
void p2m_launch_build_quad(const float *flat, int64_t n_flat, int32_t profile, int32_t nrt, int32_t nmht, int32_t nchit,
                           int32_t n_maps, int32_t slot, float *quad, hipStream_t s);
size_t p2m_tile_lds_bytes(int mode, int n_maps, int log2w, int membership, int nrt, int wg);
int p2m_exact_vectors(int n_maps, int log2w, int membership, int wg);
int p2m_tile_wg(int mode, int n_maps, int log2w, int membership, int nrt, int wg);
int p2m_tile_occupancy(int mode, int n_maps, int wg, size_t lds);
int p2m_launch_tile_paint(const TileArgs &a, int mode, int n_maps, int grid, int wg, hipStream_t s);
int p2m_launch_fallback(const FallbackArgs &a, int64_t n_max, hipStream_t s);
#define P2M_MOM_BLOCKS 256       /* most workgroups of the moments kernel */
#define P2M_MOM_PART 5           /* doubles each writes: sums of x, x^2, x^3, its mean, squares about it */
int64_t p2m_moments_chunk(int64_t n);
void p2m_launch_moments(const float *m32, const double *m64, int64_t n, double *part, unsigned long long *hist, int nb,
                        float dy, hipStream_t s);
void p2m_launch_f64_to_f32(const double *in, float *out, int64_t n, hipStream_t s);
void p2m_launch_f32_to_f64(const float *in, double *out, int64_t n, hipStream_t s);

int p2m_launch_selftest_math(int op, const double *x, const double *y, double *out, int64_t n, hipStream_t s);
int p2m_launch_copy_calib(const void *src, void *dst, int64_t n4, hipStream_t s);

/* make_maptable kernel (p2m_maptable.hip) */
int p2m_launch_make_maptable(int32_t model, double nu, double alpha_cmb, int32_t nchit, int32_t nmht, int32_t nrt,
                             const double *d_rofz, const double *d_zofr, float *d_table, hipStream_t s);

#endif
