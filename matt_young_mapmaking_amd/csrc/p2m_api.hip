/*
 * p2m_api.hip -- host runtime behind the C ABI of include/pks2map_gpu.h.
 *
 * Owns the device state of one pks2map run: distance tables, profile tables,
 * maps, per-halo records, (halo, tile) pairs.  A paint call decodes the
 * catalogue in chunks (appending painted halos to one device array), lists
 * the tiles that every disc may reach, sorted by tile, and paints all tiles
 * in one launch, so each map pixel is written once per call.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <ctime>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/pks2map_gpu.h"
#include "p2m_convert.h"
#include "p2m_kernels.h"

/* Scratch of the map products: the 10000-bin dP/dy histogram (u64), then the
 * workgroups' partial sums of one map.  p2m_products keeps one per context;
 * p2m_products_noalloc uses one array per GPU, kept for the life of the
 * process, whose device address comes from hipGetSymbolAddress once per
 * device (the array's name is a host-side stand-in in host code). */
#define P2M_NDPDY 10000
#define P2M_NOALLOC_BYTES (128 * 1024)
#define P2M_PROD_PART_OFF (8 * P2M_NDPDY)
#define P2M_PROD_PART_BYTES (8 * P2M_MOM_PART * P2M_MOM_BLOCKS)
#define P2M_PROD_BYTES (P2M_PROD_PART_OFF + P2M_PROD_PART_BYTES)
static_assert(P2M_PROD_BYTES <= P2M_NOALLOC_BYTES, "no-alloc scratch layout");
static __device__ __align__(256) unsigned char scratch[P2M_NOALLOC_BYTES];
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[64];

/* the device address of this device's scratch (the device must be current) */
static int scratch_for_device(int device, void **out)
{
    if (device < 0 || device >= 64) return P2M_E_INVALID;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *ptr = nullptr;
        if (hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
            (void)hipGetLastError();
            return P2M_E_HIP;
        }
        g_scratch_ptr[device] = ptr;
    }
    *out = g_scratch_ptr[device];
    return 0;
}

/* last HIP failure of this thread, reported by p2m_strerror(P2M_E_HIP) */
static thread_local char g_hip_detail[256] = "";

static int hip_fail(hipError_t e, const char *what, int line)
{
    snprintf(g_hip_detail, sizeof(g_hip_detail), "HIP runtime error: %s (%s) at p2m_api.hip:%d: %s",
             hipGetErrorName(e), hipGetErrorString(e), line, what);
    (void)hipGetLastError();
    return P2M_E_HIP;
}

#define HIPCHK(x)                                                  \
    do {                                                           \
        hipError_t e_ = (x);                                       \
        if (e_ != hipSuccess) return hip_fail(e_, #x, __LINE__);   \
    } while (0)

namespace {

const double CKMS = 2.99792458e10 / 1e5;   /* cosmology.f90:23 */

struct Ctr {                 /* layout of one shard row of the device counter block; PAIRS, GAPS and
                                PIX are the decode's (halo, tile) pairs, halos that may have a ring
                                gap and disc pixels (about);
                                ERR counts failed device-side range
                                checks, LOST the tiles marked for the repaint pass */
    enum { ERR = 0, DEC = 1, LOST = 2, PAIRS = 4, N_FLAT = 5, N_CAND = 6, N_CAND0 = 7, PAINT = 8, GAPS = 11, PIX = 15,
           TOTAL = P2M_CTR_STRIDE, ALL = P2M_CTR_STRIDE * P2M_SHARDS };
};

}  // namespace

struct p2m_ctx {
    p2m_config cfg;
    hipStream_t stream = nullptr;
    hipEvent_t ev[10] = {};
    hipStream_t fs_stream = nullptr;            /* the flat-sky painter, beside the binning */
    hipEvent_t ev_dec = nullptr, ev_fs = nullptr;
    /* one host block, page-locked if that is to be had, of words for readbacks
     * and of a copy of the products' scratch */
    unsigned long long *h_pin = nullptr;
    char *h_prod = nullptr;
    bool host_pinned = true;
    char *d_prod = nullptr;                /* the products' scratch, in d_ctr's allocation */
    bool have_run = false;
    bool have_table[P2M_MAXMAPS] = {false};
    p2m_run run;
    double cut_low = 0, cut_high = 0, mypi = 0;
    std::vector<double> rofz, zofr;
    double *d_rofz = nullptr, *d_zofr = nullptr;
    CosmoDev cdev;
    int32_t hdr_i[3] = {0, 0, 0};
    float hdr_f[6] = {0, 0, 0, 0, 0, 0};
    TabGeom g;
    float *d_flat[P2M_MAXMAPS] = {nullptr};
    float *d_quad = nullptr;                    /* corner-quad table of all maps (tiled painters) */
    int64_t n_flat = 0, n_quad = 0;
    float *d_inv_node2f = nullptr;
    uint4 *d_fb = nullptr;
    int64_t fb_cap = 0;
    double fr_clamp64 = 0.0;
    float fr_clamp = 0.f, u_k1 = 0.f, u_k0 = 0.f, u_max = 0.f;
    int32_t ir_clamp = 1;
    float u_band = 2.5e-4f;     /* half-width of the deferral band around cell boundaries, in cells */
    int64_t hpnpix = 0, fsnpix = 0;
    double *d_hp64[P2M_MAXMAPS] = {nullptr};
    float *d_hp32[P2M_MAXMAPS] = {nullptr};
    double *d_fs64[P2M_MAXMAPS] = {nullptr};
    uint32_t *d_count = nullptr, *d_fs_count = nullptr;
    unsigned long long *d_hash = nullptr, *d_fs_hash = nullptr;
    bool hp_zero = true;        /* next paint may store instead of accumulate */
    bool hp_valid = true;       /* device HEALPix arrays hold the map (false after a lazy clear) */
    HaloRec *d_halo = nullptr;
    uint32_t *d_flat_idx = nullptr;
    PairHalo *d_pair_halo = nullptr;              /* what the binning reads of a halo (tiled painters) */
    TileHalo *d_hot = nullptr;                    /* what the FP32 painter stages of it */
    uint32_t *d_n_pairs = nullptr;                /* tiles per halo, and their scan */
    unsigned long long *d_pair_off = nullptr;
    uint32_t *d_keys = nullptr, *d_vals = nullptr;  /* (halo, tile) pairs: as listed, then sorted by tile (one allocation) */
    int64_t pair_cap = 0;
    int counted_log2w = 0;                        /* the tile shape that n_pairs were counted at, and their sum */
    unsigned long long counted_pairs = 0;
    bool ask_gaps = false;                        /* the decode marked halos that may have a ring gap */
    int64_t halo_cap = 0;
    unsigned long long *d_ctr = nullptr;
    int log2w = 0, wg = 0;
    bool tuned = false;
    TileShape shape = {0, 0, 0};
    int32_t *d_band_tile = nullptr; /* first tile of each band */
    int n_cu = 0;                   /* compute units of the device */
    TileDesc *d_tile_desc = nullptr;
    RingDesc *d_ring = nullptr;     /* geometry of every ring */
    uint32_t *d_fs_cnt = nullptr;   /* flat-sky pairs per tile (0 between calls), and their scan */
    unsigned long long *d_fs_off = nullptr;
    uint2 *d_fs_pairs = nullptr;
    unsigned long long flat_pairs = 0;      /* the decode's count of them */
    int64_t fs_cap = 0;
    int64_t n_tiles = 0;
    unsigned long long *d_tile_off = nullptr;
    void *d_scan_tmp = nullptr;
    size_t scan_tmp_bytes = 0;
    void *d_scan_tmp_fs = nullptr;              /* the flat-sky painter's own scan storage */
    size_t scan_tmp_fs_bytes = 0;
    /* host catalogues: two device slots that pieces of a block are copied
     * into on the copy stream, decoded from on the painter's stream */
    hipStream_t h2d_stream = nullptr;
    hipEvent_t ev_copy[2] = {nullptr, nullptr}, ev_free[2] = {nullptr, nullptr};
    hipEvent_t ev_push = nullptr, ev_h2d_end = nullptr;
    float *d_slot[2] = {nullptr, nullptr};
    int64_t slot_cap = 0;                       /* halos per slot */
    /* the streamed pass in progress (p2m_stream_*; p2m_paint* run one) */
    bool in_stream = false;
    int64_t stream_total = 0, stream_pushed = 0, stream_h2d_bytes = 0;
    int n_host_push = 0, n_pieces = 0;
    bool stream_pinned = true;
    /* per tile: 1 if the tile's deferred pixels did not all fit in the list
     * (the tile then wrote nothing and is painted again) */
    uint8_t *d_lost = nullptr;
    unsigned int *d_tile_next = nullptr;   /* tile-queue counters */
    unsigned char *d_split = nullptr;      /* slices of split tiles: count, units, states, parts */
    size_t split_bytes = 0;
    int n_redo = 0;
    /* the FP32 painter's last launch, kept for the repaint pass */
    TileArgs last_t;
    FallbackArgs last_f;
    int64_t n_chunks = 0;                   /* chunks of the call decoded */
    int last_grid = 0, last_wg = 0;
    bool last_fast = false;
    uint32_t *d_cand = nullptr;
    int64_t cand_cap = 0;
    void *d_conv = nullptr;        /* a piece of a map in the other precision (p2m_fetch_maps) */
    int64_t conv_cap = 0;          /* its values */
    void *d_sort_tmp = nullptr;
    size_t sort_tmp_bytes = 0;
    p2m_stats st;
};

/* ------------------------------------------------------------------ helpers */
static int dmalloc(void **p, size_t bytes)
{
    if (bytes == 0) { *p = nullptr; return 0; }
    if (hipMalloc(p, bytes) != hipSuccess) { *p = nullptr; (void)hipGetLastError(); return P2M_E_NOMEM; }
    return 0;
}
static void dfree(void *p) { if (p) (void)hipFree(p); }

/* the same for a context that may hold memory it can do without: the
 * conversion buffer of p2m_fetch_maps, given back where device memory is short */
static int grow(p2m_ctx *c, void **p, size_t bytes)
{
    const int rc = dmalloc(p, bytes);
    if (!rc || !c->d_conv) return rc;
    dfree(c->d_conv);
    c->d_conv = nullptr;
    c->conv_cap = 0;
    return dmalloc(p, bytes);
}

/* cosmology.f90:123-133 (dzdr) and 109-119 (drdz), FP64 */
static double dzdr(double h, double om, double z)
{
    double z1 = 1.0 + z;
    return ((h * 100.0) / CKMS) * p2m_sqrt((om * ((z1 * z1) * z1) + 1.0) - om);
}

static double host_lookup(const std::vector<double> &t, double tmin, double dt, double x)
{
    if (x != x) return x;
    int n = (int)t.size();
    double u = (x - tmin) / dt + 1.0;
    if (u < 1.0) return t[0];
    if (u >= (double)n) return t[n - 1];
    int itab = (int)u;
    double fint = ((x - (double)(itab - 1) * dt) - tmin) / dt;
    return (1.0 - fint) * t[itab - 1] + fint * t[itab];
}

static bool is_pow2(int32_t x) { return x > 0 && (x & (x - 1)) == 0; }

static int build_tiles(p2m_ctx *c, int log2w)
{
    int32_t ns = c->cfg.nside;
    if (ns <= 0) return 0;
    if (c->log2w == log2w && c->d_tile_desc) return 0;
    const TileShape g = tile_shape(ns, log2w);
    const int32_t nb = n_bands(g);
    std::vector<int32_t> band_tile((size_t)nb + 1);
    int64_t acc = 0;
    for (int32_t b = 0; b < nb; ++b) {
        int32_t r0, r1;
        band_tile[(size_t)b] = (int32_t)acc;
        acc += band_sectors(g, b, r0, r1);
    }
    band_tile[(size_t)nb] = (int32_t)acc;
    /* a pair's key holds the tile in 24 bits (at most 1.3e7 tiles: 64 pixels, nside 8192) */
    if (acc >= (1 << 24)) return P2M_E_SIZE;
    c->n_tiles = acc;
    dfree(c->d_band_tile); dfree(c->d_tile_off); dfree(c->d_tile_desc); dfree(c->d_lost);
    c->d_band_tile = nullptr; c->d_tile_off = nullptr; c->d_tile_desc = nullptr; c->d_lost = nullptr;
    c->log2w = 0;
    int rc = 0;
    rc |= grow(c, (void **)&c->d_lost, (size_t)((acc + 3) / 4) * 4);
    if (!c->d_tile_next) rc |= grow(c, (void **)&c->d_tile_next, sizeof(unsigned int) * P2M_TQ_MAX * P2M_TQ_STRIDE);
    rc |= grow(c, (void **)&c->d_tile_desc, sizeof(TileDesc) * acc);
    rc |= grow(c, (void **)&c->d_band_tile, sizeof(int32_t) * (size_t)(nb + 1));
    rc |= grow(c, (void **)&c->d_tile_off, sizeof(unsigned long long) * (c->n_tiles + 1));
    if (rc) return P2M_E_NOMEM;
    HIPCHK(hipMemcpy(c->d_band_tile, band_tile.data(), sizeof(int32_t) * (size_t)(nb + 1), hipMemcpyHostToDevice));
    p2m_launch_tile_desc(g, c->d_band_tile, c->d_tile_desc, c->stream);
    p2m_launch_fill_u32((uint32_t *)c->d_lost, (acc + 3) / 4, 0u, c->stream);
    HIPCHK(hipGetLastError());
    if (!c->d_ring) {
        if (grow(c, (void **)&c->d_ring, sizeof(RingDesc) * (size_t)(4 * ns - 1))) return P2M_E_NOMEM;
        p2m_launch_ring_desc(ns, c->d_ring, c->stream);
        HIPCHK(hipGetLastError());
    }
    c->shape = g;
    c->log2w = log2w;
    return 0;
}

/* ------------------------------------------------------------------ ABI */
extern "C" {

const char *p2m_version(void) { return "p2m 1.0 (gfx950)"; }

const char *p2m_strerror(int code)
{
    switch (code) {
    case P2M_OK: return "ok";
    case P2M_E_INVALID: return "invalid argument";
    case P2M_E_SIZE: return "buffer or header size mismatch";
    case P2M_E_HIP: return g_hip_detail[0] ? g_hip_detail : "HIP runtime error";
    case P2M_E_NOMEM: return "allocation failed";
    case P2M_E_RADIUS: return "disc radius outside [0, pi]";
    case P2M_E_STATE: return "call out of order (run parameters or table missing)";
    case P2M_E_IO: return "file could not be written";
    case P2M_E_NODEVICE: return "no GPU visible";
    case P2M_E_INTERNAL: return g_hip_detail[0] ? g_hip_detail : "device-side consistency check failed";
    default: return "unknown error";
    }
}

int p2m_create(p2m_ctx **out, const p2m_config *cfg)
{
    if (!out || !cfg) return P2M_E_INVALID;
    *out = nullptr;
    if (cfg->nside < 0 || (cfg->nside > 0 && (!is_pow2(cfg->nside) || cfg->nside > 8192))) return P2M_E_INVALID;
    if (cfg->npix_fs < 0 || cfg->npix_fs > 65536) return P2M_E_INVALID;
    if (cfg->n_maps < 1 || cfg->n_maps > P2M_MAXMAPS) return P2M_E_INVALID;
    if (cfg->model < 1 || cfg->model > 3) return P2M_E_INVALID;
    if (cfg->profile < 1 || cfg->profile > 2) return P2M_E_INVALID;
    if (cfg->precision < P2M_PREC_PLAIN_FP64 || cfg->precision > P2M_PREC_FP32_COMP) return P2M_E_INVALID;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) { (void)hipGetLastError(); return P2M_E_NODEVICE; }
    if (cfg->device < 0 || cfg->device >= ndev) return P2M_E_INVALID;
    HIPCHK(hipSetDevice(cfg->device));
    p2m_ctx *c = new p2m_ctx();
    c->cfg = *cfg;
    {
        int ncu = 0;
        if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, cfg->device) == hipSuccess) c->n_cu = ncu;
        else (void)hipGetLastError();
    }
    if (c->cfg.chunk_halos <= 0) c->cfg.chunk_halos = 1 << 26;
    if (c->cfg.chunk_halos > (1LL << 30)) c->cfg.chunk_halos = 1LL << 30;   /* chunk indices are 32-bit */
    memset(&c->st, 0, sizeof(c->st));
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) { delete c; return P2M_E_HIP; }
    if (hipStreamCreateWithFlags(&c->fs_stream, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&c->h2d_stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&c->ev_dec, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->ev_fs, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->ev_copy[0], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->ev_copy[1], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->ev_free[0], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->ev_free[1], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->ev_push, hipEventDisableTiming) != hipSuccess ||
        hipEventCreate(&c->ev_h2d_end) != hipSuccess) {
        (void)hipGetLastError();
        p2m_destroy(c);
        return P2M_E_HIP;
    }
    for (int i = 0; i < 10; ++i) (void)hipEventCreate(&c->ev[i]);
    {
        /* this device's scratch of p2m_products_noalloc, resolved once */
        void *sp = nullptr;
        int e = scratch_for_device(cfg->device, &sp);
        if (e) { p2m_destroy(c); return e; }
    }
    const size_t pin_bytes = sizeof(unsigned long long) * (Ctr::ALL + 8), host_bytes = pin_bytes + P2M_PROD_BYTES + P2M_PROD_PART_BYTES;
    if (hipHostMalloc((void **)&c->h_pin, host_bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        c->host_pinned = false;
        c->h_pin = (unsigned long long *)malloc(host_bytes);
        if (!c->h_pin) { p2m_destroy(c); return P2M_E_NOMEM; }
    }
    c->h_prod = (char *)c->h_pin + pin_bytes;
    c->hpnpix = cfg->nside > 0 ? 12LL * cfg->nside * cfg->nside : 0;
    c->fsnpix = (int64_t)cfg->npix_fs * cfg->npix_fs;
    int rc = 0;
    for (int m = 0; m < cfg->n_maps && !rc; ++m) {
        if (c->hpnpix) {
            if (cfg->precision == P2M_PREC_FP32_COMP) rc |= dmalloc((void **)&c->d_hp32[m], sizeof(float) * c->hpnpix);
            else rc |= dmalloc((void **)&c->d_hp64[m], sizeof(double) * c->hpnpix);
        }
        if (c->fsnpix) rc |= dmalloc((void **)&c->d_fs64[m], sizeof(double) * c->fsnpix);
    }
    if (!rc && (cfg->flags & P2M_FLAG_MEMBERSHIP)) {
        if (c->hpnpix) {
            rc |= dmalloc((void **)&c->d_count, sizeof(uint32_t) * c->hpnpix);
            rc |= dmalloc((void **)&c->d_hash, sizeof(unsigned long long) * c->hpnpix);
        }
        if (c->fsnpix) {
            rc |= dmalloc((void **)&c->d_fs_count, sizeof(uint32_t) * c->fsnpix);
            rc |= dmalloc((void **)&c->d_fs_hash, sizeof(unsigned long long) * c->fsnpix);
        }
    }
    if (!rc) rc |= dmalloc((void **)&c->d_ctr, sizeof(unsigned long long) * Ctr::ALL + P2M_PROD_BYTES);
    if (!rc) c->d_prod = (char *)(c->d_ctr + Ctr::ALL);
    if (rc) { p2m_destroy(c); return P2M_E_NOMEM; }
    *out = c;
    int e = p2m_clear(c);
    if (e) { p2m_destroy(c); *out = nullptr; return e; }
    return 0;
}

void p2m_destroy(p2m_ctx *c)
{
    if (!c) return;
    (void)hipSetDevice(c->cfg.device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    if (c->fs_stream) (void)hipStreamSynchronize(c->fs_stream);
    if (c->h2d_stream) (void)hipStreamSynchronize(c->h2d_stream);
    dfree(c->d_slot[0]); dfree(c->d_slot[1]); dfree(c->d_lost); dfree(c->d_tile_next); dfree(c->d_split);
    for (int i = 0; i < 2; ++i) {
        if (c->ev_copy[i]) (void)hipEventDestroy(c->ev_copy[i]);
        if (c->ev_free[i]) (void)hipEventDestroy(c->ev_free[i]);
    }
    if (c->ev_push) (void)hipEventDestroy(c->ev_push);
    if (c->ev_h2d_end) (void)hipEventDestroy(c->ev_h2d_end);
    if (c->h2d_stream) (void)hipStreamDestroy(c->h2d_stream);
    for (int m = 0; m < P2M_MAXMAPS; ++m) {
        dfree(c->d_hp64[m]); dfree(c->d_hp32[m]); dfree(c->d_fs64[m]); dfree(c->d_flat[m]);
    }
    dfree(c->d_quad);
    dfree(c->d_count); dfree(c->d_hash); dfree(c->d_fs_count); dfree(c->d_fs_hash);
    dfree(c->d_rofz); dfree(c->d_zofr); dfree(c->d_inv_node2f); dfree(c->d_fb);
    dfree(c->d_halo); dfree(c->d_flat_idx); dfree(c->d_n_pairs); dfree(c->d_pair_off); dfree(c->d_ctr);
    dfree(c->d_band_tile); dfree(c->d_tile_off); dfree(c->d_scan_tmp); dfree(c->d_scan_tmp_fs);
    dfree(c->d_tile_desc); dfree(c->d_ring); dfree(c->d_fs_cnt); dfree(c->d_fs_off); dfree(c->d_fs_pairs);
    dfree(c->d_cand);
    dfree(c->d_hot); dfree(c->d_pair_halo); dfree(c->d_keys); dfree(c->d_sort_tmp);
    for (int i = 0; i < 10; ++i) if (c->ev[i]) (void)hipEventDestroy(c->ev[i]);
    if (c->h_pin && c->host_pinned) (void)hipHostFree(c->h_pin);
    if (!c->host_pinned) free(c->h_pin);
    dfree(c->d_conv);
    if (c->ev_dec) (void)hipEventDestroy(c->ev_dec);
    if (c->ev_fs) (void)hipEventDestroy(c->ev_fs);
    if (c->fs_stream) (void)hipStreamDestroy(c->fs_stream);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

int p2m_clear(p2m_ctx *c)
{
    if (!c) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    HIPCHK(hipSetDevice(c->cfg.device));
    /* the tiled painters store every HEALPix pixel on the first paint after a
     * clear, so only the plain painter (atomics) needs a zeroed map */
    const bool tiled = c->cfg.precision != P2M_PREC_PLAIN_FP64;
    for (int m = 0; m < c->cfg.n_maps; ++m) {
        if (c->d_hp64[m] && !tiled) p2m_launch_fill_f64(c->d_hp64[m], c->hpnpix, c->stream);
        if (c->d_fs64[m]) p2m_launch_fill_f64(c->d_fs64[m], c->fsnpix, c->stream);
    }
    if (c->d_count && !tiled) p2m_launch_fill_u32(c->d_count, c->hpnpix, 0u, c->stream);
    if (c->d_hash && !tiled) p2m_launch_fill_u64(c->d_hash, c->hpnpix, c->stream);
    if (c->d_fs_count) p2m_launch_fill_u32(c->d_fs_count, c->fsnpix, 0u, c->stream);
    if (c->d_fs_hash) p2m_launch_fill_u64(c->d_fs_hash, c->fsnpix, c->stream);
    HIPCHK(hipGetLastError());
    /* no wait: later work on the painter's stream is ordered after the
     * fills, and every readback waits for the stream first */
    c->hp_zero = true;
    c->hp_valid = !tiled;
    return 0;
}

/* Zero-fill the HEALPix arrays if a lazy clear left them unwritten. */
static int ensure_hp_valid(p2m_ctx *c)
{
    if (c->hp_valid) { HIPCHK(hipStreamSynchronize(c->stream)); return 0; }
    for (int m = 0; m < c->cfg.n_maps; ++m) {
        if (c->d_hp64[m]) p2m_launch_fill_f64(c->d_hp64[m], c->hpnpix, c->stream);
        if (c->d_hp32[m]) p2m_launch_fill_f32(c->d_hp32[m], c->hpnpix, c->stream);
    }
    if (c->d_count) p2m_launch_fill_u32(c->d_count, c->hpnpix, 0u, c->stream);
    if (c->d_hash) p2m_launch_fill_u64(c->d_hash, c->hpnpix, c->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(c->stream));
    c->hp_valid = true;
    return 0;
}

int p2m_set_run(p2m_ctx *c, const p2m_run *r)
{
    if (!c || !r) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (!(r->h > 0) || !(r->omegam > 0)) return P2M_E_INVALID;
    HIPCHK(hipSetDevice(c->cfg.device));
    c->run = *r;
    /* set_rofztable, cosmology.f90:51-76 */
    const int n = 10000;
    double dz = (6.0 - 0.0) / (double)(n - 1);
    c->rofz.assign(n, 0.0);
    for (int i = 2; i <= n; ++i) {
        double z = (double)(i - 1) * dz + 0.0;
        c->rofz[i - 1] = c->rofz[i - 2] + (1.0 / dzdr(r->h, r->omegam, z)) * dz;
    }
    /* set_zofrtable, cosmology.f90:80-105 */
    double dr = (1.3e4 - 0.0) / (double)(n - 1);
    c->zofr.assign(n, 0.0);
    for (int i = 2; i <= n; ++i) {
        double z = c->zofr[i - 2];
        c->zofr[i - 1] = c->zofr[i - 2] + dzdr(r->h, r->omegam, z) * dr;
    }
    if (!c->d_rofz && grow(c, (void **)&c->d_rofz, sizeof(double) * n)) return P2M_E_NOMEM;
    if (!c->d_zofr && grow(c, (void **)&c->d_zofr, sizeof(double) * n)) return P2M_E_NOMEM;
    HIPCHK(hipMemcpy(c->d_rofz, c->rofz.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(c->d_zofr, c->zofr.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    c->mypi = 4.0 * p2m_atan(1.0);                         /* pks2map.f90:88 */
    c->cdev.rofz = c->d_rofz; c->cdev.zofr = c->d_zofr;
    c->cdev.drofz = dz; c->cdev.dzofr = dr; c->cdev.rofz_min = 0.0; c->cdev.zofr_min = 0.0;
    c->cdev.nrofz = n; c->cdev.nzofr = n;
    c->cdev.omegam = r->omegam; c->cdev.omegal = r->omegal;
    c->cdev.rho_0 = (2.775e11 * r->omegam) * (r->h * r->h);     /* pks2map.f90:127 */
    c->cdev.rhocrit_0 = 2.775e11 * (r->h * r->h);               /* :128 */
    c->cdev.mypi = c->mypi;
    c->cut_low = host_lookup(c->rofz, 0.0, dz, r->zmin);        /* :134 */
    c->cut_high = host_lookup(c->rofz, 0.0, dz, r->zmax);       /* :135 */
    c->have_run = true;
    return 0;
}

int p2m_rofz(p2m_ctx *c, double z, double *chi)
{
    if (!c || !chi) return P2M_E_INVALID;
    if (!c->have_run) return P2M_E_STATE;
    *chi = host_lookup(c->rofz, 0.0, 6.0 / 9999.0, z);
    return 0;
}

int p2m_zofr(p2m_ctx *c, double chi, double *z)
{
    if (!c || !z) return P2M_E_INVALID;
    if (!c->have_run) return P2M_E_STATE;
    *z = host_lookup(c->zofr, 0.0, 1.3e4 / 9999.0, chi);
    return 0;
}

int p2m_load_table(p2m_ctx *c, int slot, const int32_t hdr_i[3], const float hdr_f[6], const float *table, int64_t n_table)
{
    if (!c || !hdr_i || !hdr_f || !table) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (slot < 0 || slot >= c->cfg.n_maps) return P2M_E_INVALID;
    if (hdr_i[0] < 2 || hdr_i[1] < 2 || hdr_i[2] < 2) return P2M_E_SIZE;
    int64_t nt = 2LL * hdr_i[0] * hdr_i[1] * hdr_i[2];
    if (n_table != nt) return P2M_E_SIZE;
    if (!(hdr_f[0] > 0 && hdr_f[1] > hdr_f[0] && hdr_f[2] > 0 && hdr_f[3] > hdr_f[2] && hdr_f[4] > 0 && hdr_f[5] > hdr_f[4]))
        return P2M_E_INVALID;
    bool any = false;
    for (int m = 0; m < c->cfg.n_maps; ++m) any |= c->have_table[m];
    if (any && (memcmp(hdr_i, c->hdr_i, sizeof(c->hdr_i)) || memcmp(hdr_f, c->hdr_f, sizeof(c->hdr_f))))
        return P2M_E_SIZE;   /* all slots share one grid */
    HIPCHK(hipSetDevice(c->cfg.device));
    memcpy(c->hdr_i, hdr_i, sizeof(c->hdr_i));
    memcpy(c->hdr_f, hdr_f, sizeof(c->hdr_f));
    if (c->cfg.precision != P2M_PREC_PLAIN_FP64 && c->cfg.nside > 0) {
        /* the tiled painters stage the radial nodes in LDS: the default tile
         * shape must fit with this table; a shape set earlier that no longer
         * fits goes back to the library's choice */
        const int ml = c->cfg.precision == P2M_PREC_FP64 ? 1 : 2;
        const int mem = c->d_count != nullptr;
        if (p2m_tile_lds_bytes(ml, c->cfg.n_maps, 10, mem, hdr_i[2], 64) > 160 * 1024) return P2M_E_SIZE;
        if (c->tuned && c->log2w && p2m_tile_lds_bytes(ml, c->cfg.n_maps, c->log2w, mem, hdr_i[2], 64) > 160 * 1024)
            c->tuned = false;
    }
    TabGeom &g = c->g;
    g.nchit = hdr_i[0]; g.nmht = hdr_i[1]; g.nrt = hdr_i[2];
    g.chimint = hdr_f[0]; g.chimaxt = hdr_f[1]; g.mhmint = hdr_f[2]; g.mhmaxt = hdr_f[3];
    g.rmint = hdr_f[4]; g.rmaxt = hdr_f[5];
    /* maptable.f90:166-168 */
    g.dchit = (p2m_log(g.chimaxt) - p2m_log(g.chimint)) / (double)(g.nchit - 1);
    g.drt = (p2m_log(g.rmaxt) - p2m_log(g.rmint)) / (double)(g.nrt - 1);
    g.dmht = (p2m_log(g.mhmaxt) - p2m_log(g.mhmint)) / (double)(g.nmht - 1);
    g.lr0 = p2m_log(g.rmint); g.lc0 = p2m_log(g.chimint); g.lm0 = p2m_log(g.mhmint);
    /* padding covers every index interpolate_table can form past the end (Q6) */
    int64_t pad = 2LL * g.nrt * (g.nmht + 2) + 4LL * g.nrt + 64;
    /* the painters read the tables through buffer resources with 32-bit byte
     * offsets: one padded table, and the corner-quad table of all slots (16
     * bytes per map and node of each cell), must each stay below 2 GiB */
    if ((nt + pad) * 4 > INT32_MAX || (nt / 2) * 16 * c->cfg.n_maps > INT32_MAX) return P2M_E_SIZE;
    c->n_flat = nt + pad;
    if (!c->d_flat[slot] && grow(c, (void **)&c->d_flat[slot], sizeof(float) * c->n_flat)) return P2M_E_NOMEM;
    std::vector<float> flat(c->n_flat, 0.f);
    memcpy(flat.data(), table, sizeof(float) * nt);
    HIPCHK(hipMemcpy(c->d_flat[slot], flat.data(), sizeof(float) * c->n_flat, hipMemcpyHostToDevice));
    if (c->cfg.precision != P2M_PREC_PLAIN_FP64) {
        c->n_quad = (int64_t)g.nchit * g.nmht * g.nrt * 4 * c->cfg.n_maps;
        if (!c->d_quad && grow(c, (void **)&c->d_quad, sizeof(float) * c->n_quad)) return P2M_E_NOMEM;
        p2m_launch_build_quad(c->d_flat[slot], c->n_flat, c->cfg.profile, g.nrt, g.nmht, g.nchit, c->cfg.n_maps, slot,
                              c->d_quad, c->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(c->stream));
    }
    /* FP32 path constants: node radii, ln r -> cell coordinate */
    std::vector<float> invf(g.nrt + 2);
    for (int k = 0; k < g.nrt + 2; ++k) invf[k] = (float)p2m_exp(-2.0 * (g.lr0 + (double)k * g.drt));
    if (!c->d_inv_node2f && grow(c, (void **)&c->d_inv_node2f, sizeof(float) * (g.nrt + 2))) return P2M_E_NOMEM;
    HIPCHK(hipMemcpy(c->d_inv_node2f, invf.data(), sizeof(float) * (g.nrt + 2), hipMemcpyHostToDevice));
    c->u_k1 = (float)(0.5 * 0.6931471805599453 / g.drt);   /* log2(r^2) -> (ln r)/drt */
    c->u_k0 = (float)(g.lr0 / g.drt);
    c->u_max = (float)(g.nrt - 1);
    /* the FP32 cell coordinate carries log2's error times u_k1 (about 10 on
     * the standard grid): a finer radial grid widens the band in proportion,
     * and a band of half a cell or more sends every interior pixel to FP64 */
    c->u_band = std::max(2.5e-4f, 2.5e-5f * c->u_k1);
    {
        /* r < rmint is clamped to rmint + 1e-5 (maptable.f90:190); its cell
         * and fraction as interpolate_table forms them (:196, :200), in FP64 */
        const double lrc = p2m_log(g.rmint + 1e-5);
        c->ir_clamp = (int)((lrc - g.lr0) / g.drt) + 1;
        c->fr_clamp64 = lrc - (g.lr0 + (double)(c->ir_clamp - 1) * g.drt);
        c->fr_clamp = (float)c->fr_clamp64;
    }
    c->have_table[slot] = true;
    return 0;
}

int p2m_set_tile(p2m_ctx *c, int32_t tile_w, int32_t tile_wg)
{
    if (!c) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (tile_w == 0 && tile_wg == 0) { c->tuned = false; return 0; }
    if (!is_pow2(tile_w) || tile_w < 64 || tile_w > (1 << p2m_tile_max_log2w())) return P2M_E_INVALID;
    if (tile_wg < 64 || tile_wg > 512 || tile_wg % 64) return P2M_E_INVALID;
    if (c->cfg.precision == P2M_PREC_FP32_COMP && tile_wg > 256) return P2M_E_INVALID;
    int l = 0;
    while ((1 << l) < tile_w) ++l;
    if (p2m_tile_lds_bytes(c->cfg.precision == P2M_PREC_FP64 ? 1 : 2, c->cfg.n_maps, l, c->d_count != nullptr,
                           c->have_table[0] ? c->g.nrt : 200, 64) > 160 * 1024)
        return P2M_E_INVALID;
    HIPCHK(hipSetDevice(c->cfg.device));
    int rc = build_tiles(c, l);
    if (rc) return rc;
    c->wg = tile_wg;
    c->tuned = true;
    return 0;
}

}  /* extern "C" */

/* ------------------------------------------------------------------ paint */
/* exclusive scan of n uint32 counts into uint64 offsets, growing the temp storage */
static int scan_counts_on(const uint32_t *cnt, unsigned long long *off, int64_t n, void **tmp, size_t *tmp_bytes,
                          hipStream_t s)
{
    size_t need = 0;
    if (p2m_scan_u32(cnt, off, n, nullptr, &need, s)) return P2M_E_HIP;
    if (need > *tmp_bytes || !*tmp) {
        dfree(*tmp); *tmp = nullptr; *tmp_bytes = 0;
        if (dmalloc(tmp, need + 256)) return P2M_E_NOMEM;
        *tmp_bytes = need + 256;
    }
    size_t bytes = *tmp_bytes;
    if (p2m_scan_u32(cnt, off, n, *tmp, &bytes, s)) return P2M_E_HIP;
    return 0;
}

static int scan_counts(p2m_ctx *c, const uint32_t *cnt, unsigned long long *off, int64_t n)
{
    return scan_counts_on(cnt, off, n, &c->d_scan_tmp, &c->scan_tmp_bytes, c->stream);
}

/* counter block summed over its shards (blocks until the stream is idle) */
static int read_counters(p2m_ctx *c, unsigned long long out[Ctr::TOTAL], unsigned long long *raw = nullptr)
{
    unsigned long long *h = c->h_pin;
    HIPCHK(hipMemcpyAsync(h, c->d_ctr, sizeof(*h) * Ctr::ALL, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (raw) memcpy(raw, h, sizeof(*h) * Ctr::ALL);
    for (int k = 0; k < Ctr::TOTAL; ++k) {
        out[k] = 0;
        for (int sh = 0; sh < P2M_SHARDS; ++sh) out[k] += h[sh * Ctr::TOTAL + k];
    }
    return 0;
}

static int ensure_halo_cap(p2m_ctx *c, int64_t n)
{
    if (n <= c->halo_cap && c->d_halo) return 0;
    dfree(c->d_halo); c->d_halo = nullptr; c->halo_cap = 0;
    dfree(c->d_flat_idx); c->d_flat_idx = nullptr;
    dfree(c->d_n_pairs); c->d_n_pairs = nullptr;
    dfree(c->d_pair_off); c->d_pair_off = nullptr;
    dfree(c->d_hot); c->d_hot = nullptr;
    dfree(c->d_pair_halo); c->d_pair_halo = nullptr;
    int64_t cap = std::max<int64_t>(n, 1024);
    if (grow(c, (void **)&c->d_halo, sizeof(HaloRec) * cap)) return P2M_E_NOMEM;
    if (grow(c, (void **)&c->d_flat_idx, sizeof(uint32_t) * cap)) return P2M_E_NOMEM;
    if (c->cfg.precision != P2M_PREC_PLAIN_FP64 && c->cfg.nside > 0) {
        if (grow(c, (void **)&c->d_pair_halo, sizeof(PairHalo) * cap)) return P2M_E_NOMEM;
        if (grow(c, (void **)&c->d_n_pairs, sizeof(uint32_t) * (cap + 1))) return P2M_E_NOMEM;
        if (grow(c, (void **)&c->d_pair_off, sizeof(unsigned long long) * (cap + 1))) return P2M_E_NOMEM;
        if (c->cfg.precision == P2M_PREC_FP32_COMP && grow(c, (void **)&c->d_hot, sizeof(TileHalo) * cap))
            return P2M_E_NOMEM;
    }
    c->halo_cap = cap;
    return 0;
}

static int decode_chunk(p2m_ctx *c, const float *d_src, int64_t n, int64_t base)
{
    DecodeArgs a;
    a.halos = d_src; a.n = n; a.index_base = base; a.first = c->n_chunks++ == 0;
    a.c = c->cdev; a.g = c->g;
    a.cut_low = c->cut_low; a.cut_high = c->cut_high; a.chihview = c->run.chihview; a.mmin = c->run.mmin;
    a.precut = (c->run.flags & P2M_RUN_PRECUT) ? 1 : 0;
    a.dmodel = c->cfg.model == 2 ? 500.0 : 200.0;
    a.profile = c->cfg.profile; a.nside = c->cfg.nside; a.npix_fs = c->cfg.npix_fs;
    a.fov = ((c->cfg.fov_deg / 360.0) * 2.0) * c->mypi;        /* pks2map.f90:92 */
    a.dpix = c->cfg.npix_fs > 0 ? a.fov / (double)c->cfg.npix_fs : 1.0;
    a.out = c->d_halo; a.cap = c->halo_cap;
    a.flat_idx = c->d_flat_idx;
    a.flat_tiles = c->cfg.precision != P2M_PREC_PLAIN_FP64;
    a.cand = c->d_cand;
    a.n_cand = c->d_ctr + Ctr::N_CAND;
    a.n_cand0 = c->d_ctr + Ctr::N_CAND0;
    a.n_flat_out = c->d_ctr + Ctr::N_FLAT;
    a.counters = c->d_ctr + Ctr::DEC;
    a.hot = c->d_hot; a.pair_halo = c->d_pair_halo; a.n_pairs = c->d_n_pairs; a.shape = c->shape;
    p2m_launch_decode(a, c->stream);
    return hipGetLastError() == hipSuccess ? 0 : P2M_E_HIP;
}

static int autotune(p2m_ctx *c, int64_t n_halo, int64_t n_flat, unsigned long long n_pix);

static int launch_flat(p2m_ctx *c, int64_t n_flat, hipStream_t s);

/* the main stream waits for whatever the flat-sky stream has enqueued */
static void fs_join(p2m_ctx *c)
{
    if (hipEventRecord(c->ev_fs, c->fs_stream) == hipSuccess) (void)hipStreamWaitEvent(c->stream, c->ev_fs, 0);
    (void)hipGetLastError();
}

/* the painters' table arguments */
static void table_args(const p2m_ctx *c, TileArgs &t)
{
    t.n_maps = c->cfg.n_maps; t.profile = c->cfg.profile;
    t.g = c->g; t.n_flat = c->n_flat;
    t.u_k1 = c->u_k1; t.u_k0 = c->u_k0; t.u_max = c->u_max; t.band = c->u_band; t.fr_clamp = c->fr_clamp; t.ir_clamp = c->ir_clamp;
    t.band_c = (float)CHORD_BAND;
    t.inv_node2f = c->d_inv_node2f;
    t.inv_drt = 1.0 / c->g.drt; t.u_max64 = (double)(c->g.nrt - 1); t.fr_clamp64 = c->fr_clamp64;
    /* ln r is off by a few 1e-12 at most for discs above 1e-4 rad */
    t.band64 = std::max(1e-7, 1e-11 * t.inv_drt);
    t.n_quad = c->n_quad; t.tab_q = c->d_quad;
    for (int m = 0; m < c->cfg.n_maps; ++m) t.tab_flat[m] = c->d_flat[m];
}

/* Splitting of tiles with many pairs (k_tile_bounds) for a launch of `grid`
 * workgroups, and its storage.  A tile is split above the mean of the
 * workgroups, but not below twice the mean tile (an even sky is never split)
 * nor below 1024 pairs, about 10 us of a workgroup; a call of up to 4096 pairs
 * is not worth the second launch.  At most n_pairs / above tiles have more
 * than `above` pairs, at most `grid`, and their slices are fewer than twice as
 * many.  Without memory for it no tile is split.  (1e6 halos of a 10-degree
 * field, tile kernel: split above 512 / 1024 / 2048 pairs nside 512 0.19 / 0.12 /
 * 0.11 ms, nside 4096 0.98 / 0.99 / 1.03; 1e5 of a 1-degree field at nside 4096
 * 0.54 / 0.56 / 0.68.  Half or twice the mean of the workgroups: 4096 1.14, 1.11.) */
static SplitArgs split_args(p2m_ctx *c, unsigned long long n_pairs, int grid, size_t part_bytes)
{
    SplitArgs s;
    memset(&s, 0, sizeof(s));
    const unsigned long long above = std::max<unsigned long long>(
        1024, std::max<unsigned long long>((n_pairs + grid - 1) / grid, 2 * n_pairs / c->n_tiles));
    if (n_pairs <= 4096 || n_pairs <= above) return s;
    const size_t o_units = 256, o_state = o_units + sizeof(SplitUnit) * 2 * P2M_TQ_MAX,
                 o_part = o_state + sizeof(SplitState) * P2M_TQ_MAX;
    const size_t parts = (size_t)(n_pairs / above), bytes = o_part + parts * part_bytes;
    if (bytes > c->split_bytes) {
        dfree(c->d_split); c->d_split = nullptr; c->split_bytes = 0;
        const size_t cap = (bytes + bytes / 8 + 255) & ~(size_t)255;
        if (grow(c, (void **)&c->d_split, cap)) return s;
        c->split_bytes = cap;
        p2m_launch_fill_u32((uint32_t *)c->d_split, (int64_t)(cap / 4), 0u, c->stream);
    }
    s.above = (uint32_t)above;
    s.unit_cap = 2 * P2M_TQ_MAX; s.part_cap = (uint32_t)parts;
    s.n = (uint32_t *)c->d_split;
    s.units = (SplitUnit *)(c->d_split + o_units);
    s.state = (SplitState *)(c->d_split + o_state);
    s.part = c->d_split + o_part;
    return s;
}

/* n_pix: the pixels of the painted discs, about */
static int paint_halos(p2m_ctx *c, int64_t n_halo, int64_t n_flat, unsigned long long n_pix, bool allow_tune)
{
    const int mode = c->cfg.precision;
    unsigned long long *pc = c->d_ctr + Ctr::PAINT;
    c->last_fast = false;
    PaintArgs pa;
    memset(&pa, 0, sizeof(pa));
    pa.halos = c->d_halo; pa.n_halo = n_halo; pa.nside = c->cfg.nside; pa.npix_fs = c->cfg.npix_fs;
    pa.n_maps = c->cfg.n_maps; pa.profile = c->cfg.profile;
    pa.fov = ((c->cfg.fov_deg / 360.0) * 2.0) * c->mypi;
    pa.dpix = c->cfg.npix_fs > 0 ? pa.fov / (double)c->cfg.npix_fs : 1.0;
    pa.g = c->g; pa.n_flat = c->n_flat;
    for (int m = 0; m < c->cfg.n_maps; ++m) { pa.tab_flat[m] = c->d_flat[m]; pa.map64[m] = c->d_hp64[m]; pa.fs64[m] = c->d_fs64[m]; }
    pa.count = c->d_count; pa.hash = c->d_hash; pa.fs_count = c->d_fs_count; pa.fs_hash = c->d_fs_hash;
    pa.counters = pc;

    if (mode != P2M_PREC_PLAIN_FP64 && c->cfg.nside > 0 && !c->tuned) {
        /* tile shape first: the tuner's trials paint and clear both maps, so
         * this call's own painting (the flat-sky map included) starts after
         * the last trial */
        if (allow_tune) { int rc = autotune(c, n_halo, n_flat, n_pix); if (rc) return rc; }
        else { int rc = build_tiles(c, 10); if (rc) return rc; c->wg = 256; c->tuned = true; }
    }
    HIPCHK(hipEventRecord(c->ev[2], c->stream));
    if (mode == P2M_PREC_PLAIN_FP64) {
        if (c->cfg.nside > 0) p2m_launch_paint_plain_hp(pa, c->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipEventRecord(c->ev[3], c->stream));
        if (c->cfg.npix_fs > 0) p2m_launch_paint_fs(pa, c->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipEventRecord(c->ev[4], c->stream));
        HIPCHK(hipEventRecord(c->ev[5], c->stream));
        c->hp_zero = false;
        return 0;
    }
    if (c->cfg.nside > 0) {
        HIPCHK(hipEventRecord(c->ev_dec, c->stream));
        /* (halo, tile) pairs: counted by the decode at the shape it knew,
         * listed in halo order, sorted by tile */
        BinArgs b;
        memset(&b, 0, sizeof(b));
        b.halos = c->d_pair_halo; b.n_halo = n_halo; b.shape = c->shape; b.band_tile = c->d_band_tile;
        b.n_pairs = c->d_n_pairs; b.pair_off = c->d_pair_off; b.recs = c->d_halo; b.counters = pc;
        const bool recount = c->counted_log2w != c->log2w;
        if (recount) p2m_launch_pair_count(b, c->stream);
        if (n_halo > 0) { int rc = scan_counts(c, c->d_n_pairs, c->d_pair_off, n_halo + 1); if (rc) return rc; }
        if (recount && n_halo > 0) {
            HIPCHK(hipMemcpyAsync(c->h_pin, c->d_pair_off + n_halo, sizeof(*c->h_pin), hipMemcpyDeviceToHost, c->stream));
            HIPCHK(hipStreamSynchronize(c->stream));
            c->counted_pairs = *c->h_pin;
        }
        c->counted_log2w = c->log2w;
        const unsigned long long n_pairs = c->counted_pairs;
        if ((int64_t)n_pairs > c->pair_cap || !c->d_keys) {
            dfree(c->d_keys); c->d_keys = nullptr; c->d_vals = nullptr; c->pair_cap = 0;
            const int64_t cap = ((int64_t)(n_pairs * 1.125) + 1024 + 63) & ~(int64_t)63;
            if (grow(c, (void **)&c->d_keys, sizeof(uint32_t) * 4 * cap)) return P2M_E_NOMEM;
            c->d_vals = c->d_keys + 2 * cap;
            c->pair_cap = cap;
        }
        b.keys = c->d_keys; b.vals = c->d_vals; b.pair_cap = n_pairs;
        /* persistent grid of exactly the resident workgroups (a multiple
         * of 8 for the XCD-aware tile order): no partial last round */
        int grid = (int)std::min<int64_t>(c->n_tiles, P2M_TQ_MAX);
        const int wg = p2m_tile_wg(mode, c->cfg.n_maps, c->log2w, c->d_count != nullptr, c->g.nrt, c->wg);
        {
            const size_t lds = p2m_tile_lds_bytes(mode, c->cfg.n_maps, c->log2w, c->d_count != nullptr, c->g.nrt, wg);
            const int occ = p2m_tile_occupancy(mode, c->cfg.n_maps, wg, lds);
            if (occ > 0 && c->n_cu > 0) {
                const int64_t res = ((int64_t)occ * c->n_cu) & ~(int64_t)7;
                if (res >= 8) grid = (int)std::min<int64_t>(grid, res);
            }
        }
        const SplitArgs split = split_args(c, n_pairs, grid, (size_t)c->cfg.n_maps * ((size_t)8 << c->log2w) +
                                                             (c->d_count ? (size_t)12 << c->log2w : 0));
        b.n_split = split.n;
        if (n_pairs > 0) {
            if (c->ask_gaps) {
                /* in the place of the decode's count of such halos */
                p2m_launch_clear_ctr(pc, 3, 1, c->stream);
                p2m_launch_ring_gaps(b, c->stream);
            }
            p2m_launch_pair_emit(b, c->stream);
            size_t need = 0;
            if (p2m_sort_pairs(c->d_keys, c->d_vals, n_pairs, c->n_tiles, nullptr, &need, c->stream)) return P2M_E_HIP;
            if (need > c->sort_tmp_bytes || !c->d_sort_tmp) {
                dfree(c->d_sort_tmp); c->d_sort_tmp = nullptr; c->sort_tmp_bytes = 0;
                if (grow(c, &c->d_sort_tmp, need + 256)) return P2M_E_NOMEM;
                c->sort_tmp_bytes = need + 256;
            }
            size_t bytes = c->sort_tmp_bytes;
            if (p2m_sort_pairs(c->d_keys, c->d_vals, n_pairs, c->n_tiles, c->d_sort_tmp, &bytes, c->stream)) return P2M_E_HIP;
        }
        const uint32_t *keys = c->d_keys + n_pairs, *vals = c->d_vals + n_pairs;     /* sorted */
        p2m_launch_tile_bounds(keys, n_pairs, c->n_tiles, c->d_tile_off, split, c->d_ctr + Ctr::ERR, c->stream);
        HIPCHK(hipGetLastError());
        if (mode == P2M_PREC_FP32_COMP) {
            /* deferred FP64 pixels: ~5e-4 of the listed pixels in practice;
             * a list that fills up costs a repaint of the tiles that lost
             * pixels, after the list has grown (P2M_FB_CAP caps it, so that
             * the repaint can be exercised) */
            int64_t need = (int64_t)(n_pix / 256) + (1 << 18);
            if (const char *e = getenv("P2M_FB_CAP")) {
                const long long cap = atoll(e);
                if (cap >= P2M_SHARDS && cap < need) need = cap;
            }
            if (need != c->fb_cap && (need > c->fb_cap || getenv("P2M_FB_CAP"))) {
                dfree(c->d_fb); c->d_fb = nullptr; c->fb_cap = 0;
                if (grow(c, (void **)&c->d_fb, sizeof(uint4) * need)) return P2M_E_NOMEM;
                c->fb_cap = need;
            }
        }
        HIPCHK(hipEventRecord(c->ev[3], c->stream));
        TileArgs t;
        memset(&t, 0, sizeof(t));
        t.halos = c->d_halo; t.hot = c->d_hot; t.shape = c->shape; t.nside = c->cfg.nside;
        t.log2w = c->log2w;
        t.accumulate = c->hp_zero ? 0 : 1;
        t.n_tiles = c->n_tiles; t.desc = c->d_tile_desc; t.ring = c->d_ring; t.tile_off = c->d_tile_off;
        t.keys = keys; t.vals = vals;
        table_args(c, t);
        t.fb = c->d_fb; t.fb_count = pc + 6; t.fb_cap = c->fb_cap;
        t.lost = c->d_lost; t.tile_next = c->d_tile_next; t.split = split; t.redo = 0; t.n_halo = n_halo; t.err = c->d_ctr + Ctr::ERR; t.n_lost = c->d_ctr + Ctr::LOST;
        for (int m = 0; m < c->cfg.n_maps; ++m) {
            t.map64[m] = c->d_hp64[m]; t.map32[m] = c->d_hp32[m];
        }
        t.count = c->d_count; t.hash = c->d_hash; t.counters = pc;
        t.wide = 2 * n_pix > (n_pairs << (c->shape.log2r + c->shape.log2c));      /* half a tile a pair */
        t.vectors = p2m_exact_vectors(c->cfg.n_maps, c->log2w, c->d_count != nullptr, wg);
        c->last_wg = wg;
        if (p2m_launch_tile_paint(t, mode, c->cfg.n_maps, grid, wg, c->stream)) return P2M_E_INVALID;
        HIPCHK(hipGetLastError());
        HIPCHK(hipEventRecord(c->ev[7], c->stream));
        if (mode == P2M_PREC_FP32_COMP) {
            FallbackArgs f;
            memset(&f, 0, sizeof(f));
            f.halos = c->d_halo; f.fb = c->d_fb; f.fb_count = pc + 6; f.fb_cap = c->fb_cap;
            f.nside = c->cfg.nside; f.n_maps = c->cfg.n_maps; f.profile = c->cfg.profile;
            f.g = c->g; f.n_flat = c->n_flat;
            for (int m = 0; m < c->cfg.n_maps; ++m) { f.tab_flat[m] = c->d_flat[m]; f.map32[m] = c->d_hp32[m]; }
            f.count = c->d_count; f.hash = c->d_hash; f.counters = pc;
            f.lost = c->d_lost; f.desc = c->d_tile_desc; f.n_tiles = c->n_tiles; f.n_halo = n_halo;
            f.err = c->d_ctr + Ctr::ERR;
            if (p2m_launch_fallback(f, (int64_t)(n_pix / 256) + 1024, c->stream)) return P2M_E_HIP;
            c->last_t = t; c->last_f = f; c->last_grid = grid;
        }
        c->last_fast = mode == P2M_PREC_FP32_COMP;
        HIPCHK(hipEventRecord(c->ev[4], c->stream));
        /* the flat-sky painter needs only the decoded records: it runs on
         * its own stream beside the binning and the tile painter.  It is the
         * shorter chain of launches, so it is queued last: a small call's
         * painting does not wait for the host to have queued it */
        HIPCHK(hipStreamWaitEvent(c->fs_stream, c->ev_dec, 0));
        { int rc = launch_flat(c, n_flat, c->fs_stream); if (rc) { fs_join(c); return rc; } }
        HIPCHK(hipEventRecord(c->ev_fs, c->fs_stream));
        HIPCHK(hipStreamWaitEvent(c->stream, c->ev_fs, 0));
    } else {
        HIPCHK(hipEventRecord(c->ev[3], c->stream));
        HIPCHK(hipEventRecord(c->ev[4], c->stream));
        { int rc = launch_flat(c, n_flat, c->stream); if (rc) return rc; }
    }
    HIPCHK(hipEventRecord(c->ev[5], c->stream));
    c->hp_zero = false;
    return 0;
}

/* Most pairs of the flat-sky painter's list (2 GiB; P2M_FS_PAIRS sets fewer):
 * more are painted in parts of the halo list, as long as the decode's count of
 * all pairs makes them; a part that has more is counted again with half its
 * halos.  (Parts of most / n_tiles halos, as if every disc reached every tile:
 * 2e4 halos on 4096 x 4096 pixels with a list of 1e5 pairs 88 ms, now 0.87.) */
#define FS_MAX_PAIRS (1LL << 28)

/* flat-sky painter on stream s, between events 8 and 9 */
static int launch_flat(p2m_ctx *c, int64_t n_flat, hipStream_t s)
{
    HIPCHK(hipEventRecord(c->ev[8], s));
    if (c->cfg.npix_fs > 0 && n_flat > 0) {
        FlatArgs f;
        memset(&f, 0, sizeof(f));
        f.halos = c->d_halo; f.npix = c->cfg.npix_fs;
        f.fov = ((c->cfg.fov_deg / 360.0) * 2.0) * c->mypi;
        f.dpix = f.fov / (double)c->cfg.npix_fs;
        f.n_tiles = p2m_flat_tiles(f.npix, &f.nj);
        for (int m = 0; m < c->cfg.n_maps; ++m) f.map[m] = c->d_fs64[m];
        f.count = c->d_fs_count; f.hash = c->d_fs_hash; f.counters = c->d_ctr + Ctr::PAINT;
        TileArgs t;
        memset(&t, 0, sizeof(t));
        table_args(c, t);
        int64_t most = FS_MAX_PAIRS;
        const int64_t pairs = (int64_t)c->flat_pairs;
        if (const char *e = getenv("P2M_FS_PAIRS")) { if (atoll(e) > 0) most = atoll(e); }
        most = std::max(most, f.n_tiles);               /* room for any one halo's */
        if (!c->d_fs_cnt) {
            const int64_t cap = f.n_tiles * p2m_flat_slices(f.n_tiles, INT64_MAX) + 1;
            dfree(c->d_fs_off); c->d_fs_off = nullptr;
            if (grow(c, (void **)&c->d_fs_off, sizeof(unsigned long long) * cap)) return P2M_E_NOMEM;
            if (grow(c, (void **)&c->d_fs_cnt, sizeof(uint32_t) * cap)) return P2M_E_NOMEM;
            p2m_launch_fill_u32(c->d_fs_cnt, cap, 0u, s);
        }
        while (std::min(pairs, most) > c->fs_cap || !c->d_fs_pairs) {
            dfree(c->d_fs_pairs); c->d_fs_pairs = nullptr; c->fs_cap = 0;
            const int64_t want = std::min(pairs, most), cap = want + want / 8 + 1024;
            if (!grow(c, (void **)&c->d_fs_pairs, sizeof(uint2) * cap)) { c->fs_cap = cap; break; }
            if (want <= f.n_tiles) return P2M_E_NOMEM;
            most = std::max(want / 2, f.n_tiles);       /* in more parts */
        }
        const bool whole = pairs <= most;
        f.slices = p2m_flat_slices(f.n_tiles, std::min(pairs, most));
        const int64_t n_lists = f.n_tiles * f.slices;
        f.cnt = c->d_fs_cnt; f.off = c->d_fs_off; f.pairs = c->d_fs_pairs; f.pair_cap = (unsigned long long)c->fs_cap;
        int64_t part = whole ? n_flat : (int64_t)((double)n_flat * (double)most * 0.875 / (double)pairs);
        for (int64_t i = 0; i < n_flat; i += f.n_list) {
            part = std::max<int64_t>(part, 1);
            f.list = c->d_flat_idx + i; f.n_list = std::min(part, n_flat - i);
            f.first = i == 0;
            p2m_launch_flat_pairs(f, 0, s);
            {
                /* its own scan storage when beside the binning */
                const bool own = s != c->stream;
                int rc = scan_counts_on(c->d_fs_cnt, c->d_fs_off, n_lists + 1, own ? &c->d_scan_tmp_fs : &c->d_scan_tmp,
                                        own ? &c->scan_tmp_fs_bytes : &c->scan_tmp_bytes, s);
                if (rc) { p2m_launch_fill_u32(c->d_fs_cnt, n_lists + 1, 0u, s); return rc; }
            }
            if (!whole) {
                unsigned long long have = 0;
                hipError_t e = hipMemcpyAsync(&have, c->d_fs_off + n_lists, sizeof(have), hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipStreamSynchronize(s);
                if (e != hipSuccess || (int64_t)have > most) {
                    p2m_launch_fill_u32(c->d_fs_cnt, n_lists + 1, 0u, s);
                    if (e != hipSuccess) return hip_fail(e, "count of flat-sky pairs", __LINE__);
                    part = f.n_list / 2;
                    f.n_list = 0;
                    continue;
                }
            }
            p2m_launch_flat_pairs(f, 1, s);
            if (p2m_launch_flat_paint(t, f, s)) return P2M_E_INVALID;
        }
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(c->ev[9], s));
    return 0;
}

/* The FP32 painter's deferred-pixel list filled up in some sub-list: grow
 * it so that every sub-list holds the whole demand, and paint the tiles
 * marked lost again (they wrote nothing; entries they did store are skipped
 * by the fallback), then decide their deferred pixels.  Repeats until no
 * tile is lost; `raw` holds the counters on entry and on return. */
static int repaint_lost(p2m_ctx *c, unsigned long long h[Ctr::TOTAL], unsigned long long raw[Ctr::ALL])
{
    unsigned long long *pc = c->d_ctr + Ctr::PAINT;
    c->n_redo = 0;
    for (int iter = 0;; ++iter) {
        unsigned long long demand = 0;
        bool over = false;
        for (int sh = 0; sh < P2M_SHARDS; ++sh) {
            const unsigned long long v = raw[sh * Ctr::TOTAL + Ctr::PAINT + 6];
            demand += v;
            if ((int64_t)v > c->fb_cap / P2M_SHARDS) over = true;
        }
        if (!over) return 0;
        c->n_redo += (int)h[Ctr::LOST];
        if (iter >= 3) {
            /* cannot happen: the grown list holds every pass's whole demand */
            p2m_launch_fill_u32((uint32_t *)c->d_lost, (c->n_tiles + 3) / 4, 0u, c->stream);
            (void)hipStreamSynchronize(c->stream);
            snprintf(g_hip_detail, sizeof(g_hip_detail), "deferred-pixel list still full after %d repaints", iter);
            return P2M_E_NOMEM;
        }
        const int64_t cap = (int64_t)P2M_SHARDS * (int64_t)(demand + 64);
        dfree(c->d_fb); c->d_fb = nullptr; c->fb_cap = 0;
        if (grow(c, (void **)&c->d_fb, sizeof(uint4) * cap)) return P2M_E_NOMEM;
        c->fb_cap = cap;
        p2m_launch_clear_ctr(pc, 6, 1, c->stream);
        p2m_launch_clear_ctr(c->d_ctr, Ctr::LOST, 1, c->stream);
        TileArgs t = c->last_t;
        t.fb = c->d_fb; t.fb_cap = cap; t.redo = 1;
        if (p2m_launch_tile_paint(t, P2M_PREC_FP32_COMP, c->cfg.n_maps, c->last_grid, c->last_wg, c->stream))
            return P2M_E_INVALID;
        HIPCHK(hipGetLastError());
        FallbackArgs f = c->last_f;
        f.fb = c->d_fb; f.fb_cap = cap;
        if (p2m_launch_fallback(f, (int64_t)demand + 1024, c->stream)) return P2M_E_HIP;
        int rc = read_counters(c, h, raw);
        if (rc) return rc;
    }
}

static int finish_stats(p2m_ctx *c)
{
    unsigned long long h[Ctr::TOTAL], raw[Ctr::ALL];
    int rc = read_counters(c, h, raw);
    if (rc) return rc;
    c->n_redo = 0;
    if (c->last_fast) {
        rc = repaint_lost(c, h, raw);
        if (rc) return rc;
    }
    if (h[Ctr::ERR]) {
        snprintf(g_hip_detail, sizeof(g_hip_detail),
                 "%llu device-side range checks failed (pair, tile or deferred entry out of range)",
                 h[Ctr::ERR]);
        return P2M_E_INTERNAL;
    }
    p2m_stats &s = c->st;
    s.n_cut = (int64_t)h[Ctr::DEC + 0];
    s.n_radius_err = (int64_t)h[Ctr::DEC + 2];
    s.n_painted = (int64_t)h[Ctr::N_CAND] - s.n_radius_err;
    s.n_listed_hp = (int64_t)h[Ctr::PAINT + 0];
    s.n_upd_hp = (int64_t)h[Ctr::PAINT + 1];
    s.n_upd_fs = (int64_t)h[Ctr::PAINT + 2];
    s.n_ring_gaps = (int64_t)h[Ctr::PAINT + 3];
    s.n_segments = (int64_t)h[Ctr::PAINT + 4];
    s.n_fallback = (int64_t)h[Ctr::PAINT + 5];
    s.n_redo_tiles = c->n_redo;
    s.cut_low = c->cut_low; s.cut_high = c->cut_high;
    float ms = 0;
    (void)hipEventElapsedTime(&ms, c->ev[0], c->ev[5]); s.ms_total = ms;
    (void)hipEventElapsedTime(&ms, c->ev[0], c->ev[1]); s.ms_decode = ms;
    float ms_fs = 0;
    if (c->cfg.precision != P2M_PREC_PLAIN_FP64) (void)hipEventElapsedTime(&ms_fs, c->ev[8], c->ev[9]);
    /* the flat-sky painter of the tiled modes runs on its own stream beside
     * the binning: its time is reported as the finish phase */
    (void)hipEventElapsedTime(&ms, c->ev[2], c->ev[3]);
    s.ms_bin = ms;
    (void)hipEventElapsedTime(&ms, c->ev[3], c->ev[4]); s.ms_paint = ms;
    if (c->cfg.precision == P2M_PREC_PLAIN_FP64) { (void)hipEventElapsedTime(&ms, c->ev[4], c->ev[5]); s.ms_finish = ms; }
    else s.ms_finish = ms_fs;
    s.ms_tile = 0.0;
    if (c->cfg.precision != P2M_PREC_PLAIN_FP64 && c->cfg.nside > 0) {
        (void)hipEventElapsedTime(&ms, c->ev[3], c->ev[7]); s.ms_tile = ms;
    }
    s.tile_w = c->log2w ? (1 << c->log2w) : 0;
    /* as launched: fewer waves than set where no more fit (p2m_tile_wg) */
    s.tile_wg = c->cfg.precision != P2M_PREC_PLAIN_FP64 && c->cfg.nside > 0 ? c->last_wg : c->wg;
    return 0;
}

/* page-locked host memory (hipHostMalloc or otherwise pinned)? */
static bool host_is_pinned(const void *p)
{
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) { (void)hipGetLastError(); return false; }
    return at.type == hipMemoryTypeHost;
}

/* A catalogue pass is begin -> push (one or more blocks) -> finish.  begin
 * sizes the per-halo buffers for n_total halos and starts the call's clock;
 * push decodes a block, copying host blocks to the device in pieces on the
 * copy stream (two device slots used in turn, each piece decoded on the
 * painter's stream as soon as it has arrived); finish bins and paints. */
static int pass_begin(p2m_ctx *c, int64_t n_total)
{
    if (!c || n_total < 0) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (!c->have_run) return P2M_E_STATE;
    for (int m = 0; m < c->cfg.n_maps; ++m) if (!c->have_table[m]) return P2M_E_STATE;
    HIPCHK(hipSetDevice(c->cfg.device));
    int rc = ensure_halo_cap(c, n_total);
    if (rc) return rc;
    if (c->cfg.precision != P2M_PREC_PLAIN_FP64 && c->cfg.nside > 0) {
        /* the decode counts tiles at the shape in force, or at the default
         * one where the painter is still to choose */
        if (!c->tuned) { rc = build_tiles(c, 10); if (rc) return rc; }
        c->counted_log2w = c->log2w;
    }
    if (n_total > 0 && n_total > c->cand_cap) {
        dfree(c->d_cand); c->d_cand = nullptr; c->cand_cap = 0;
        if (grow(c, (void **)&c->d_cand, sizeof(uint32_t) * n_total)) return P2M_E_NOMEM;
        c->cand_cap = n_total;
    }
    p2m_launch_fill_u64(c->d_ctr, Ctr::ALL, c->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(c->ev[0], c->stream));
    c->in_stream = true;
    c->stream_total = n_total;
    c->stream_pushed = 0;
    c->stream_h2d_bytes = 0;
    c->n_host_push = 0;
    c->n_pieces = 0;
    c->n_chunks = 0;
    c->stream_pinned = true;
    return 0;
}

static int pass_push_impl(p2m_ctx *c, const float *src, bool on_device, int64_t n, int64_t index_base)
{
    if (n == 0) return 0;
    if (!on_device) {
        /* the previous host block's copies have finished: its buffer is the
         * caller's again (the double-buffer contract of p2m_stream_push) */
        if (c->n_host_push > 0) HIPCHK(hipEventSynchronize(c->ev_push));
        const bool pinned = host_is_pinned(src);
        c->stream_pinned = c->stream_pinned && pinned;
        /* pieces of 2^21 records (58.7 MB): long enough for the DMA engine's
         * full rate, short enough that the decode trails the copy closely */
        const int64_t piece = std::min<int64_t>(std::min<int64_t>(c->cfg.chunk_halos, 1 << 21), n);
        if (piece > c->slot_cap || !c->d_slot[0] || !c->d_slot[1]) {
            /* slots in use by an earlier piece are released only after the
             * painter's stream has passed them */
            HIPCHK(hipStreamSynchronize(c->stream));
            dfree(c->d_slot[0]); dfree(c->d_slot[1]);
            c->d_slot[0] = c->d_slot[1] = nullptr; c->slot_cap = 0;
            const int64_t cap = std::max<int64_t>(piece, 1 << 16);
            if (grow(c, (void **)&c->d_slot[0], sizeof(float) * 7 * cap)) return P2M_E_NOMEM;
            if (grow(c, (void **)&c->d_slot[1], sizeof(float) * 7 * cap)) return P2M_E_NOMEM;
            c->slot_cap = cap;
            c->n_pieces = 0;
        }
        /* copies start after the call's start mark, i.e. after every earlier
         * use of the slots on the painter's stream */
        if (c->n_host_push == 0) HIPCHK(hipStreamWaitEvent(c->h2d_stream, c->ev[0], 0));
        for (int64_t c0 = 0; c0 < n; c0 += piece) {
            const int64_t nc = std::min(piece, n - c0);
            const int slot = c->n_pieces & 1;
            if (c->n_pieces >= 2) HIPCHK(hipStreamWaitEvent(c->h2d_stream, c->ev_free[slot], 0));
            HIPCHK(hipMemcpyAsync(c->d_slot[slot], src + 7 * c0, sizeof(float) * 7 * nc, hipMemcpyHostToDevice,
                                  c->h2d_stream));
            HIPCHK(hipEventRecord(c->ev_copy[slot], c->h2d_stream));
            HIPCHK(hipStreamWaitEvent(c->stream, c->ev_copy[slot], 0));
            int rc = decode_chunk(c, c->d_slot[slot], nc, index_base + c0);
            if (rc) return rc;
            HIPCHK(hipEventRecord(c->ev_free[slot], c->stream));
            c->n_pieces++;
        }
        HIPCHK(hipEventRecord(c->ev_push, c->h2d_stream));
        c->stream_h2d_bytes += (int64_t)sizeof(float) * 7 * n;
        c->n_host_push++;
        return 0;
    }
    const int64_t chunk = c->cfg.chunk_halos;
    for (int64_t c0 = 0; c0 < n; c0 += chunk) {
        const int64_t nc = std::min(chunk, n - c0);
        int rc = decode_chunk(c, src + 7 * c0, nc, index_base + c0);
        if (rc) return rc;
    }
    return 0;
}

static int pass_push(p2m_ctx *c, const float *src, bool on_device, int64_t n, int64_t index_base)
{
    if (!c || n < 0 || (!src && n > 0) || index_base < 0) return P2M_E_INVALID;
    if (!c->in_stream) return P2M_E_STATE;
    if (n > c->stream_total - c->stream_pushed) return P2M_E_SIZE;
    HIPCHK(hipSetDevice(c->cfg.device));
    int rc = pass_push_impl(c, src, on_device, n, index_base);
    if (rc) {
        /* the pass is abandoned: wait for what was queued */
        (void)hipStreamSynchronize(c->h2d_stream);
        (void)hipStreamSynchronize(c->stream);
        c->in_stream = false;
        return rc;
    }
    c->stream_pushed += n;
    return 0;
}

static int pass_finish(p2m_ctx *c, bool allow_tune)
{
    if (!c) return P2M_E_INVALID;
    if (!c->in_stream) return P2M_E_STATE;
    c->in_stream = false;
    HIPCHK(hipSetDevice(c->cfg.device));
    if (c->n_host_push > 0) HIPCHK(hipEventRecord(c->ev_h2d_end, c->h2d_stream));
    HIPCHK(hipEventRecord(c->ev[1], c->stream));
    unsigned long long hc[Ctr::TOTAL];
    int rc = read_counters(c, hc);
    if (rc) return rc;
    int64_t n_halo = (int64_t)std::min<unsigned long long>(hc[Ctr::N_CAND], (unsigned long long)c->halo_cap);
    int64_t n_flat = (int64_t)std::min<unsigned long long>(hc[Ctr::N_FLAT], (unsigned long long)c->halo_cap);
    c->counted_pairs = hc[Ctr::PAIRS];
    c->flat_pairs = hc[Ctr::PAINT + 2];
    c->ask_gaps = hc[Ctr::GAPS] != 0;
    rc = paint_halos(c, n_halo, n_flat, hc[Ctr::PIX], allow_tune);
    if (rc) {
        /* nothing queued may outlive the call */
        (void)hipStreamSynchronize(c->fs_stream);
        (void)hipStreamSynchronize(c->stream);
        return rc;
    }
    c->hp_valid = true;
    c->st.n_in = c->stream_pushed;
    rc = finish_stats(c);
    if (rc) return rc;
    c->st.h2d_bytes = c->stream_h2d_bytes;
    c->st.h2d_pinned = c->n_host_push > 0 && c->stream_pinned ? 1 : 0;
    c->st.ms_h2d = 0.0;
    if (c->n_host_push > 0) {
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, c->ev[0], c->ev_h2d_end);
        c->st.ms_h2d = ms;
    }
    return 0;
}

static int paint_common(p2m_ctx *c, const float *src, bool on_device, int64_t n, int64_t index_base, bool allow_tune)
{
    if (!c || (!src && n > 0) || n < 0) return P2M_E_INVALID;
    int rc = pass_begin(c, n);
    if (rc) return rc;
    rc = pass_push(c, src, on_device, n, index_base);
    if (rc) return rc;
    return pass_finish(c, allow_tune);
}

extern "C" {

int p2m_paint(p2m_ctx *c, const float *halos, int64_t n, int64_t index_base)
{
    return paint_common(c, halos, false, n, index_base, true);
}

int p2m_paint_device(p2m_ctx *c, const float *d_halos, int64_t n, int64_t index_base)
{
    return paint_common(c, d_halos, true, n, index_base, true);
}

int p2m_stream_begin(p2m_ctx *c, int64_t n_total) { return pass_begin(c, n_total); }

int p2m_stream_push(p2m_ctx *c, const float *halos, int64_t n, int64_t index_base)
{
    return pass_push(c, halos, false, n, index_base);
}

int p2m_stream_finish(p2m_ctx *c) { return pass_finish(c, true); }

int p2m_host_alloc(p2m_ctx *c, int64_t bytes, void **ptr)
{
    if (!c || !ptr || bytes <= 0) return P2M_E_INVALID;
    *ptr = nullptr;
    HIPCHK(hipSetDevice(c->cfg.device));
    if (hipHostMalloc(ptr, (size_t)bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        *ptr = nullptr;
        return P2M_E_NOMEM;
    }
    return 0;
}

int p2m_host_free(p2m_ctx *c, void *ptr)
{
    if (!c) return P2M_E_INVALID;
    if (!ptr) return 0;
    HIPCHK(hipSetDevice(c->cfg.device));
    /* a block may still be read by a queued copy */
    HIPCHK(hipStreamSynchronize(c->h2d_stream));
    HIPCHK(hipHostFree(ptr));
    return 0;
}

int p2m_get_stats(p2m_ctx *c, p2m_stats *st)
{
    if (!c || !st) return P2M_E_INVALID;
    *st = c->st;
    return 0;
}

}  /* extern "C" */

/* What the painter's stream holds by now, then a copy to the caller's memory,
 * on the null stream: the copy engine of a context's own stream is chosen when
 * the stream is first used, and one that others have taken before copies at
 * half the rate (50 MB 0.93 ms or 1.94 ms; always 0.93 ms here). */
static int copy_out(p2m_ctx *c, void *dst, const void *src, size_t bytes)
{
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return 0;
}

/* A device map to host memory in the other precision: converted on the
 * device, 2^24 values at a time through a buffer that the context keeps, and
 * copied straight to the caller's memory; less at a time, or by the host, where
 * device memory is short.  (Copied to a host vector first and converted there,
 * a 4096 x 4096 flat map took 36 ms; 1.2 ms now, the copy.) */
namespace {
struct ConvertOps {
    p2m_ctx *c;
    char *dst;
    const char *src;
    bool to_double;
    size_t in() const { return to_double ? sizeof(float) : sizeof(double); }
    size_t out() const { return to_double ? sizeof(double) : sizeof(float); }
    bool buffer(int64_t k)
    {
        if (k <= c->conv_cap) return true;
        dfree(c->d_conv); c->d_conv = nullptr; c->conv_cap = 0;
        if (dmalloc(&c->d_conv, sizeof(double) * k)) return false;
        c->conv_cap = k;
        return true;
    }
    int on_device(int64_t i, int64_t k)
    {
        if (to_double) p2m_launch_f32_to_f64((const float *)src + i, (double *)c->d_conv, k, c->stream);
        else p2m_launch_f64_to_f32((const double *)src + i, (float *)c->d_conv, k, c->stream);
        HIPCHK(hipGetLastError());
        return copy_out(c, dst + out() * i, c->d_conv, out() * k);
    }
    int on_host(int64_t i, int64_t k)
    {
        void *h = malloc(in() * k);
        if (!h) return P2M_E_NOMEM;
        const int rc = copy_out(c, h, src + in() * i, in() * k);
        for (int64_t j = 0; !rc && j < k; ++j) {
            if (to_double) ((double *)dst)[i + j] = (double)((const float *)h)[j];
            else ((float *)dst)[i + j] = (float)((const double *)h)[j];
        }
        free(h);
        return rc;
    }
};
}  // namespace

/* A map of up to 256 KB is converted by the host: the launch and its wait take
 * longer (nside 8 to 32 to float 17 to 25 us, 35 to 42 through the device; nside 64
 * 32 and 30, to double 25 and 38). */
static int copy_converted(p2m_ctx *c, void *dst, const void *src, int64_t n, bool to_double)
{
    ConvertOps o = {c, (char *)dst, (const char *)src, to_double};
    if (n > 0 && (int64_t)o.in() * n <= 256 * 1024) return o.on_host(0, n);
    return convert_out(o, n, 1 << 24, 1 << 16);
}

static int fetch_map(p2m_ctx *c, const float *d32, const double *d64, int64_t n, float *h32, double *h64)
{
    if (n <= 0) return 0;
    int rc = 0;
    if (h32) rc = d64 ? copy_converted(c, h32, d64, n, false) : copy_out(c, h32, d32, sizeof(float) * n);
    if (!rc && h64) rc = d64 ? copy_out(c, h64, d64, sizeof(double) * n) : copy_converted(c, h64, d32, n, true);
    return rc;
}

extern "C" {

int p2m_fetch_maps(p2m_ctx *c, int slot, float *hp32, double *hp64, float *fs32, double *fs64)
{
    if (!c) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (slot < 0 || slot >= c->cfg.n_maps) return P2M_E_INVALID;
    HIPCHK(hipSetDevice(c->cfg.device));
    { int rc = ensure_hp_valid(c); if (rc) return rc; }
    int rc = fetch_map(c, c->d_hp32[slot], c->d_hp64[slot], c->hpnpix, hp32, hp64);
    if (!rc) rc = fetch_map(c, nullptr, c->d_fs64[slot], c->fsnpix, fs32, fs64);
    return rc;
}

int p2m_fetch_membership(p2m_ctx *c, uint32_t *hc, uint64_t *hh, uint32_t *fc, uint64_t *fh)
{
    if (!c) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (!(c->cfg.flags & P2M_FLAG_MEMBERSHIP)) return P2M_E_STATE;
    HIPCHK(hipSetDevice(c->cfg.device));
    { int rc = ensure_hp_valid(c); if (rc) return rc; }
    if (c->hpnpix > 0) {
        if (hc) HIPCHK(hipMemcpy(hc, c->d_count, sizeof(uint32_t) * c->hpnpix, hipMemcpyDeviceToHost));
        if (hh) HIPCHK(hipMemcpy(hh, c->d_hash, sizeof(uint64_t) * c->hpnpix, hipMemcpyDeviceToHost));
    }
    if (c->fsnpix > 0) {
        if (fc) HIPCHK(hipMemcpy(fc, c->d_fs_count, sizeof(uint32_t) * c->fsnpix, hipMemcpyDeviceToHost));
        if (fh) HIPCHK(hipMemcpy(fh, c->d_fs_hash, sizeof(uint64_t) * c->fsnpix, hipMemcpyDeviceToHost));
    }
    return 0;
}

}  /* extern "C" */

/* ------------------------------------------------------------------ autotuner */
/* Times the binning + tile paint for each candidate tile shape on the
 * halos already decoded, keeps the fastest, and restores the maps. */
static int autotune(p2m_ctx *c, int64_t n_halo, int64_t n_flat, unsigned long long n_pix)
{
    static const int cand[][2] = {{9, 256}, {10, 256}, {11, 256}, {11, 128}};
    int mode_ld = c->cfg.precision == P2M_PREC_FP64 ? 1 : 2;
    int best_l = 10, best_wg = 256;
    /* small problems: the default shape */
    if (n_halo < 200000 || getenv("P2M_NO_AUTOTUNE")) {
        int rc = build_tiles(c, best_l); if (rc) return rc;
        c->wg = best_wg; c->tuned = true;
        return 0;
    }
    /* tune on a copy of the maps' state: paint into the maps, then clear
     * (the call that triggers tuning starts from the maps' current state,
     * so remember whether they were zero and re-zero after each trial) */
    bool was_zero = c->hp_zero;
    if (!was_zero) {
        int rc = build_tiles(c, best_l); if (rc) return rc;
        c->wg = best_wg; c->tuned = true;
        return 0;
    }
    float best_ms = 1e30f;
    int tried_l = 0, tried_wg = 0;
    for (auto &cd : cand) {
        if (p2m_tile_lds_bytes(mode_ld, c->cfg.n_maps, cd[0], c->d_count != nullptr, c->g.nrt, 64) > 160 * 1024) continue;
        /* the workgroup that would be launched; the same as the last trial's
         * where LDS holds no more waves */
        const int wg = p2m_tile_wg(mode_ld, c->cfg.n_maps, cd[0], c->d_count != nullptr, c->g.nrt, cd[1]);
        if (cd[0] == tried_l && wg == tried_wg) continue;
        tried_l = cd[0]; tried_wg = wg;
        int rc = build_tiles(c, cd[0]); if (rc) return rc;
        c->wg = wg; c->tuned = true;
        c->hp_zero = true;
        /* each trial starts from zero paint counters, as a call does: the
         * deferred-pixel and overflow lists are appended at their counters */
        p2m_launch_clear_ctr(c->d_ctr, Ctr::PAINT, Ctr::TOTAL - Ctr::PAINT, c->stream);
        rc = paint_halos(c, n_halo, n_flat, n_pix, false);
        if (rc == P2M_E_INVALID) {
            /* a shape the painter rejects at launch, before the trial's
             * flat-sky paint is queued */
            (void)p2m_clear(c);
            continue;
        }
        if (rc) return rc;
        HIPCHK(hipStreamSynchronize(c->stream));
        float ms = 0;
        (void)hipEventElapsedTime(&ms, c->ev[2], c->ev[4]);
        if (ms < best_ms) { best_ms = ms; best_l = cd[0]; best_wg = wg; }
        rc = p2m_clear(c); if (rc) return rc;
        /* a trial's tiles that lost deferred pixels are not repainted: the
         * maps are cleared anyway, and so are the marks */
        p2m_launch_fill_u32((uint32_t *)c->d_lost, (c->n_tiles + 3) / 4, 0u, c->stream);
    }
    /* counters were polluted by the trials: reset the paint counters */
    p2m_launch_clear_ctr(c->d_ctr, Ctr::PAINT, Ctr::TOTAL - Ctr::PAINT, c->stream);
    p2m_launch_clear_ctr(c->d_ctr, Ctr::LOST, 1, c->stream);
    int rc = build_tiles(c, best_l); if (rc) return rc;
    c->wg = best_wg; c->tuned = true; c->hp_zero = true;
    return 0;
}

/* ------------------------------------------------------------------ products + writers */

/* Moments, RMS and dP/dy of one slot's maps, each map read once; the sums
 * and the histogram go through `scratch` (P2M_PROD_BYTES of device memory)
 * and one pinned copy, with one wait for the painter's stream. */
static int products(p2m_ctx *c, int slot, char *scratch, double moments[6], double rms[2], float *dpdy)
{
    if (!c) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (slot < 0 || slot >= c->cfg.n_maps) return P2M_E_INVALID;
    HIPCHK(hipSetDevice(c->cfg.device));
    { int rc = ensure_hp_valid(c); if (rc) return rc; }
    char *h = c->h_prod;
    unsigned long long *d_hist = (unsigned long long *)scratch;
    double *d_part = (double *)(scratch + P2M_PROD_PART_OFF);
    const float dy = 1e-4f / (float)P2M_NDPDY;                 /* pks2map.f90:39-40 */
    const int64_t n[2] = {c->fsnpix, c->hpnpix};
    const char *hpart[2] = {h + P2M_PROD_BYTES, h + P2M_PROD_PART_OFF};
    if (n[0] > 0) {
        p2m_launch_moments(nullptr, c->d_fs64[slot], n[0], d_part, nullptr, P2M_NDPDY, dy, c->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(h + P2M_PROD_BYTES, d_part, P2M_PROD_PART_BYTES, hipMemcpyDeviceToHost, c->stream));
    }
    if (n[1] > 0) {
        /* the scratch keeps the last call's contents: cleared by a fill kernel */
        if (dpdy) p2m_launch_fill_u64(d_hist, P2M_NDPDY, c->stream);
        p2m_launch_moments(c->d_hp32[slot], c->d_hp64[slot], n[1], d_part, dpdy ? d_hist : nullptr, P2M_NDPDY, dy,
                           c->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(h, scratch, P2M_PROD_BYTES, hipMemcpyDeviceToHost, c->stream));
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    double res[2][4] = {{0}};
    for (int which = 0; which < 2; ++which) {
        if (n[which] <= 0) continue;
        const double *p = (const double *)hpart[which];
        const int64_t chunk = p2m_moments_chunk(n[which]);
        const int64_t nb = (n[which] + chunk - 1) / chunk;
        const double dn = (double)n[which];
        double s[3] = {0, 0, 0};
        for (int64_t b = 0; b < nb; ++b)
            for (int k = 0; k < 3; ++k) s[k] += p[b * P2M_MOM_PART + k];
        const double mean = s[0] / dn;
        double sq = 0.0;
        for (int64_t b = 0; b < nb; ++b) {
            const double cnt = (double)(b + 1 < nb ? chunk : n[which] - b * chunk);
            const double d = p[b * P2M_MOM_PART + 3] - mean;
            sq += p[b * P2M_MOM_PART + 4] + cnt * (d * d);
        }
        for (int k = 0; k < 3; ++k) res[which][k] = s[k] / dn;
        res[which][3] = p2m_sqrt(sq / dn);
    }
    if (n[1] > 0 && dpdy) {
        /* dpdy = dpdy / real(hpnpix); cumulative, in float and in order (pks2map.f90:347, 355-357) */
        const unsigned long long *hist = (const unsigned long long *)h;
        for (int i = 0; i < P2M_NDPDY; ++i) dpdy[i] = (float)hist[i] / (float)n[1];
        for (int i = 1; i < P2M_NDPDY; ++i) dpdy[i] = dpdy[i - 1] + dpdy[i];
    }
    if (moments) { for (int k = 0; k < 3; ++k) { moments[k] = res[0][k]; moments[3 + k] = res[1][k]; } }
    if (rms) { rms[0] = res[0][3]; rms[1] = res[1][3]; }
    return 0;
}

extern "C" {

int p2m_products(p2m_ctx *c, int slot, double moments[6], double rms[2], float dpdy[10000])
{
    if (!c) return P2M_E_INVALID;
    return products(c, slot, c->d_prod, moments, rms, dpdy);
}

/* The same in this device's process-wide scratch array; calls that overlap
 * on one GPU share that array and race. */
int p2m_products_noalloc(p2m_ctx *c, int slot, double moments[6], double rms[2], float dpdy[10000])
{
    if (!c) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (slot < 0 || slot >= c->cfg.n_maps) return P2M_E_INVALID;
    HIPCHK(hipSetDevice(c->cfg.device));
    void *base = nullptr;
    { int rc = scratch_for_device(c->cfg.device, &base); if (rc) return rc; }
    return products(c, slot, (char *)base, moments, rms, dpdy);
}

}  /* extern "C" */

/* FITS card helpers (FITS standard 4.0, sec. 4.2) */
static std::string card(const char *key, const std::string &val, const char *comment)
{
    char b[81];
    std::string s;
    if (val.empty()) {
        snprintf(b, sizeof(b), "%-80s", key);
        return std::string(b, 80);
    }
    snprintf(b, sizeof(b), "%-8s= %20s / %s", key, val.c_str(), comment ? comment : "");
    s = b;
    s.resize(80, ' ');
    return s;
}
static std::string sval(const char *v)
{
    std::string s = "'";
    s += v;
    while (s.size() < 9) s += ' ';
    s += "'";
    while (s.size() < 20) s += ' ';
    return s;
}
static std::string ival(long long v) { char b[32]; snprintf(b, sizeof(b), "%lld", v); return b; }

static bool write_block(FILE *f, const std::vector<std::string> &cards)
{
    std::string txt;
    for (auto &c : cards) txt += c;
    std::string end = "END";
    end.resize(80, ' ');
    txt += end;
    txt.resize(((txt.size() + 2879) / 2880) * 2880, ' ');
    return fwrite(txt.data(), 1, txt.size(), f) == txt.size();
}

/* HEALPix map as FITS BINTABLE (fits_s_inc.f90:787-960 via cfitsio in the
 * reference; the same HDU structure and keywords written directly).  The map
 * streams from the device in pieces of 2^24 pixels through two page-locked
 * buffers: the copy of piece k+1 runs while piece k is byte-swapped to
 * big-endian and written, as the reference writes its rows piece by piece
 * (fits_s_inc.f90:921-933).  An FP64 map is rounded to float on the device
 * first (the reference's map is real). */
static int write_fits_dev(p2m_ctx *c, int slot, const char *path)
{
    const int64_t npix = c->hpnpix;
    const int32_t nside = c->cfg.nside;
    int64_t repeat = 1024;
    if (npix < 1024) repeat = 1;
    if (nside > 1024 * 256) repeat = nside / 256;
    int64_t nrows = npix / repeat;
    char date[32];
    time_t t = time(nullptr);
    struct tm tmv;
    gmtime_r(&t, &tmv);
    strftime(date, sizeof(date), "%Y-%m-%d", &tmv);
    std::vector<std::string> prim = {
        card("SIMPLE", "T", "file does conform to FITS standard"),
        card("BITPIX", ival(32), "number of bits per data pixel"),
        card("NAXIS", ival(0), "number of data axes"),
        card("EXTEND", "T", "FITS dataset may contain extensions"),
        card("DATE", sval(date), "file creation date (YYYY-MM-DD)")};
    char tform[32];
    snprintf(tform, sizeof(tform), "%lldE", (long long)repeat);
    std::vector<std::string> ext = {
        card("XTENSION", sval("BINTABLE"), "binary table extension"),
        card("BITPIX", ival(8), "8-bit bytes"),
        card("NAXIS", ival(2), "2-dimensional binary table"),
        card("NAXIS1", ival(4 * repeat), "width of table in bytes"),
        card("NAXIS2", ival(nrows), "number of rows in table"),
        card("PCOUNT", ival(0), "size of special data area"),
        card("GCOUNT", ival(1), "one data group (required keyword)"),
        card("TFIELDS", ival(1), "number of fields in each row"),
        card("TTYPE1", sval("simulation"), "label for field   1"),
        card("TFORM1", sval(tform), "data format of field: 4-byte REAL"),
        card("NSIDE", ival(nside), "the nside of the map"),
        card("ORDERING", sval("RING"), "the nside of the map")};
    const int64_t piece = std::min<int64_t>(npix, 1 << 24);
    float *hb[2] = {nullptr, nullptr};
    float *d32 = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    FILE *f = nullptr;
    int rc = 0;
    if (hipHostMalloc((void **)&hb[0], sizeof(float) * piece, hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc((void **)&hb[1], sizeof(float) * piece, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        rc = P2M_E_NOMEM;
    }
    if (!rc && c->d_hp64[slot] && grow(c, (void **)&d32, sizeof(float) * 2 * piece)) rc = P2M_E_NOMEM;
    if (!rc && (hipEventCreateWithFlags(&ev[0], hipEventDisableTiming) != hipSuccess ||
                hipEventCreateWithFlags(&ev[1], hipEventDisableTiming) != hipSuccess)) {
        (void)hipGetLastError();
        rc = P2M_E_HIP;
    }
    if (!rc) {
        f = fopen(path, "wb");
        if (!f) rc = P2M_E_IO;
    }
    bool ok = !rc && write_block(f, prim) && write_block(f, ext);
    if (!rc && !ok) rc = P2M_E_IO;
    const int64_t npieces = (npix + piece - 1) / piece;
    auto enqueue = [&](int64_t k) -> int {
        const int64_t i0 = k * piece, nk = std::min(piece, npix - i0);
        const int bslot = (int)(k & 1);
        const float *src = c->d_hp32[slot] + (c->d_hp32[slot] ? i0 : 0);
        if (c->d_hp64[slot]) {
            p2m_launch_f64_to_f32(c->d_hp64[slot] + i0, d32 + bslot * piece, nk, c->stream);
            src = d32 + bslot * piece;
        }
        if (hipMemcpyAsync(hb[bslot], src, sizeof(float) * nk, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
            hipEventRecord(ev[bslot], c->stream) != hipSuccess) {
            (void)hipGetLastError();
            return P2M_E_HIP;
        }
        return 0;
    };
    if (!rc && npieces > 0) rc = enqueue(0);
    for (int64_t k = 0; !rc && k < npieces; ++k) {
        if (k + 1 < npieces) rc = enqueue(k + 1);
        if (rc) break;
        const int bslot = (int)(k & 1);
        if (hipEventSynchronize(ev[bslot]) != hipSuccess) { (void)hipGetLastError(); rc = P2M_E_HIP; break; }
        const int64_t nk = std::min(piece, npix - k * piece);
        uint32_t *u = reinterpret_cast<uint32_t *>(hb[bslot]);
        for (int64_t j = 0; j < nk; ++j) u[j] = __builtin_bswap32(u[j]);
        if (fwrite(u, 4, (size_t)nk, f) != (size_t)nk) rc = P2M_E_IO;
        /* the buffer is refilled by the copy enqueued two pieces later, after
         * this write has returned */
    }
    if (!rc) {
        int64_t bytes = npix * 4, pad = (2880 - bytes % 2880) % 2880;
        std::vector<char> z(pad, 0);
        if (pad && fwrite(z.data(), 1, pad, f) != (size_t)pad) rc = P2M_E_IO;
    }
    (void)hipStreamSynchronize(c->stream);
    if (f && fclose(f) != 0 && !rc) rc = P2M_E_IO;
    if (rc && f) remove(path);
    for (int i = 0; i < 2; ++i) {
        if (hb[i]) (void)hipHostFree(hb[i]);
        if (ev[i]) (void)hipEventDestroy(ev[i]);
    }
    dfree(d32);
    return rc;
}

extern "C" int p2m_write_outputs(p2m_ctx *c, int slot, const char *base, int write_fs, int write_hp, int write_dp)
{
    if (!c || !base) return P2M_E_INVALID;
    if (c->in_stream) return P2M_E_STATE;
    if (slot < 0 || slot >= c->cfg.n_maps) return P2M_E_INVALID;
    std::string b(base);
    int rc = 0;
    if (write_dp && c->hpnpix > 0) {
        std::vector<float> dpdy(10000);
        rc = p2m_products(c, slot, nullptr, nullptr, dpdy.data());
        if (rc) return rc;
        std::string p = b + "_dp.bin";
        FILE *f = fopen(p.c_str(), "wb");
        if (!f) return P2M_E_IO;
        int32_t nd = 10000;
        float mx = 1e-4f;
        bool ok = fwrite(&nd, 4, 1, f) == 1 && fwrite(&mx, 4, 1, f) == 1 && fwrite(dpdy.data(), 4, 10000, f) == 10000;
        if (fclose(f) != 0) ok = false;
        if (!ok) { remove(p.c_str()); return P2M_E_IO; }
    }
    if (write_fs && c->fsnpix > 0) {
        std::vector<float> m(c->fsnpix);
        rc = p2m_fetch_maps(c, slot, nullptr, nullptr, m.data(), nullptr);
        if (rc) return rc;
        std::string p = b + "_fs.map";
        FILE *f = fopen(p.c_str(), "wb");
        if (!f) return P2M_E_IO;
        int32_t np = c->cfg.npix_fs;
        float fov = (float)(((c->cfg.fov_deg / 360.0) * 2.0) * c->mypi);
        bool ok = fwrite(&np, 4, 1, f) == 1 && fwrite(&np, 4, 1, f) == 1 && fwrite(&fov, 4, 1, f) == 1 &&
                  fwrite(&fov, 4, 1, f) == 1 && fwrite(m.data(), 4, (size_t)c->fsnpix, f) == (size_t)c->fsnpix;
        if (fclose(f) != 0) ok = false;
        if (!ok) { remove(p.c_str()); return P2M_E_IO; }
    }
    if (write_hp && c->hpnpix > 0) {
        HIPCHK(hipSetDevice(c->cfg.device));
        rc = ensure_hp_valid(c);
        if (rc) return rc;
        std::string p = b + "_hp.fits";
        rc = write_fits_dev(c, slot, p.c_str());
        if (rc) return rc;
    }
    return 0;
}

extern "C" int p2m_selftest_math(int32_t device, int32_t op, const double *x, const double *y, double *out, int64_t n)
{
    if (!x || !out || n < 0 || op < 0 || op > 9) return P2M_E_INVALID;
    if ((op == 6 || op == 9) && !y) return P2M_E_INVALID;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) { (void)hipGetLastError(); return P2M_E_NODEVICE; }
    if (device < 0 || device >= ndev) return P2M_E_INVALID;
    HIPCHK(hipSetDevice(device));
    if (n == 0) return 0;
    double *dx = nullptr, *dy = nullptr, *dout = nullptr;
    size_t b = sizeof(double) * (size_t)n;
    int rc = dmalloc((void **)&dx, b);
    if (!rc && y) rc = dmalloc((void **)&dy, b);
    if (!rc) rc = dmalloc((void **)&dout, b);
    if (!rc && hipMemcpy(dx, x, b, hipMemcpyHostToDevice) != hipSuccess) rc = P2M_E_HIP;
    if (!rc && y && hipMemcpy(dy, y, b, hipMemcpyHostToDevice) != hipSuccess) rc = P2M_E_HIP;
    if (!rc && p2m_launch_selftest_math(op, dx, dy, dout, n, 0)) rc = P2M_E_HIP;
    if (!rc && hipDeviceSynchronize() != hipSuccess) rc = P2M_E_HIP;
    if (!rc && hipMemcpy(out, dout, b, hipMemcpyDeviceToHost) != hipSuccess) rc = P2M_E_HIP;
    dfree(dx); dfree(dy); dfree(dout);
    (void)hipGetLastError();
    return rc;
}

extern "C" int p2m_selftest_copy(int32_t device, int64_t n_bytes, int32_t reps, double *ms)
{
    if (n_bytes <= 0 || n_bytes % 16 || n_bytes > (1LL << 34) || reps <= 0 || !ms) return P2M_E_INVALID;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) { (void)hipGetLastError(); return P2M_E_NODEVICE; }
    if (device < 0 || device >= ndev) return P2M_E_INVALID;
    HIPCHK(hipSetDevice(device));
    void *a = nullptr, *b = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = dmalloc(&a, (size_t)n_bytes);
    if (!rc) rc = dmalloc(&b, (size_t)n_bytes);
    if (!rc && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)) rc = P2M_E_HIP;
    if (!rc) {
        p2m_launch_fill_f32((float *)a, n_bytes / 4, 0);
        if (p2m_launch_copy_calib(a, b, n_bytes / 16, 0)) rc = P2M_E_HIP;      /* warm-up */
    }
    if (!rc && hipEventRecord(e0, 0) != hipSuccess) rc = P2M_E_HIP;
    for (int r = 0; r < reps && !rc; ++r)
        if (p2m_launch_copy_calib(a, b, n_bytes / 16, 0)) rc = P2M_E_HIP;
    if (!rc && hipEventRecord(e1, 0) != hipSuccess) rc = P2M_E_HIP;
    if (!rc && hipEventSynchronize(e1) != hipSuccess) rc = P2M_E_HIP;
    float t = 0.f;
    if (!rc && hipEventElapsedTime(&t, e0, e1) != hipSuccess) rc = P2M_E_HIP;
    if (!rc) *ms = (double)t / reps;
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    dfree(a); dfree(b);
    (void)hipGetLastError();
    return rc;
}
