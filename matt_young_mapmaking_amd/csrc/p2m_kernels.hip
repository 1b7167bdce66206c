/*
 * p2m_kernels.hip -- gfx950 kernels of the halo->map painter.
 *
 *  k_cull, k_setup   catalogue decode: radial and mass cuts over every record,
 *                    then the FP64 per-halo setup of the survivors
 *                    (pks2map.f90:144-160, 264, 284-298; haloproject.f90:47-55,
 *                    93-128; maptable.f90:184-202; query_disc prologue)
 *  k_pair_count, k_pair_emit, k_tile_bounds
 *                    (halo, tile) pairs of the painted halos, radix-sorted by
 *                    tile: tiles are 16 rings by a sector of azimuth
 *  k_tile_fast       FP32 painter: workgroups take tiles from a queue per
 *                    XCD, their waves the halos' pixel runs on the tile's rings
 *                    (pix_tools.F90:712-800, pixel_routines.F90:1823-1879);
 *                    per pixel the FP32 chord^2 test and profile value,
 *                    summed in an FP64 LDS tile and written once as FP32;
 *                    pixels near a disc edge or a table-cell edge go to
 *  k_fallback        the exact FP64 decision and value (haloproject.f90:60-75,
 *                    maptable.f90:176-216)
 *  k_tile_exact      FP64 painter over the same tiles, the reference's
 *                    arithmetic where it decides, FP64 LDS tile
 *  k_paint_plain_hp  baseline: one work item per halo, naive query_disc loop,
 *                    pix2vec_ring/angdist/interpolate_table per pixel, FP64
 *                    global atomics (haloproject.f90:55-75)
 *  k_fs_pairs, k_fs_paint, k_paint_fs
 *                    flat-sky painter over (halo, tile) pairs; one work item
 *                    per halo for the baseline (haloproject.f90:136-152)
 *  k_moments         map moments and the dP/dy histogram (pks2map.f90:321-357)
 */
#include "p2m_kernels.h"
#include "p2m_fast64.h"

#include <hipcub/hipcub.hpp>
#include <type_traits>

/* ===================================================================== */
/* helpers                                                                */
/* ===================================================================== */

__device__ static inline double dbl_of(uint32_t lo, uint32_t hi)
{
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

/* Loaded words that the code below needs on every path: an empty asm that
 * uses them, so that the compiler issues their loads together here instead
 * of moving each behind the branch that first uses it (a memory round trip
 * per branch). */
__device__ static inline void pin4(uint4 v)
{
    asm volatile("" ::"v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w));
}

__global__ void k_fill_u32(uint32_t *p, int64_t n, uint32_t v)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_fill_u64(unsigned long long *p, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0ULL;
}
__global__ void k_fill_f64(double *p, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0.0;
}
__global__ void k_fill_f32(float *p, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0.0f;
}

static inline int fill_grid(int64_t n) { int64_t g = (n + 255) / 256; return (int)(g < 16384 ? (g < 1 ? 1 : g) : 16384); }

void p2m_launch_fill_u32(uint32_t *p, int64_t n, uint32_t v, hipStream_t s) { if (n > 0) hipLaunchKernelGGL(k_fill_u32, dim3(fill_grid(n)), dim3(256), 0, s, p, n, v); }
void p2m_launch_fill_u64(unsigned long long *p, int64_t n, hipStream_t s) { if (n > 0) hipLaunchKernelGGL(k_fill_u64, dim3(fill_grid(n)), dim3(256), 0, s, p, n); }
void p2m_launch_fill_f64(double *p, int64_t n, hipStream_t s) { if (n > 0) hipLaunchKernelGGL(k_fill_f64, dim3(fill_grid(n)), dim3(256), 0, s, p, n); }
__global__ void k_clear_ctr(unsigned long long *ctr, int first, int count)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < P2M_SHARDS * count) ctr[(t / count) * P2M_CTR_STRIDE + first + t % count] = 0ULL;
}

void p2m_launch_clear_ctr(unsigned long long *ctr, int first, int count, hipStream_t s)
{
    if (count > 0) hipLaunchKernelGGL(k_clear_ctr, dim3((P2M_SHARDS * count + 255) / 256), dim3(256), 0, s, ctr, first, count);
}

void p2m_launch_fill_f32(float *p, int64_t n, hipStream_t s) { if (n > 0) hipLaunchKernelGGL(k_fill_f32, dim3(fill_grid(n)), dim3(256), 0, s, p, n); }

/* wave-aggregated append: returns the slot of this lane (or garbage if !take) */
__device__ static inline unsigned long long wave_append(unsigned long long *counter, bool take)
{
    unsigned long long mask = __ballot(take);
    int lane = __lane_id();
    int leader = __ffsll((long long)mask) - 1;
    unsigned long long base = 0;
    if (mask == 0) return 0;
    if (lane == leader) base = atomicAdd(counter, (unsigned long long)__popcll(mask));
    base = __shfl(base, leader);
    unsigned long long below = lane == 0 ? 0ULL : (mask & ((~0ULL) >> (64 - lane)));
    return base + (unsigned long long)__popcll(below);
}

__device__ static inline void wave_count(unsigned long long *counter, unsigned long long v)
{
    /* sum v over the wave, one atomic into this wave's shard of a statistics counter */
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    const unsigned shard = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) % P2M_SHARDS;
    if (__lane_id() == 0 && v) atomicAdd(counter + shard * P2M_CTR_STRIDE, v);
}

/* sum v over the workgroup, one atomic per workgroup into its shard of a
 * statistics counter; every thread calls */
__device__ static inline void block_count(unsigned long long *counter, unsigned long long v, unsigned long long *lds16)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    int wv = threadIdx.x >> 6;
    __syncthreads();
    if (__lane_id() == 0) lds16[wv] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) t += lds16[k];
        if (t) atomicAdd(counter + (blockIdx.x % P2M_SHARDS) * P2M_CTR_STRIDE, t);
    }
}

/* Inclusive prefix sum over the 64 lanes of a wave in registers: DPP row
 * shifts by 1, 2, 4 and 8 scan each row of 16 lanes, then row broadcasts of
 * lane 15 (into rows 1 and 3) and lane 31 (into rows 2 and 3) add the
 * preceding rows' totals.  Lanes whose DPP source lies outside the row, and
 * the rows a broadcast masks off, add 0.  Every lane of the wave must be
 * active. */
__device__ static inline uint32_t wave_incl_scan(uint32_t v)
{
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);   /* row_shr:1 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);   /* row_shr:2 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);   /* row_shr:4 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);   /* row_shr:8 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   /* row_bcast:15 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   /* row_bcast:31 */
    return v;
}

/* tiles of the flat-sky map (64 columns j by 16 rows k) that a halo's box meets */
#define FS_LOG2C 6
#define FS_LOG2R 4
struct FlatBox {
    int32_t j0, nj, k0, nk;
    __device__ uint32_t n() const { return (uint32_t)nj * (uint32_t)nk; }
};
__device__ static inline FlatBox flat_box(const HaloRec &h)
{
    const int32_t j0 = (h.jmin - 1) >> FS_LOG2C, k0 = (h.kmin - 1) >> FS_LOG2R;
    return {j0, ((h.jmax - 1) >> FS_LOG2C) - j0 + 1, k0, ((h.kmax - 1) >> FS_LOG2R) - k0 + 1};
}

/* ===================================================================== */
/* decode                                                                 */
/* ===================================================================== */

#define CULL_SPAN 8192
#define CULL_U 4                   /* records per thread in flight in k_cull */

/* Cull pass over every record: the radial cut (pks2map.f90:144-160) and the
 * mass cut on the unconverted mass (:264, :296).  A workgroup takes spans of
 * CULL_SPAN consecutive records, collects the survivors' chunk indices in
 * LDS (wave-aggregated LDS atomics), then reserves their range with one
 * global atomic per span and copies them out coalesced.  The FP64 setup
 * then runs on full waves of survivors. */
__global__ void __launch_bounds__(256) k_cull(DecodeArgs A)
{
    const CosmoDev &c = A.c;
    __shared__ uint32_t buf[CULL_SPAN];
    __shared__ unsigned int nbuf;
    __shared__ unsigned long long base_s;
    __shared__ unsigned long long lds16[16];
    const double mconst = ((4.0 / 3.0) * c.mypi) * c.rho_0;
    unsigned long long tot_cut = 0;
    const int64_t nspan = (A.n + CULL_SPAN - 1) / CULL_SPAN;
    const int lane = __lane_id();
    const unsigned long long below = lane == 0 ? 0ULL : ((~0ULL) >> (64 - lane));
    for (int64_t sp = blockIdx.x; sp < nspan; sp += gridDim.x) {
        if (threadIdx.x == 0) nbuf = 0;
        __syncthreads();
        const int64_t i0 = sp * CULL_SPAN;
        /* CULL_U records per thread per step, all four fields of each loaded
         * before any is used: the loads of a step are in flight together */
        for (int kb = 0; kb < CULL_SPAN; kb += CULL_U * (int)blockDim.x) {
            float r0[CULL_U], r1[CULL_U], r2[CULL_U], r6[CULL_U];
#pragma unroll
            for (int u = 0; u < CULL_U; ++u) {
                const int64_t i = i0 + kb + u * (int)blockDim.x + (int)threadIdx.x;
                const float *p = A.halos + 7 * (i < A.n ? i : 0);
                r0[u] = p[0]; r1[u] = p[1]; r2[u] = p[2]; r6[u] = p[6];
            }
#pragma unroll
            for (int u = 0; u < CULL_U; ++u) {
                const int64_t i = i0 + kb + u * (int)blockDim.x + (int)threadIdx.x;
                bool take = false;
                if (i < A.n && kb + u * (int)blockDim.x < CULL_SPAN) {
                    const double xh = (double)r2[u], yh = (double)r1[u], zh = (double)r0[u];
                    const double xs = xh - A.chihview;
                    const double chih = p2m_sqrt((xs * xs + yh * yh) + zh * zh);
                    if (A.precut || !(chih > A.cut_high || chih < A.cut_low)) {
                        tot_cut++;
                        const double mass = mconst * cube((double)r6[u]);
                        take = !(mass < A.mmin);
                    }
                }
                const unsigned long long mask = __ballot(take);
                if (mask) {
                    unsigned int off = 0;
                    if (lane == 0) off = atomicAdd(&nbuf, (unsigned int)__popcll(mask));
                    off = __shfl(off, 0);
                    if (take) buf[off + (unsigned int)__popcll(mask & below)] = (uint32_t)i;
                }
            }
        }
        __syncthreads();
        const unsigned int cnt = nbuf;
        if (threadIdx.x == 0 && cnt) base_s = atomicAdd(A.n_cand, (unsigned long long)cnt);
        __syncthreads();
        for (unsigned int k = threadIdx.x; k < cnt; k += blockDim.x) A.cand[base_s + k] = buf[k];
        __syncthreads();
    }
    block_count(&A.counters[0], tot_cut, lds16);
}

/* FP64 per-halo setup of the survivors: redshift, mass conversion, disc
 * radius (pks2map.f90:284-298, haloproject.f90:47), the query_disc and
 * discphirange_at_z prologues (pixel_routines.F90:1981-2010,
 * pix_tools.F90:729-738), the per-halo part of interpolate_table
 * (maptable.f90:184-202) and the flat-sky box (haloproject.f90:101-128).
 *
 * Bound: FP64 VALU (the elementary functions must give the reference's bits)
 * at three waves a SIMD.  With one arc tangent for either octant, one
 * polynomial where only a sine or a cosine is asked for, and no arc sines for
 * halos that cannot reach the flat-sky field, 1.7e7 halos take 2.10 ms, before
 * 2.33 (both with the cull), 3.5e7 4.0 and 4.26.  Writing a wave's records out
 * through LDS, side by side, is no faster (2.13 ms); held to four waves a SIMD
 * it spills (2.33 ms). */
__global__ void __launch_bounds__(256) k_setup(DecodeArgs A)
{
    const CosmoDev &c = A.c;
    const TabGeom &g = A.g;
    __shared__ unsigned long long lds16[16];
    unsigned long long tot_rad = 0, tot_pairs = 0, tot_pix = 0, tot_gaps = 0, tot_flat = 0;
    const unsigned long long kbeg = *A.n_cand0, kend = *A.n_cand;
    for (unsigned long long k0 = kbeg + blockIdx.x * (unsigned long long)blockDim.x; k0 < kend;
         k0 += (unsigned long long)gridDim.x * blockDim.x) {
        const unsigned long long k = k0 + threadIdx.x;
        bool painted = false;
        uint32_t rings = 1u;               /* rings the disc meets: none (first 1, last 0) */
        double ztop = 1.0, zbot = -1.0;
        HaloRec h;
        if (k < kend) {
            const int64_t i = A.cand[k];
            const float *p = A.halos + 7 * i;
            const float p0 = p[0], p1 = p[1], p2 = p[2], p6 = p[6];
            const double xh = (double)p2, yh = (double)p1, zh = (double)p0;
            const double xs = xh - A.chihview;
            const double chih = p2m_sqrt((xs * xs + yh * yh) + zh * zh);
            const double mass = (((4.0 / 3.0) * c.mypi) * c.rho_0) * cube((double)p6);   /* pks2map.f90:264 */
            double vh = 1.0;
            if (A.profile == 2) {
                double px = p0, py = p1, pz = p2;
                double vr = (px * (double)p[3] + py * (double)p[4]) + pz * (double)p[5];
                vr = vr / p2m_sqrt((px * px + py * py) + pz * pz);
                vh = -vr / 3.0e5;
            }
            const double chi_pre = p2m_sqrt((xh * xh + yh * yh) + zh * zh);          /* :289 */
            const double redshift = tab_lookup(c.zofr, c.nzofr, c.zofr_min, c.dzofr, chi_pre);  /* :290 */
            const double mh = p2m_sqrt(deltacrit_z(c, redshift) / A.dmodel) * mass;    /* :295 */
            const double rh = p2m_pow(((((3.0 * mh) / 4.0) / c.mypi) / 200.0) / rhocrit_z(c, redshift), 1.0 / 3.0); /* :298 */
            const double dtheta = 4.0 * p2m_asin(rh / chih);                      /* haloproject.f90:47 */
            if (!(dtheta >= 0.0 && dtheta <= HPX_PI)) {
                tot_rad++;   /* pixel_routines.F90:1962 would abort */
                /* an inert record: no rings, no flat-sky box */
                h = HaloRec();
                h.dtheta = -1.0; h.irmin = 0; h.irmax = -1; h.flat = 0;
                h.cat = A.index_base + i;
            } else {
                painted = true;
                const double ux = xs / chih, uy = yh / chih, uz = zh / chih;
                h.hx = uz; h.hy = uy; h.hz = ux;
                h.dtheta = dtheta;
                h.vh = vh;
                h.cat = A.index_base + i;
                const double norm = p2m_sqrt((h.hx * h.hx + h.hy * h.hy) + h.hz * h.hz);
                const double z0 = h.hz / norm;
                h.irmin = 0; h.irmax = -1;
                rings = 1u;
                if (A.nside > 0) {
                    const double rlat0 = p2m_asin(z0);
                    const double rlat1 = rlat0 + dtheta, rlat2 = rlat0 - dtheta;
                    const double zmax = (rlat1 >= HPX_HALFPI) ? 1.0 : p2m_sin(rlat1);
                    const int32_t irmin = ring_num(A.nside, zmax);
                    h.irmin = irmin - 1 > 1 ? irmin - 1 : 1;
                    const double zmin = (rlat2 <= -HPX_HALFPI) ? -1.0 : p2m_sin(rlat2);
                    const int32_t irmax = ring_num(A.nside, zmin);
                    h.irmax = irmax + 1 < 4 * A.nside - 1 ? irmax + 1 : 4 * A.nside - 1;
                    rings = disc_rings(A.nside, zmax, zmin, h.irmin, h.irmax);
                    ztop = zmax; zbot = zmin;
                }
                h.cosang = p2m_cos(dtheta);
                const double x0 = h.hx / norm, y0 = h.hy / norm;
                h.zz0 = h.hz / norm;
                h.phi0 = 0.0;
                if (x0 != 0.0 || y0 != 0.0) h.phi0 = p2m_atan2(y0, x0);
                h.a = x0 * x0 + y0 * y0;
                h.s0 = p2m_sqrt(h.a);
                const double sh = p2m_sin(0.5 * dtheta);
                h.thr = 4.0 * (sh * sh);
                double chi = tab_lookup(c.rofz, c.nrofz, c.rofz_min, c.drofz, redshift);
                h.chi_r = chi;
                h.chi_out = chi > g.chimaxt ? 1 : 0;
                if (chi < g.chimint) chi = g.chimint + 1e-5;
                double mc = mh;
                if (mc < g.mhmint) mc = g.mhmint + 1e-5;
                if (mc > g.mhmaxt) mc = g.mhmaxt - 1e-5;
                const double lc = p2m_log(chi), lm = p2m_log(mc);
                h.ichi = (int)((lc - g.lc0) / g.dchit) + 1;
                h.imh = (int)((lm - g.lm0) / g.dmht) + 1;
                h.fc = lc - (g.lc0 + (double)(h.ichi - 1) * g.dchit);
                h.fm = lm - (g.lm0 + (double)(h.imh - 1) * g.dmht);
                h.flat = 0; h.th = 0.0; h.ph = 0.0;
                h.jmin = h.jmax = h.kmin = h.kmax = 0;
                /* |asin(u)| >= |u|: most halos' boxes are outside the field
                 * for certain, and need no arc sines */
                const double reach = A.fov / 2.0 + 1.1 * dtheta + 1e-6;
                if (A.npix_fs > 0 && !(uz < 0.0) && !(p2m_fabs(ux) > reach) && !(p2m_fabs(uy) > reach)) {
                    const double th = p2m_asin(ux), ph = p2m_asin(uy);
                    h.th = th; h.ph = ph;
                    double thetamin = th - 1.1 * dtheta, thetamax = th + 1.1 * dtheta;
                    double phimin = ph - 1.1 * dtheta, phimax = ph + 1.1 * dtheta;
                    const double hf = A.fov / 2.0;
                    if (!(thetamax < -hf || thetamin > hf) && !(phimax < -hf || phimin > hf)) {
                        if (thetamin <= -hf) thetamin = -hf + 1e-10;
                        if (thetamax >= hf) thetamax = hf - 1e-10;
                        if (phimin <= -hf) phimin = -hf + 1e-10;
                        if (phimax >= hf) phimax = hf - 1e-10;
                        int jmin = (int)((thetamin + hf) / A.dpix) + 1; if (jmin < 1) jmin = 1;
                        int jmax = (int)((thetamax + hf) / A.dpix) + 1; if (jmax > A.npix_fs) jmax = A.npix_fs;
                        int kmin = (int)((phimin + hf) / A.dpix) + 1; if (kmin < 1) kmin = 1;
                        int kmax = (int)((phimax + hf) / A.dpix) + 1; if (kmax > A.npix_fs) kmax = A.npix_fs;
                        if (jmax >= jmin && kmax >= kmin) {
                            h.flat = 1; h.jmin = jmin; h.jmax = jmax; h.kmin = kmin; h.kmax = kmax;
                        }
                    }
                }
            }
        }
        const bool flat = k < kend && painted && h.flat;
        if (k < kend && k < (unsigned long long)A.cap) {
            A.out[k] = h;
            if (A.hot) {
                TileHalo t;
                t.zz0 = h.zz0; t.s0 = h.s0; t.phi0 = h.phi0; t.thr = h.thr;
                t.thr_hi = (float)(h.thr * (1.0 + CHORD_BAND));
                t.chi2 = (float)(h.chi_r * h.chi_r);
                const float v = h.chi_out ? 0.0f : (float)h.vh, fc = (float)h.fc, fm = (float)h.fm;
                t.w00 = v * ((1.0f - fc) * (1.0f - fm));
                t.w10 = v * (fc * (1.0f - fm));
                t.w01 = v * ((1.0f - fc) * fm);
                t.w11 = v * (fc * fm);
                /* a halo beyond the table's chi range paints zeros (weights 0); its
                 * cell indices may lie outside the table, so point it at column 0 */
                t.colbase = h.chi_out ? 0 : g.nrt * ((h.imh - 1) + g.nmht * (h.ichi - 1));
                t.pad = 0;
                A.hot[k] = t;
            }
            if (A.pair_halo) {
                PairHalo q;
                q.turn = (float)(h.phi0 * (1.0 / HPX_TWOPI));
                q.half = disc_half_turn(h.thr, h.s0);
                q.rings = rings;
                if (gaps_possible(A.nside, ztop, zbot, h.a, q.half, rings)) { q.rings |= RINGS_ASK_GAPS; tot_gaps++; }
                A.pair_halo[k] = q;
                const uint32_t np = halo_tile_count(A.shape, q.turn, q.half, rings);
                A.n_pairs[k] = np;
                tot_pairs += np;
                /* pixels of the disc, about: its share of the sphere is chord^2 / 4 */
                if (painted) tot_pix += 1ULL + (unsigned long long)(3.0 * A.nside * A.nside * h.thr);
            }
        }
        const unsigned long long fs = wave_append(A.n_flat_out, flat);
        if (flat) {
            A.flat_idx[fs] = (uint32_t)k;
            if (A.flat_tiles) tot_flat += flat_box(h).n();
        }
    }
    block_count(&A.counters[2], tot_rad, lds16);
    block_count(&A.counters[3], tot_pairs, lds16);
    block_count(&A.counters[14], tot_pix, lds16);
    block_count(&A.counters[10], tot_gaps, lds16);
    block_count(&A.counters[9], tot_flat, lds16);
}

/* n_cand0 <- n_cand: the first candidate slot of the next chunk */
__global__ void k_mark_cand(DecodeArgs A)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *A.n_cand0 = *A.n_cand;
}

void p2m_launch_decode(const DecodeArgs &a, hipStream_t s)
{
    if (a.n <= 0) return;
    int64_t gc = (a.n + CULL_SPAN - 1) / CULL_SPAN;
    if (gc > 2048) gc = 2048;
    int64_t g = (a.n + 255) / 256;
    if (g > 8192) g = 8192;
    if (!a.first) hipLaunchKernelGGL(k_mark_cand, dim3(1), dim3(64), 0, s, a);      /* 0 and 0 before the first */
    hipLaunchKernelGGL(k_cull, dim3((unsigned)gc), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_setup, dim3((unsigned)g), dim3(256), 0, s, a);
}

/* ===================================================================== */
/* baseline: plain FP64 painter, one work item per halo                   */
/* ===================================================================== */

__global__ void __launch_bounds__(64) k_paint_plain_hp(PaintArgs A)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    unsigned long long n_list = 0, n_upd = 0, n_gaps = 0;
    if (i < A.n_halo) {
        HaloRec h = A.halos[i];
        const int32_t nside = A.nside;
        int last = 0, pend = 0;
        for (int32_t ring = h.irmin; ring <= h.irmax; ++ring) {
            int32_t npr, kshift; int64_t first;
            ring_info(nside, ring, npr, kshift, first);
            int32_t lo = 0;
            int32_t np = disc_ring_run(h, nside, ring, npr, kshift, lo);
            if (np == 0) { if (last) pend = 1; continue; }
            if (pend) { n_gaps++; pend = 0; }
            last = 1;
            n_list += np;
            for (int32_t k = 0; k < np; ++k) {
                int32_t ip = lo + k; if (ip >= npr) ip -= npr;
                int64_t pix = first + ip;
                double v2[3];
                pix2vec_ring(nside, pix, v2);
                double angle = angdist(h.hx, h.hy, h.hz, v2[0], v2[1], v2[2]);
                if (angle < h.dtheta) {
                    n_upd++;
                    for (int m = 0; m < A.n_maps; ++m) {
                        double val = h.vh * interp_exact(h, A.g, A.tab_flat[m], A.n_flat, A.profile, angle);
                        atomicAdd(&A.map64[m][pix], val);
                    }
                    if (A.count) {
                        atomicAdd(&A.count[pix], 1u);
                        atomicAdd(&A.hash[pix], (unsigned long long)halo_hash(h.cat));
                    }
                }
            }
        }
    }
    wave_count(&A.counters[0], n_list);
    wave_count(&A.counters[1], n_upd);
    wave_count(&A.counters[3], n_gaps);
}

void p2m_launch_paint_plain_hp(const PaintArgs &a, hipStream_t s)
{
    if (a.n_halo <= 0) return;
    hipLaunchKernelGGL(k_paint_plain_hp, dim3((unsigned)((a.n_halo + 63) / 64)), dim3(64), 0, s, a);
}

/* ===================================================================== */
/* baseline flat-sky painter: one work item per halo, FP64, global atomics */
/* ===================================================================== */

__global__ void __launch_bounds__(256) k_paint_fs(PaintArgs A)
{
    unsigned long long n_upd = 0;
    const int64_t hidx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (hidx < A.n_halo) {
        const HaloRec &hr = A.halos[hidx];
        if (hr.flat) {
            HaloRec h = hr;
            double hf = A.fov / 2.0;
            for (int k = h.kmin; k <= h.kmax; ++k) {
                double phip = -hf + ((double)k - 0.5) * A.dpix;
                for (int j = h.jmin; j <= h.jmax; ++j) {
                    double thetap = -hf + ((double)j - 0.5) * A.dpix;
                    double dphi = phip - h.ph, dth = thetap - h.th;
                    double angle = p2m_sqrt(dphi * dphi + dth * dth);
                    if (angle < h.dtheta) {
                        int64_t pix = (int64_t)(j - 1) + (int64_t)A.npix_fs * (k - 1);
                        n_upd++;
                        for (int m = 0; m < A.n_maps; ++m)
                            atomicAdd(&A.fs64[m][pix], h.vh * interp_exact(h, A.g, A.tab_flat[m], A.n_flat, A.profile, angle));
                        if (A.fs_count) {
                            atomicAdd(&A.fs_count[pix], 1u);
                            atomicAdd(&A.fs_hash[pix], (unsigned long long)halo_hash(h.cat));
                        }
                    }
                }
            }
        }
    }
    wave_count(&A.counters[2], n_upd);
}

void p2m_launch_paint_fs(const PaintArgs &a, hipStream_t s)
{
    if (a.n_halo <= 0 || a.npix_fs <= 0) return;
    hipLaunchKernelGGL(k_paint_fs, dim3((unsigned)((a.n_halo + 255) / 256)), dim3(256), 0, s, a);
}

/* ===================================================================== */
/* binning of halos into tiles                                            */
/* ===================================================================== */

/* A painted halo reaches few tiles (about two at 1024 pixels, where its
 * disc covers 13 rings on average), so the binning works on (halo, tile)
 * pairs: they are counted per halo, listed in halo order with the tile as
 * key, and radix-sorted by tile.  A pair's key holds the halo's rows in that
 * tile below the tile's number, key = tile << 8 | first row << 4 | rows - 1,
 * and only the tile's bits are sorted; its value is the halo's slot.  What a
 * halo covers of a row is left to the painter, which has the row's geometry
 * and the halo's constants at hand.
 *
 * Before, the (halo, ring) runs of every disc were cut at ring tiles,
 * counted per tile through an LDS hash and scattered: 13 items a halo, two
 * passes bound by load latency and LDS atomics.  Binning time, scans and sort
 * included: 2e7 halos at nside 4096, 2.2e6 painted, 1.35 -> 0.33 ms; 2e7
 * heavy halos at nside 2048, 1.7e7 painted, 6.0 -> 1.0 ms; 4e7 at nside 4096
 * 17.9 -> 2.75 ms. */
/* the fields of a record that the exact disc query reads */
struct DiscRec { double cosang, zz0, a, phi0; };
__device__ static inline DiscRec disc_rec(const HaloRec &h) { return {h.cosang, h.zz0, h.a, h.phi0}; }

/* ring gaps of the halos marked RINGS_ASK_GAPS (launched only where the
 * setup marked any) */
__global__ void __launch_bounds__(256) k_ring_gaps(BinArgs B)
{
    __shared__ unsigned long long lds16[16];
    unsigned long long gaps = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < B.n_halo; i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t rings = B.halos[i].rings;
        if (rings & RINGS_ASK_GAPS) gaps += (unsigned long long)ring_gaps(disc_rec(B.recs[i]), B.shape.nside, rings & ~RINGS_ASK_GAPS);
    }
    block_count(&B.counters[3], gaps, lds16);
}

__global__ void __launch_bounds__(256) k_pair_count(BinArgs B)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < B.n_halo; i += (int64_t)gridDim.x * blockDim.x) {
        const PairHalo h = B.halos[i];
        B.n_pairs[i] = halo_tile_count(B.shape, h.turn, h.half, h.rings);
    }
}

/* Lists the pairs, `per` halos a wave.  A lane lists its halo's, unless they
 * are more than 64: a disc over hundreds of tiles is listed by the whole wave,
 * the bands' geometry over the lanes, then band by band the sectors (100 discs
 * of 0.27 rad at nside 1024, 430 tiles each: 158 us by their lanes alone, 15
 * now). */
#define WIDE_PAIRS 64
__global__ void __launch_bounds__(256) k_pair_emit(BinArgs B, int per)
{
    if (B.n_split && blockIdx.x == 0 && threadIdx.x < 2) B.n_split[threadIdx.x] = 0u;
    const int lane = __lane_id();
    const int64_t waves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (int64_t w = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6; w * per < B.n_halo; w += waves) {
        const int64_t i = w * per + lane;
        PairHalo h = {0.0f, 0.0f, 1u};
        unsigned long long o = 0;
        uint32_t n = 0;
        if (lane < per && i < B.n_halo) { h = B.halos[i]; o = B.pair_off[i]; n = B.n_pairs[i]; }
        auto list = [&](unsigned long long at, int64_t halo, int32_t band, int32_t k, int32_t row, int32_t rows) {
            if (at < B.pair_cap) {
                B.keys[at] = ((uint32_t)(B.band_tile[band] + k) << 8) | ((uint32_t)row << 4) | (uint32_t)(rows - 1);
                B.vals[at] = (uint32_t)halo;
            }
        };
        if (n <= WIDE_PAIRS)
            halo_tiles(B.shape, h.turn, h.half, h.rings, [&](int32_t band, int32_t k, int32_t row, int32_t rows) {
                list(o++, i, band, k, row, rows);
            });
        for (unsigned long long wide = __ballot(n > WIDE_PAIRS); wide; wide &= wide - 1) {
            const int l = __ffsll((long long)wide) - 1;
            const float turn = __shfl(h.turn, l), half = __shfl(h.half, l);
            unsigned long long at = __shfl(o, l);
            int32_t ra, rb, b0, b1;
            halo_bands(B.shape, (uint32_t)__shfl((int)h.rings, l), ra, rb, b0, b1);
            for (int32_t band = b0; band <= b1; band += 64) {
                BandTiles t = {1, 0, 0, 0, 0};
                if (band + lane <= b1) t = band_tiles(B.shape, band + lane, turn, half, ra, rb);
                const int bands = b1 - band < 63 ? b1 - band + 1 : 64;
                for (int b = 0; b < bands; ++b) {
                    const int32_t K = __shfl(t.K, b), k0 = __shfl(t.k0, b), m = __shfl(t.n, b);
                    const int32_t row = __shfl(t.row, b), rows = __shfl(t.rows, b);
                    for (int32_t k = lane; k < m; k += 64) list(at + k, w * per + l, band + b, k0 + k < K ? k0 + k : k0 + k - K, row, rows);
                    at += m;
                }
            }
        }
    }
}

/* tile_off[t] = the first sorted pair of tile t or a later one, by binary
 * search (empty stretches of the sky leave long runs of equal offsets).
 *
 * A tile of more than S.above pairs is listed for painting in slices: a
 * catalogue of a small field has all its pairs in a few tiles, and a
 * workgroup for each leaves the rest of the GPU idle.  Tile kernel, unsplit
 * and split: 1e6 halos of a 10 x 10 degree field, nside 512 0.97 -> 0.12 ms
 * (FP64 3.29 -> 0.19), nside 1024 1.56 -> 0.20 (FP64 2.76 -> 0.34), nside 4096 2.08 ->
 * 0.99 (FP64 4.79 -> 2.53); 1e5 of a 1 x 1 degree field at nside 4096 2.41 -> 0.56. */
__device__ static inline unsigned long long first_of_tile(const uint32_t *__restrict__ keys, unsigned long long lo,
                                                          unsigned long long hi, int64_t t)
{
    while (lo < hi) {
        const unsigned long long mid = (lo + hi) >> 1;
        if ((int64_t)(keys[mid] >> 8) < t) lo = mid + 1; else hi = mid;
    }
    return lo;
}

__global__ void __launch_bounds__(256) k_tile_bounds(const uint32_t *__restrict__ keys, unsigned long long n, int64_t n_tiles,
                                                     unsigned long long *tile_off, SplitArgs S, unsigned long long *err)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t <= n_tiles; t += (int64_t)gridDim.x * blockDim.x) {
        const unsigned long long lo = first_of_tile(keys, 0, n, t);
        tile_off[t] = lo;
        if (S.above && t < n_tiles && lo + S.above < n && (int64_t)(keys[lo + S.above] >> 8) == t) {
            const uint32_t cnt = (uint32_t)(first_of_tile(keys, lo, n, t + 1) - lo), slices = (cnt - 1) / S.above + 1;
            const uint32_t at = atomicAdd(&S.n[0], slices), part = atomicAdd(&S.n[1], 1u);
            const uint32_t per = cnt / slices, more = cnt - per * slices;
            /* both fit by the choice of `above` */
            if ((uint64_t)at + slices <= S.unit_cap && part < S.part_cap)
                for (uint32_t k = 0; k < slices; ++k)
                    S.units[at + k] = {(uint32_t)t, part, k * per + (k < more ? k : more), per + (k < more ? 1u : 0u), slices, {0, 0, 0}};
            else
                atomicAdd(err, 1ULL);
        }
    }
}

static unsigned bin_grid(int64_t n) { int64_t g = (n + 255) / 256; return (unsigned)(g > 8192 ? 8192 : (g < 1 ? 1 : g)); }
void p2m_launch_pair_count(const BinArgs &b, hipStream_t s)
{
    if (b.n_halo > 0) hipLaunchKernelGGL(k_pair_count, dim3(bin_grid(b.n_halo)), dim3(256), 0, s, b);
}
void p2m_launch_ring_gaps(const BinArgs &b, hipStream_t s)
{
    if (b.n_halo > 0) hipLaunchKernelGGL(k_ring_gaps, dim3(bin_grid(b.n_halo)), dim3(256), 0, s, b);
}
void p2m_launch_pair_emit(const BinArgs &b, hipStream_t s)
{
    if (b.n_halo <= 0) return;
    /* few halos: a wave each, so that wide discs are spread out */
    const int64_t per = std::min<int64_t>(b.n_halo / 8192 + 1, 64);
    hipLaunchKernelGGL(k_pair_emit, dim3(bin_grid((b.n_halo + per - 1) / per * 64)), dim3(256), 0, s, b, (int)per);
}
void p2m_launch_tile_bounds(const uint32_t *keys, unsigned long long n, int64_t n_tiles, unsigned long long *tile_off,
                            const SplitArgs &split, unsigned long long *err, hipStream_t s)
{
    hipLaunchKernelGGL(k_tile_bounds, dim3(bin_grid(n_tiles + 1)), dim3(256), 0, s, keys, n, n_tiles, tile_off, split, err);
}

/* stable radix sort of the pairs by their tile: keys and vals hold 2n
 * entries, input then output */
int p2m_sort_pairs(uint32_t *keys, uint32_t *vals, unsigned long long n, int64_t n_tiles, void *tmp, size_t *tmp_bytes,
                   hipStream_t s)
{
    int bits = 1;
    while ((1LL << bits) < n_tiles && bits < 24) ++bits;
    hipError_t e;
    if (n <= (unsigned long long)INT32_MAX)
        e = hipcub::DeviceRadixSort::SortPairs(tmp, *tmp_bytes, keys, keys + n, vals, vals + n, (int)n, 8, 8 + bits, s);
    else
        e = hipcub::DeviceRadixSort::SortPairs(tmp, *tmp_bytes, keys, keys + n, vals, vals + n, (size_t)n, 8, 8 + bits, s);
    return e == hipSuccess ? 0 : -1;
}

/* Exclusive scan of uint32 counts into uint64 offsets with a 64-bit
 * accumulator.  Up to 16384 counts by one workgroup, consecutive ones a
 * thread: one launch instead of two (2569 counts: 5 us instead of 6 us and the
 * gap between them). */
#define SCAN_SMALL 16384
__global__ void __launch_bounds__(1024) k_scan_small(const uint32_t *__restrict__ cnt, unsigned long long *__restrict__ off, int n)
{
    __shared__ unsigned long long sums[16];
    const int per = (n + 1023) / 1024, i0 = (int)threadIdx.x * per, wv = (int)threadIdx.x >> 6, lane = __lane_id();
    uint32_t v[SCAN_SMALL / 1024];
    unsigned long long t = 0;
#pragma unroll
    for (int k = 0; k < SCAN_SMALL / 1024; ++k) {
        v[k] = k < per && i0 + k < n ? cnt[i0 + k] : 0u;
        t += v[k];
    }
    unsigned long long incl = t;
    for (int step = 1; step < 64; step <<= 1) {
        const unsigned long long u = __shfl_up(incl, step);
        if (lane >= step) incl += u;
    }
    if (lane == 63) sums[wv] = incl;
    __syncthreads();
    unsigned long long o = incl - t;
    for (int w = 0; w < wv; ++w) o += sums[w];
#pragma unroll
    for (int k = 0; k < SCAN_SMALL / 1024; ++k) {
        if (k < per && i0 + k < n) off[i0 + k] = o;
        o += v[k];
    }
}

int p2m_scan_u32(const uint32_t *cnt, unsigned long long *off, int64_t n, void *tmp, size_t *tmp_bytes, hipStream_t s)
{
    if (n <= SCAN_SMALL) {
        if (!tmp) *tmp_bytes = 0;
        else if (n > 0) hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, cnt, off, (int)n);
        return 0;
    }
    hipError_t e = hipcub::DeviceScan::ExclusiveScan(tmp, *tmp_bytes, cnt, off, hipcub::Sum(), 0ULL, (int)n, s);
    return e == hipSuccess ? 0 : -1;
}

/* geometry of every ring */
__global__ void k_ring_desc(int32_t nside, RingDesc *out)
{
    const int32_t r = blockIdx.x * blockDim.x + threadIdx.x + 1;
    if (r > 4 * nside - 1) return;
    RingDesc d;
    int32_t kshift;
    double den;
    ring_info(nside, r, d.npr, kshift, d.first);
    ring_zsth(nside, r, d.zr, d.sth);
    ring_phi_param(nside, r, d.off, den);
    d.kphi = HPX_HALFPI / den;
    d.e_row = (float)(2e-15 / (d.sth * d.sth));
    d.pad = 0;
    out[r - 1] = d;
}

void p2m_launch_ring_desc(int32_t nside, RingDesc *out, hipStream_t s)
{
    const int n = 4 * nside - 1;
    hipLaunchKernelGGL(k_ring_desc, dim3((n + 255) / 256), dim3(256), 0, s, nside, out);
}

__global__ void __launch_bounds__(256) k_tile_desc(TileShape g, int32_t nb, const int32_t *band_tile, TileDesc *desc)
{
    const int32_t b = blockIdx.x;
    if (b >= nb) return;
    TileDesc d;
    int32_t r1;
    d.K = band_sectors(g, b, d.ring0, r1);
    d.rows = r1 - d.ring0 + 1;
    for (int32_t k = threadIdx.x; k < d.K; k += blockDim.x) {
        d.k = k;
        desc[band_tile[b] + k] = d;
    }
}

void p2m_launch_tile_desc(const TileShape &g, const int32_t *band_tile, TileDesc *desc, hipStream_t s)
{
    const int32_t nb = n_bands(g);
    if (nb > 0) hipLaunchKernelGGL(k_tile_desc, dim3((unsigned)nb), dim3(256), 0, s, g, nb, band_tile, desc);
}

/* ===================================================================== */
/* tiled painters                                                         */
/* ===================================================================== */

/* ------------------------------------------------------------------ */
/* common parts                                                         */
/* ------------------------------------------------------------------ */

/* Workgroup barrier for LDS traffic only: waits for this wave's LDS
 * operations, not for its outstanding global loads and stores, then
 * s_barrier.  (__syncthreads also drains global memory, which exposes the
 * latency of the map stores at every tile boundary.) */
__device__ static inline void lds_barrier()
{
    /* LDS-only release and acquire fences around the barrier: the compiler
     * keeps LDS accesses on their side of it, and the hardware waits only
     * for LDS traffic (lgkmcnt), not for outstanding global memory */
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_waitcnt(0xc07f);      /* lgkmcnt(0); vmcnt, expcnt unconstrained */
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

/* The lanes of a wave that pass data through LDS without a barrier: LDS
 * serves a wave's operations in order, but the compiler must not move a
 * lane's loads over other lanes' stores. */
__device__ static inline void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

#define ASK_RUN 0x80000000u        /* a deferred pixel's halo word: it must lie in the halo's exact run */
#define COUNT_LISTED 0x80000000u   /* its row word: it is counted as listed if it does */
#define WSEG 64                    /* segments a wave stages at a time */
#define WPIX 4096                  /* pixels of a wave's bitmap of segment starts */
#define FB_LDS 24                  /* deferred pixels of a tile buffered in LDS (flushed per tile) */
#define MAXROWS 16

/* a row of the tile: its ring's geometry and its pixels */
struct __attribute__((aligned(16))) TileRow {
    double zr, sth, kphi;
    int64_t pix0;                  /* first map pixel */
    uint16_t ip0, width;           /* first in-ring pixel, pixels */
    int32_t npr;                   /* pixels of the ring (4 den: phi = (ip + off) pi/2 / den) */
    float off, e_row;
    __device__ double den() const { return (double)(npr >> 2); }
    __device__ double ik() const { return den() * (2.0 / HPX_PI); }      /* 1 / kphi */
    __device__ int32_t kshift() const { return off > 0.25f ? 1 : 0; }
};

struct TileCtl {
    TileRow rows[2][MAXROWS];
    /* the per-tile control words and rows come in two slots, used by
     * alternate tiles, so that a tile's end needs no barrier before the next
     * begins */
    uint32_t nfb[2];               /* deferred pixels of the tile */
    uint32_t lost[2];              /* a deferred pixel of the tile found the list full */
    int32_t next_tile[2];          /* the tile this workgroup paints next */
    unsigned long long fb_base;    /* list slot of the tile's deferred pixels */
    uint32_t last;                 /* a slice's end: SLICE_LAST, SLICE_LOST */
    uint32_t stat[4];              /* its counts */
    uint4 fb[FB_LDS];
};

__device__ static inline void stage_row(TileRow &R, const RingDesc &d, int32_t K, int32_t k)
{
    const int32_t i0 = sector_start(d.npr, K, k);
    R.zr = d.zr; R.sth = d.sth; R.kphi = d.kphi;
    R.off = (float)d.off;
    R.ip0 = (uint16_t)i0;
    R.width = (uint16_t)(sector_start(d.npr, K, k + 1) - i0);
    R.npr = d.npr;
    R.pix0 = d.first + i0;
    R.e_row = d.e_row;
}

/* bitwise or over the wave, in every lane; all lanes active */
__device__ static inline uint32_t wave_or(uint32_t v)
{
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);   /* row_shr:1 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);   /* row_shr:2 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);   /* row_shr:4 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);   /* row_shr:8 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   /* row_bcast:15 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   /* row_bcast:31 */
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

/* The (halo, row) segments of a wave's next pairs, one per lane: the leading
 * pairs (key, val hold pair `lane`, has whether there is one) whose rows add
 * up to at most WSEG.  Returns how many pairs were taken; every pair has 1 to
 * 16 rows, so at least one is.  A lane's pair is found from the bits that the
 * pairs set at their first lanes: the number of bits at or below the lane. */
struct Seg {
    uint32_t val;                  /* the pair's value */
    int32_t row;                   /* row of the tile */
    int32_t lane0, rows;           /* first lane and rows of the pair */
    bool act;                      /* this lane holds a segment */
};

__device__ static inline int wave_segments(uint32_t key, uint32_t val, bool has, Seg &g)
{
    const int lane = __lane_id();
    const uint32_t nr = has ? (key & 15u) + 1u : 0u;
    const uint32_t incl = wave_incl_scan(nr), excl = incl - nr;
    const bool take = has && incl <= WSEG;
    const unsigned long long tm = __ballot(take);
    const int n = __popcll(tm);
    const int S = __builtin_amdgcn_readlane((int)incl, n - 1);
    const uint32_t bit = take ? 1u << (excl & 31u) : 0u;
    const uint32_t mlo = wave_or(excl < 32u ? bit : 0u), mhi = wave_or(excl < 32u ? 0u : bit);
    const unsigned long long m = ((unsigned long long)mhi << 32) | mlo;
    g.act = lane < S;
    const int below = (int)__builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, 0u));
    int j = below + (int)((m >> lane) & 1ULL) - 1;
    j = j < 0 ? 0 : j;
    g.val = __shfl(val, j);
    const uint32_t pk = __shfl(excl | (((key >> 4) & 15u) << 8) | (nr << 16), j);
    g.lane0 = (int32_t)(pk & 255u);
    g.rows = (int32_t)(pk >> 16);
    g.row = (int32_t)((pk >> 8) & 15u) + lane - g.lane0;
    return n;
}

/* The part of a run (lo, np > 0 of a ring of npr pixels) in a row of `width`
 * pixels from ip0: in-row pixels [a, a + len), and how many of them the run
 * holds.  A run that leaves the row and comes round into it again leaves a
 * gap [c, d) in it (a sector is at most a quarter of its ring, so the run
 * then covers three quarters): the segment is the whole row and hole is
 * set. */
__device__ static inline int32_t clip_run(int32_t lo, int32_t np, const TileRow &R, int32_t &a, int32_t &len, int32_t &c,
                                          int32_t &d)
{
    int32_t rel = lo - (int32_t)R.ip0;
    if (rel < 0) rel += R.npr;
    const int32_t e = rel + np, w = R.width, back = e - R.npr;     /* pixels [0, back) after coming round */
    c = d = 0;
    if (rel >= w) { a = 0; len = back > 0 ? (back < w ? back : w) : 0; return len; }
    if (back <= 0) { a = rel; len = (e < w ? e : w) - rel; return len; }
    a = 0; len = w;
    if (back >= rel) return w;
    c = back; d = rel;
    return w - (d - c);
}

/* Which segment a wave's pixel belongs to: the wave's pixels are numbered
 * segment by segment (start: this lane's first pixel, len of them, the
 * segments without pixels left out of the numbering), and bit p of a bitmap is
 * set if a segment starts at pixel p + 1, so that pixel p's segment is the number
 * of bits below p.  Returns this lane's 64 bits of the window of WPIX pixels
 * from base: pixels base + 64 c .. are the bits of lane c. */
__device__ static inline unsigned long long start_bits(unsigned long long *bits, uint32_t base, uint32_t start, bool has)
{
    const int lane = __lane_id();
    bits[lane] = 0ULL;
    wave_lds_fence();
    const uint32_t at = start - 1u - base;         /* wraps below the window */
    if (has && start > 0u && at < WPIX) atomicOr(reinterpret_cast<uint32_t *>(bits) + (at >> 5), 1u << (at & 31u));
    wave_lds_fence();
    return bits[lane];
}

/* where wave w of nw (1 to 8) starts in n pairs: equal shares, the last ones
 * shorter; divided by constants up to four waves (all that k_tile_fast takes) */
__device__ static inline uint32_t wave_share(uint32_t n, int w, int nw)
{
    uint32_t c;
    switch (nw) {
    case 1: c = n; break;
    case 2: c = (n + 1) / 2; break;
    case 3: c = (n + 2) / 3; break;
    case 4: c = (n + 3) / 4; break;
    default: c = n / (uint32_t)nw + 1; break;
    }
    const uint32_t s = c * (uint32_t)w;
    return s < n ? s : n;
}

/* Where most pairs are whole tiles (the insides of wide discs), a tile has few
 * of them: the FP64 painter's waves then share each by rows, every wave
 * goes over all pairs and takes its part of a pair's rows, if the pair has
 * eight or more; the others are the first wave's. */
__device__ static inline bool narrow_pair(uint32_t &key, int part, int parts)
{
    const int rows = (int)(key & 15u) + 1;
    if (rows < 8) return part == 0;
    const int r0 = rows * part / parts, r1 = rows * (part + 1) / parts;
    key = (key & ~255u) | ((((key >> 4) & 15u) + (uint32_t)r0) << 4) | (uint32_t)(r1 - r0 - 1);
    return true;
}

/* Tiles come from one queue per XCD: workgroup b runs on XCD b % 8 and
 * claims the next tile of that XCD's contiguous eighth of the tiles (sector
 * by sector along a band, so the tiles in flight on an XCD share halos and
 * map lines in its L2) from the XCD's counter.  A workgroup that becomes
 * resident late, or whose tiles run long, leaves the remaining tiles to the
 * others.  Where there is a workgroup for every tile, each has a queue of its
 * own that holds one: claims from shared ones, by all workgroups at once, took
 * 30 us of the launch (3000 halos at nside 64: 48 -> 18 us). */
#define NO_UNIT 0x7fffffff         /* past the end of every queue */
struct TileQueue {
    unsigned int *ctr;
    int64_t xb, xe;
    __device__ TileQueue(const TileArgs &A)
    {
        const bool xq = (gridDim.x % 8) == 0 && A.n_tiles >= 8, all = (int64_t)gridDim.x >= A.n_tiles;
        const int xcd = xq ? (int)(blockIdx.x % 8) : 0;
        xb = xq ? (int64_t)xcd * A.n_tiles / 8 : 0;
        xe = xq ? (int64_t)(xcd + 1) * A.n_tiles / 8 : A.n_tiles;
        if (all) {
            xb += xq ? blockIdx.x / 8 : blockIdx.x;
            xe = xb < xe ? xb + 1 : xb;
        }
        ctr = A.tile_next + (all ? (int)blockIdx.x : xcd) * P2M_TQ_STRIDE;
    }
    __device__ int32_t first() const { return claim(); }
    __device__ int32_t claim() const { return (int32_t)(xb + (int64_t)atomicAdd(ctr, 1u)); }
};

/* The slices of split tiles, in eighths likewise; a workgroup's first is its
 * own number, so that not all of them claim at once. */
struct SliceQueue {
    unsigned int *ctr;
    int64_t xb, xe;
    int32_t own, wgs;
    __device__ SliceQueue(const TileArgs &A)
    {
        const uint32_t n_units = *A.split.n, n = n_units < A.split.unit_cap ? n_units : A.split.unit_cap;
        const bool xq = (gridDim.x % 8) == 0;
        const int xcd = xq ? (int)(blockIdx.x % 8) : 0, queues = xq ? 8 : 1;
        xb = (int64_t)xcd * n / queues;
        xe = (int64_t)(xcd + 1) * n / queues;
        own = (int32_t)(blockIdx.x / queues);
        wgs = (int32_t)(gridDim.x / queues);
        ctr = A.tile_next + xcd * P2M_TQ_STRIDE + P2M_TQ_STRIDE / 2;
    }
    __device__ int32_t first() const { return (int32_t)xb + own; }
    __device__ int32_t claim() const { return (int32_t)xb + wgs + (int32_t)atomicAdd(ctr, 1u); }
};

/* The kernel's first argument, read again from where the launch left it: the
 * loop over the slices takes its arguments from here, so that none of them is
 * held for it in the loop over the tiles (held, they spilled 170 scalar registers
 * instead of 70, and 2e7 halos at nside 4096 with statistics took 2.66 ms, not 2.63). */
__device__ static inline const TileArgs &launch_args()
{
    auto p = (const __attribute__((address_space(4))) TileArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const TileArgs *)p;
}

/* Number u of a queue: tile u, or slice u of the split tiles.  Its tile and
 * pairs, the same in every lane. */
struct PaintUnit {
    int64_t t;
    uint64_t sbeg;
    uint32_t cnt;
};
template <bool SLICES>
__device__ static inline PaintUnit paint_unit(const TileArgs &A, const unsigned long long *__restrict__ toff, int64_t u)
{
    if constexpr (SLICES) {
        const SplitUnit &s = A.split.units[u];
        const int64_t t = (int64_t)__builtin_amdgcn_readfirstlane((int)s.tile);
        return {t, toff[t] + (uint32_t)__builtin_amdgcn_readfirstlane((int)s.from), (uint32_t)__builtin_amdgcn_readfirstlane((int)s.cnt)};
    }
    const uint64_t b = toff[u];
    return {u, b, (uint32_t)(toff[u + 1] - b)};
}

/* The end of a slice, by every thread of the workgroup after the barrier
 * that follows its painting: the LDS tile is added to the tile's part, and
 * the workgroup that is the last of them takes the sums back into its LDS tile
 * (its own pixels, as it will write and clear them) and leaves the part 0.
 * Returns SLICE_LAST if the caller is it, SLICE_LOST if any slice was lost.
 * The additions are device-scope atomics; the fences order them before the
 * arrival, and the last one's reads after it.  No workgroup waits for
 * another. */
#define SLICE_LAST 1u
#define SLICE_LOST 2u
template <int NM>
__device__ static inline uint32_t join_slice(const TileArgs &A, TileCtl *ctl, int64_t unit, int npx, bool lost,
                                             double *acc, unsigned long long *lhash, uint32_t *lcount)
{
    const int W = 1 << A.log2w;
    const SplitUnit su = A.split.units[unit];
    unsigned char *base = A.split.part + (size_t)su.part * ((size_t)NM * W * 8 + (A.count ? (size_t)W * 12 : 0));
    double *sum = (double *)base;
    unsigned long long *hsum = (unsigned long long *)(sum + (size_t)NM * W);
    uint32_t *csum = (uint32_t *)(hsum + W);
    SplitState *st = A.split.state + su.part;
#pragma unroll 1
    for (int p = threadIdx.x; p < npx; p += blockDim.x) {
#pragma unroll 1
        for (int m = 0; m < NM; ++m) {
            const double v = acc[m * W + p];
            if (v != 0.0) atomicAdd(&sum[m * W + p], v);
        }
        if (A.count && lcount[p]) {
            atomicAdd(&csum[p], lcount[p]);
            atomicAdd(&hsum[p], lhash[p]);
        }
    }
    if (lost && threadIdx.x == 0) atomicOr(&st->lost, 1u);
    __threadfence();
    lds_barrier();
    if (threadIdx.x == 0) {
        uint32_t r = 0;
        if (atomicAdd(&st->arrived, 1u) + 1u == su.slices) {
            __threadfence();
            r = SLICE_LAST | (atomicExch(&st->lost, 0u) ? SLICE_LOST : 0u);
            (void)atomicExch(&st->arrived, 0u);
        }
        ctl->last = r;
    }
    lds_barrier();
    const uint32_t r = ctl->last;
    if (r & SLICE_LAST) {
        __threadfence();
#pragma unroll 1
        for (int p = threadIdx.x; p < npx; p += blockDim.x) {
#pragma unroll 1
            for (int m = 0; m < NM; ++m)
                acc[m * W + p] = __longlong_as_double((long long)atomicExch((unsigned long long *)&sum[m * W + p], 0ULL));
            if (A.count) {
                lcount[p] = atomicExch(&csum[p], 0u);
                lhash[p] = atomicExch(&hsum[p], 0ULL);
            }
        }
    }
    return r;
}

/* ------------------------------------------------------------------ */
/* FP64 tiled painter                                                   */
/*                                                                      */
/* A tile's pixel vectors are formed once, and kept in LDS, with the reference's arithmetic (pix2vec_ring from the    */
/* ring's z and sin(theta) and the pixel's phi); per pixel and halo sin^2(theta) is the squared     */
/* cross product, the same bits as the reference's, the table cell and      */
/* fraction follow from its logarithm, the value from the corner-quad table; */
/* it is accumulated in an FP64 LDS tile (ds_add_f64) and written to the    */
/* FP64 map.  Where a decision could differ from the reference's -- sin^2     */
/* within rounding of the disc edge's, the radial coordinate of a cell       */
/* boundary -- and for wide discs, the reference's arithmetic is carried    */
/* out in place: angdist against the disc radius, interpolate_table.        */
/*                                                                      */
/* Bound: FP64 VALU.  Carrying that out for every pixel took five times     */
/* the operations (a sine, a cosine, an arc tangent, a tangent and a        */
/* logarithm with their quotients, eight table loads): 2e6 halos at nside  */
/* 2048 1.85 ms, 1.25 ms now.  (The chord relation of the FP32 painter needs */
/* no vectors and was as fast, but its rounding is another than the cross   */
/* product's: 1e-16 of the chord, 1.3e-12 of a value near a halo's centre.)  */
/* ------------------------------------------------------------------ */

/* the per-segment values, one set per wave */
struct ExactWave {
    unsigned long long bits[WPIX / 64];   /* segment starts */
    double hx[WSEG], hy[WSEG], hz[WSEG];
    double edge[WSEG];             /* sin^2(dtheta) (1 + EDGE_BAND) */
    double chi2[WSEG];             /* chi^2 */
    double w00[WSEG], w10[WSEG], w01[WSEG], w11[WSEG];     /* corner weights times the velocity factor */
    int32_t qoff[WSEG];            /* in-tile pixel minus the wave's pixel number */
    int32_t colbase[WSEG];
    uint32_t slot[WSEG];           /* halo; SLOW: every pixel takes the reference's arithmetic */
    uint32_t hole[WSEG];           /* in-tile pixels the run leaves out: first | end << 12 | row << 24 */
};
/* relative half-width of the band around the disc edge: sin^2 and the edge's are
 * rounded a few times */
#define EDGE_BAND 1e-13
#define SLOW 0x80000000u
/* Pairs above which a tile's pixel vectors are all formed at its start; fewer
 * do not reach most of its pixels, and each is formed when a disc first meets
 * it.  Nside 2048, ms all at the start / all on demand: 7 pairs a tile 0.27 /
 * 0.24, 11: 0.62 / 0.54, 21: 0.70 / 0.63, 35: 0.81 / 0.77, 70: 1.24 / 1.28. */
#define MANY_PAIRS 40u

/* interpolate_table (maptable.f90:176-216) on staged per-halo values, the
 * same operations in the same order as interp_exact; the table through a
 * raw buffer over its n_flat floats, whose out-of-range reads return 0 as
 * tab_flat's bounds test does (the flat index is never negative: r >= rmint
 * and the cells are clamped to >= 1) */
__device__ static inline double tab_buf(__amdgpu_buffer_rsrc_t tr, const TabGeom &g, int p, int ir, int imh, int ichi)
{
    const int64_t idx = (int64_t)(p - 1) + 2 * ((int64_t)(ir - 1) + (int64_t)g.nrt * ((int64_t)(imh - 1) + (int64_t)g.nmht * (int64_t)(ichi - 1)));
    return (double)__uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(tr, (int)(idx * 4), 0, 0));
}

__device__ static inline double interp_staged(int chi_out, double chi_r, double fc, double fm, int imh, int ichi,
                                              const TabGeom &g, __amdgpu_buffer_rsrc_t tr, int profile, double theta)
{
    if (chi_out) return 0.0;
    double r = chi_r * p2m_tan(theta);
    if (r > g.rmaxt) return 0.0;
    if (r < g.rmint) r = g.rmint + 1e-5;
    double lr = p2m_log(r);
    int ir = (int)((lr - g.lr0) / g.drt) + 1;
    double fr = lr - (g.lr0 + (double)(ir - 1) * g.drt);
    double v = tab_buf(tr, g, profile, ir, imh, ichi) * (1.0 - fr) * (1.0 - fc) * (1.0 - fm);
    v = v + tab_buf(tr, g, profile, ir + 1, imh, ichi) * (fr) * (1.0 - fc) * (1.0 - fm);
    v = v + tab_buf(tr, g, profile, ir, imh + 1, ichi) * (1.0 - fr) * (fc) * (1.0 - fm);
    v = v + tab_buf(tr, g, profile, ir + 1, imh + 1, ichi) * (fr) * (fc) * (1.0 - fm);
    v = v + tab_buf(tr, g, profile, ir, imh, ichi + 1) * (1.0 - fr) * (1.0 - fc) * (fm);
    v = v + tab_buf(tr, g, profile, ir + 1, imh, ichi + 1) * (fr) * (1.0 - fc) * (fm);
    v = v + tab_buf(tr, g, profile, ir, imh + 1, ichi + 1) * (1.0 - fr) * (fc) * (fm);
    v = v + tab_buf(tr, g, profile, ir + 1, imh + 1, ichi + 1) * (fr) * (fc) * (fm);
    return v;
}

/* NF consecutive floats of a raw buffer at byte offset vo + so, in loads of
 * 16 and 8 bytes (dword alignment is enough for buffer loads) */
template <int NF>
__device__ static inline void load_floats(__amdgpu_buffer_rsrc_t r, int vo, int so, float *f)
{
    int k = 0;
#pragma unroll
    for (; k + 4 <= NF; k += 4) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, vo + 4 * k, so, 0);
        f[k] = __uint_as_float((uint32_t)v[0]); f[k + 1] = __uint_as_float((uint32_t)v[1]);
        f[k + 2] = __uint_as_float((uint32_t)v[2]); f[k + 3] = __uint_as_float((uint32_t)v[3]);
    }
#pragma unroll
    for (; k + 2 <= NF; k += 2) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, vo + 4 * k, so, 0);
        f[k] = __uint_as_float((uint32_t)v[0]); f[k + 1] = __uint_as_float((uint32_t)v[1]);
    }
#pragma unroll
    for (; k < NF; ++k) f[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, vo + 4 * k, so, 0));
}

/* The value of a pixel at lr = ln r, cell coordinate u (ub: u kept within the
 * table) of segment s's halo, for every map: the cell and fraction of
 * interpolate_table (r < rmint clamped, r > rmaxt 0), a lerp of the two radial
 * columns.  The coordinate only chooses the cell: the fraction is the
 * difference of ln r and the node's, as the reference forms it (formed as
 * (u - cell) drt, of coordinates up to several hundred, it was up to 3.6e-15
 * and 9.7e-16 rms from the reference's; now 9.0e-16 and 2.2e-16). */
template <int NM, typename Wave, typename F>
__device__ static inline void quad_value(const TileArgs &A, __amdgpu_buffer_rsrc_t tab, const Wave &w, int s, double lr,
                                         double u, double ub, F add)
{
    const bool clampr = u < 0.0;                  /* r < rmint: r = rmint + 1e-5 */
    const int cl = min((int)ub, A.g.nrt - 2), cell = clampr ? A.ir_clamp - 1 : cl;
    const double fr = clampr ? A.fr_clamp64 : lr - (A.g.lr0 + (double)cl * A.g.drt);
    const double gr = 1.0 - fr;
    float tq[8 * NM];
    load_floats<8 * NM>(tab, (w.colbase[s] + cell) * (16 * NM), 0, tq);
    const double w00 = w.w00[s], w10 = w.w10[s], w01 = w.w01[s], w11 = w.w11[s];
    const bool zero = u > A.u_max64;               /* r > rmaxt */
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const float *c0v = tq + 4 * m, *c1v = tq + 4 * (NM + m);
        double v0m = w00 * (double)c0v[0], v1m = w00 * (double)c1v[0];
        v0m = __builtin_fma(w10, (double)c0v[1], v0m); v1m = __builtin_fma(w10, (double)c1v[1], v1m);
        v0m = __builtin_fma(w01, (double)c0v[2], v0m); v1m = __builtin_fma(w01, (double)c1v[2], v1m);
        v0m = __builtin_fma(w11, (double)c0v[3], v0m); v1m = __builtin_fma(w11, (double)c1v[3], v1m);
        add(m, zero ? 0.0 : __builtin_fma(fr, v1m, gr * v0m));
    }
}

/* per-thread statistics of a painter */
struct PaintStats {
    unsigned long long listed, upd, segs, err;
};

/* SPECIAL: an instantiation of its own for two kinds of calls, as their
 * branches cost the other one 4% (2e6 halos at nside 2048).
 *  - Pairs are mostly the insides of wide discs (A.wide).  Their pixels all
 *    take the reference's arithmetic, so a step of such pixels alone leaves out
 *    the quick one, and the waves share the pairs by rows.  100 discs of 0.27
 *    rad at nside 1024: 0.94 -> 0.61 ms.
 *  - Tiles of many pixels and maps (exact_vectors): a tile's pixel vectors take
 *    the LDS that the waves need for their own values, so each is formed as it
 *    is used.  1e6 halos at nside 1024, six maps with membership, tiles of 2048
 *    pixels: one wave a CU 2.02, six 0.63 ms. */
template <int NM, bool SLICES, bool SPECIAL>
__device__ static __forceinline__ void paint_exact(const TileArgs &A, const TileDesc *__restrict__ tdesc,
                                                   const unsigned long long *__restrict__ toff, const RingDesc *__restrict__ rdesc)
{
    extern __shared__ unsigned char smem_raw[];
    const int W = 1 << A.log2w, log2c = A.shape.log2c;
    /* LDS: acc (NM*W doubles) | hash (W u64) count (W u32) if membership | TileCtl | pixel vectors (2W doubles) |
     * ExactWave per wave */
    double *acc = (double *)smem_raw;
    const size_t acc_bytes = (size_t)NM * W * 8;
    unsigned long long *lhash = (unsigned long long *)(smem_raw + acc_bytes);
    uint32_t *lcount = (uint32_t *)(smem_raw + acc_bytes + (A.count ? (size_t)W * 8 : 0));
    const size_t mem_bytes = A.count ? (size_t)W * 12 : 0;
    TileCtl *ctl = (TileCtl *)(smem_raw + ((acc_bytes + mem_bytes + 15) & ~(size_t)15));
    const int tid = threadIdx.x, lane = __lane_id(), wv = tid >> 6, nwv = (int)(blockDim.x >> 6);
    /* x and y of the tile's pixel vectors, NaN until a wave has needed one (several may form it: the same bits) */
    double *vx = (double *)(ctl + 1), *vy = vx + W;
    const bool vectors = !SPECIAL || A.vectors, by_rows = SPECIAL && A.wide;
    ExactWave *ew = (ExactWave *)(vectors ? vy + W : vx) + wv;
    PaintStats st = {0, 0, 0, 0};
    const __amdgpu_buffer_rsrc_t tab =
        __builtin_amdgcn_make_buffer_rsrc((void *)A.tab_q, (short)0, (int)(A.n_quad * 4), 0x00020000);
    const std::conditional_t<SLICES, SliceQueue, TileQueue> queue(A);
    if (tid == 0) ctl->next_tile[0] = queue.first();
    for (int p = tid; p < W; p += blockDim.x) {
        for (int m = 0; m < NM; ++m) acc[m * W + p] = 0.0;
        if (vectors) vx[p] = vy[p] = __builtin_nan("");
        if (A.count) { lcount[p] = 0; lhash[p] = 0ULL; }
    }
    lds_barrier();
    for (int par = 0;; par ^= 1) {
        const int64_t unit = (int64_t)__builtin_amdgcn_readfirstlane(ctl->next_tile[par]);
        if (unit >= queue.xe) break;
        const PaintUnit U = paint_unit<SLICES>(A, toff, unit);
        const TileDesc G = tdesc[U.t];
        const uint64_t sbeg = U.sbeg;
        const TileRow *rows = ctl->rows[par];
        if (tid < G.rows) stage_row(ctl->rows[par][tid], rdesc[G.ring0 - 1 + tid], G.K, G.k);
        if (!SLICES && tid == 0) ctl->next_tile[par ^ 1] = queue.claim();
        lds_barrier();
        /* a split tile is painted in slices: not here */
        const bool split = !SLICES && A.split.above && U.cnt > A.split.above;
        const uint32_t cnt = split ? 0u : U.cnt;
        /* x and y of an in-tile pixel's vector */
        auto vector_of = [&](int o, double &x, double &y) {
            const TileRow &Q = rows[o >> log2c];
            const double phi = (((double)((int)Q.ip0 + (o & ((1 << log2c) - 1))) + (double)Q.off) * HPX_HALFPI) / Q.den();
            double sn, cs;
            p2m_sincos(phi, &sn, &cs);
            x = Q.sth * cs;
            y = Q.sth * sn;
        };
        if (vectors && cnt > MANY_PAIRS) {
            for (int p = tid; p < G.rows << log2c; p += blockDim.x) vector_of(p, vx[p], vy[p]);
            lds_barrier();
        }
        const int wv_u = __builtin_amdgcn_readfirstlane(wv);
        uint64_t pos = sbeg + (by_rows ? 0u : wave_share(cnt, wv_u, nwv));
        const uint64_t end = sbeg + (by_rows ? cnt : wave_share(cnt, wv_u + 1, nwv));
        while (pos < end) {
            const bool has = by_rows ? lane == 0 : pos + (uint64_t)lane < end;
            const uint64_t at = by_rows ? pos : (has ? pos + (uint64_t)lane : end - 1);
            Seg g;
            uint32_t key = A.keys[at];
            if (by_rows && !narrow_pair(key, wv_u, nwv)) { ++pos; continue; }
            pos += (uint64_t)wave_segments(key, A.vals[at], has, g);
            uint32_t slot = g.val;
            /* a pair must name a record and rows of the tile; one that does
             * not is counted as an error and painted empty */
            if (g.act && !((uint64_t)slot < (uint64_t)A.n_halo && g.row < G.rows)) { st.err++; g.act = false; }
            if (!g.act) { slot = 0; g.row = 0; }
            const HaloRec &h = A.halos[slot];
            const TileRow R = rows[g.row];
            const int32_t ring = G.ring0 + g.row;
            int32_t lo = 0, np = 0, a = 0, len = 0, c = 0, d = 0;
            const double thr = h.thr;
            if (g.act) {
                /* the run as in k_tile_fast, the exact one in place where that is open */
                const double off = (double)R.off, ik = R.ik(), phi0 = h.phi0;
                const double dz = R.zr - h.zz0, ds = R.sth - h.s0;
                const double ipcd = __builtin_rint(phi0 * ik - off);
                int32_t ipc = (int32_t)ipcd, np_max;
                if (ipc < 0) ipc += R.npr;
                if (ipc >= R.npr) ipc -= R.npr;
                np = disc_ring_run_chord(thr, dz * dz + ds * ds, (float)((4.0 * R.sth) * h.s0), R.e_row,
                                         (float)(0.5 * ((ipcd + off) * R.kphi - phi0)), (float)(2.0 * ik), ipc, R.npr, lo, np_max);
                if (np < 0) np = disc_ring_run_z(disc_rec(h), ring2z(A.nside, ring), R.npr, R.kshift(), lo);
            }
            if (np > 0) st.listed += (unsigned long long)clip_run(lo, np, R, a, len, c, d);
            st.segs += len > 0;
            const uint32_t incl = wave_incl_scan((uint32_t)len), start = incl - (uint32_t)len;
            const uint32_t P = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            const unsigned long long some = __ballot(len > 0);
            wave_lds_fence();
            if (len > 0) {
                const int k = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(some >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)some, 0u));
                const bool slow = h.chi_out || !(thr < F64_SMALL_Q) || !(h.chi_r > 1e-30);
                const double gm = 1.0 - h.fm, gc = 1.0 - h.fc;
                ew->hx[k] = h.hx; ew->hy[k] = h.hy; ew->hz[k] = h.hz;
                /* sin^2(dtheta) from the chord^2 of the edge */
                ew->edge[k] = (thr * (1.0 - 0.25 * thr)) * (1.0 + EDGE_BAND);
                ew->chi2[k] = slow ? 1.0 : h.chi_r * h.chi_r;
                ew->w00[k] = h.vh * (gc * gm); ew->w10[k] = h.vh * (h.fc * gm);
                ew->w01[k] = h.vh * (gc * h.fm); ew->w11[k] = h.vh * (h.fc * h.fm);
                const int32_t o0 = g.row << log2c;
                ew->qoff[k] = o0 + a - (int32_t)start;
                ew->colbase[k] = A.g.nrt * ((h.imh - 1) + A.g.nmht * (h.ichi - 1));
                ew->slot[k] = slot | (slow ? SLOW : 0u);
                ew->hole[k] = (uint32_t)(d > c ? o0 + c : 0) | ((uint32_t)(d > c ? o0 + d : 0) << 12) | ((uint32_t)g.row << 24);
            }
            uint32_t before = 0;
            for (uint32_t base = 0; base < P; base += WPIX) {
                const unsigned long long sb = start_bits(ew->bits, base, start, len > 0);
                const uint32_t pe = P - base < WPIX ? P : base + WPIX;
                for (uint32_t p0 = base; p0 < pe; p0 += 64) {
                    const int ch = (int)((p0 - base) >> 6);
                    const uint32_t mlo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)sb, ch);
                    const uint32_t mhi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(sb >> 32), ch);
                    const int s = (int)__builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, before));
                    before += (uint32_t)(__builtin_popcount(mlo) + __builtin_popcount(mhi));
                    const uint32_t p = p0 + (uint32_t)lane;
                    const bool in = p < pe;
                    /* every lane computes (those past the end on the wave's last
                     * segment's values), the decisions are masks: the step is
                     * one stretch of code but for the stores and the rare
                     * pixels that take the reference's arithmetic */
                    const uint32_t hole = ew->hole[s], sl = ew->slot[s];
                    const int row = (int)(hole >> 24), o = in ? (int)p + ew->qoff[s] : 0;
                    const bool far = (int32_t)sl >= 0;                 /* not SLOW */
                    /* the cross product of angdist */
                    const double ax = ew->hx[s], ay = ew->hy[s], az = ew->hz[s], bz = rows[row].zr;
                    double bx, by;
                    if (vectors) {
                        bx = vx[o];
                        by = vy[o];
                        if (__ballot(in & ((bx != bx) | (by != by)))) {
                            if (in & ((bx != bx) | (by != by))) {
                                vector_of(o, bx, by);
                                vx[o] = bx;
                                vy[o] = by;
                            }
                        }
                    } else {
                        vector_of(o, bx, by);
                    }
                    const bool gap = (o >= (int)(hole & 0xfffu)) & (o < (int)((hole >> 12) & 0xfffu));
                    bool cand = in & !gap, plain = false;
                    if (!SPECIAL || __ballot(in & far)) {
                        const double v0 = ay * bz - az * by, v1 = az * bx - ax * bz, v2 = ax * by - ay * bx;
                        const double q = (v0 * v0 + v1 * v1) + v2 * v2, edge = ew->edge[s];
                        const double lr = __builtin_fma(0.5, f64_log(q * ew->chi2[s]), f64_lntan_sin2(q));
                        const double u = (lr - A.g.lr0) * A.inv_drt;
                        const double ub = __builtin_fmin(__builtin_fmax(u, 0.0), A.u_max64);
                        cand = cand & !(far & (q > edge));
                        plain = cand & far & (q < edge * (1.0 - 2.0 * EDGE_BAND)) & (q > 1e-60) &
                                (__builtin_fabs(u - __builtin_rint(ub)) > A.band64);
                        if (plain) quad_value<NM>(A, tab, *ew, s, lr, u, ub, [&](int m, double v) { atomicAdd(&acc[m * W + o], v); });
                    }
                    bool taken = plain;
                    if (__ballot(cand & !plain)) {
                        if (cand & !plain) {
                            /* the reference's arithmetic */
                            const HaloRec &hr = A.halos[sl & ~SLOW];
                            const double angle = angdist(hr.hx, hr.hy, hr.hz, bx, by, bz);
                            if (angle < hr.dtheta) {
                                taken = true;
                                for (int m = 0; m < NM; ++m) {
                                    const __amdgpu_buffer_rsrc_t tr =
                                        __builtin_amdgcn_make_buffer_rsrc((void *)A.tab_flat[m], (short)0, (int)(A.n_flat * 4), 0x00020000);
                                    atomicAdd(&acc[m * W + o], hr.vh * interp_staged(hr.chi_out, hr.chi_r, hr.fc, hr.fm, hr.imh, hr.ichi,
                                                                                     A.g, tr, A.profile, angle));
                                }
                            }
                        }
                    }
                    st.upd += taken;
                    if (A.count && taken) {
                        atomicAdd(&lcount[o], 1u);
                        atomicAdd(&lhash[o], (unsigned long long)halo_hash(A.halos[sl & ~SLOW].cat));
                    }
                }
            }
        }
        lds_barrier();
        /* every thread writes its pixels and clears them for the next tile;
         * branch on accumulate outside the loops (no speculative map loads) */
        const int npx = G.rows << log2c;
        bool keep = split;
        if constexpr (SLICES) keep = !(join_slice<NM>(A, ctl, unit, npx, false, acc, lhash, lcount) & SLICE_LAST);
        auto out = [&](auto add) {
            for (int p = tid; p < npx; p += blockDim.x) {
                const TileRow &R = rows[p >> log2c];
                const int col = p & ((1 << log2c) - 1);
                if (col < (int)R.width && !keep) {
                    const int64_t pix = R.pix0 + col;
                    for (int m = 0; m < NM; ++m) {
                        if constexpr (decltype(add)::value) A.map64[m][pix] += acc[m * W + p];
                        else A.map64[m][pix] = acc[m * W + p];
                    }
                    if (A.count) {
                        if constexpr (decltype(add)::value) { A.count[pix] += lcount[p]; A.hash[pix] += lhash[p]; }
                        else { A.count[pix] = lcount[p]; A.hash[pix] = lhash[p]; }
                    }
                }
                for (int m = 0; m < NM; ++m) acc[m * W + p] = 0.0;
                if (vectors) vx[p] = vy[p] = __builtin_nan("");
                if (A.count) { lcount[p] = 0; lhash[p] = 0ULL; }
            }
        };
        if (A.accumulate) out(std::true_type{}); else out(std::false_type{});
        if constexpr (SLICES) {        /* one at a time: a slice claimed ahead is one that no idle workgroup takes */
            lds_barrier();
            if (tid == 0) ctl->next_tile[par ^ 1] = queue.claim();
            lds_barrier();
        }
    }
    unsigned long long *red = (unsigned long long *)ctl->fb;
    block_count(&A.counters[0], st.listed, red);
    block_count(&A.counters[1], st.upd, red);
    block_count(&A.counters[4], st.segs, red);
    block_count(A.err, st.err, red);
}

template <int NM, bool SPECIAL>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(NM == 1 ? 3 : 2))) k_tile_exact(TileArgs A, const TileDesc *__restrict__ tdesc,
                                                    const unsigned long long *__restrict__ toff,
                                                    const RingDesc *__restrict__ rdesc)
{
    paint_exact<NM, false, SPECIAL>(A, tdesc, toff, rdesc);
    const TileArgs &B = launch_args();
    if (B.split.above && *B.split.n != 0u) paint_exact<NM, true, SPECIAL>(B, B.desc, B.tile_off, B.ring);
}

/* --------------------------------------------------------------------- */
/* flat-sky painter                                                        */
/*                                                                         */
/* (halo, tile) pairs of the boxes (haloproject.f90:101-135), grouped by     */
/* tile of 64 columns by 16 rows with a counting sort: k_fs_pairs counts     */
/* them per tile, the counts are scanned, k_fs_pairs lists them.  A workgroup */
/* takes a tile (or a slice of its pairs, where the map has few), its waves work as  */
/* those of the FP64 tiled painter do, on rows of the discs instead of ring    */
/* runs: theta^2 is formed with the reference's operations and gives the same  */
/* bits, the value follows from its logarithm, the reference's own arithmetic  */
/* (haloproject.f90:136-150) is carried out within rounding of the disc edge    */
/* and of a cell boundary and for wide discs.  Pixels are summed in LDS.         */
/*                                                                         */
/* Bound: FP64 VALU.  Before, a wave took 64 box pixels (35% of them outside   */
/* their disc), each with a search for its halo, the reference's arithmetic     */
/* and an atomic into the map: 6e4 halos on 4096 x 4096 pixels (2.7e8 updates)   */
/* 8.2 ms, of which the values 3.5 ms and the atomics 1.5 ms; 1.17 ms now, pairs  */
/* included.  2e4 halos on 1024 x 1024 0.23 -> 0.083 ms.  Five waves a SIMD or    */
/* four, 1024 to 4096 workgroups where a map has few tiles: the same time.        */
/* --------------------------------------------------------------------- */

/* Counts (EMIT false) or lists the pairs of the listed halos, `per` halos a
 * wave, the lanes over the flattened (halo, tile) pairs so that a box of
 * many tiles is shared out.  The listing takes the counts down again to 0,
 * as they are found by the next call. */
template <bool EMIT>
__global__ void __launch_bounds__(256) k_fs_pairs(FlatArgs F, int per)
{
    const int lane = __lane_id();
    if (!EMIT && F.first && blockIdx.x == 0)
        for (int i = threadIdx.x; i < P2M_SHARDS; i += blockDim.x) F.counters[i * P2M_CTR_STRIDE + 2] = 0ULL;
    const int64_t w = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6, first = w * per;
    if (first >= F.n_list) return;
    const int64_t at = first + lane;
    const bool has = lane < per && at < F.n_list;
    const uint32_t slot = F.list[has ? at : first];
    const HaloRec &h = F.halos[slot];
    const FlatBox b = flat_box(h);
    const uint32_t n = has ? b.n() : 0u;
    const uint32_t incl = wave_incl_scan(n), excl = incl - n;
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    const int32_t kmin = h.kmin - 1, kmax = h.kmax - 1;
    for (uint32_t base = 0; base < total; base += 64) {
        const uint32_t item = base + (uint32_t)lane;
        int o = 0;                          /* the last lane whose pairs start at or before item */
        for (int step = 32; step > 0; step >>= 1)
            if (__shfl(excl, o + step) <= item) o += step;
        const uint32_t q = item - __shfl(excl, o);
        const int32_t nj = __shfl(b.nj, o), j0 = __shfl(b.j0, o), k0 = __shfl(b.k0, o);
        const int32_t klo = __shfl(kmin, o), khi = __shfl(kmax, o);
        const uint32_t sl = __shfl(slot, o);
        if (item < total) {
            const int32_t dk = (int32_t)(q / (uint32_t)nj), tk = k0 + dk, tj = j0 + (int32_t)(q - (uint32_t)dk * (uint32_t)nj);
            /* the slice: another for every wave */
            const int64_t t = (int64_t)tk * F.nj + tj + F.n_tiles * (int64_t)((uint32_t)w % (uint32_t)F.slices);
            if constexpr (EMIT) {
                const int32_t r0 = max(klo - (tk << FS_LOG2R), 0), r1 = min(khi - (tk << FS_LOG2R), (1 << FS_LOG2R) - 1);
                const unsigned long long pos = F.off[t] + (atomicSub(&F.cnt[t], 1u) - 1u);
                if (pos < F.pair_cap) F.pairs[pos] = make_uint2((uint32_t)(r0 << 4 | (r1 - r0)), sl);
            } else {
                atomicAdd(&F.cnt[t], 1u);
            }
        }
    }
}

/* the per-segment values, one set per wave */
struct FlatWave {
    unsigned long long bits[WPIX / 64];   /* segment starts */
    double th[WSEG], dphi2[WSEG];
    double edge[WSEG];             /* dtheta^2 (1 + EDGE_BAND) */
    double chi2[WSEG];             /* chi^2 */
    double w00[WSEG], w10[WSEG], w01[WSEG], w11[WSEG];     /* corner weights times the velocity factor */
    int32_t qoff[WSEG];            /* in-tile pixel minus the wave's pixel number */
    int32_t colbase[WSEG];
    uint32_t slot[WSEG];           /* halo; SLOW: every pixel takes the reference's arithmetic */
};

template <int NM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NM == 1 ? 5 : 3))) k_fs_paint(TileArgs A, FlatArgs F)
{
    extern __shared__ unsigned char smem_raw[];
    const int W = 1 << (FS_LOG2C + FS_LOG2R);
    __shared__ unsigned long long lds16[16];
    double *acc = (double *)smem_raw;                       /* NM * W */
    const int tid = threadIdx.x, lane = __lane_id(), wv = __builtin_amdgcn_readfirstlane(tid >> 6), nwv = (int)(blockDim.x >> 6);
    FlatWave *fw = (FlatWave *)(acc + NM * W) + wv;
    const int32_t t = (int32_t)(blockIdx.x % (unsigned)F.n_tiles), tk = t / F.nj, tj = t - tk * F.nj;
    const uint64_t sbeg = F.off[blockIdx.x];
    const uint32_t cnt = (uint32_t)(F.off[blockIdx.x + 1] - sbeg);
    if (cnt == 0) return;
    for (int p = tid; p < NM * W; p += blockDim.x) acc[p] = 0.0;
    __syncthreads();
    const __amdgpu_buffer_rsrc_t tab =
        __builtin_amdgcn_make_buffer_rsrc((void *)A.tab_q, (short)0, (int)(A.n_quad * 4), 0x00020000);
    const int32_t j1 = (tj << FS_LOG2C) + 1, k1 = (tk << FS_LOG2R) + 1;       /* the tile's first column and row */
    const double hf = F.fov / 2.0, inv_dpix = 1.0 / F.dpix;
    unsigned long long upd = 0;
    uint64_t pos = sbeg + wave_share(cnt, wv, nwv);
    const uint64_t end = sbeg + wave_share(cnt, wv + 1, nwv);
    while (pos < end) {
        const bool has = pos + (uint64_t)lane < end;
        const uint2 pr = F.pairs[has ? pos + (uint64_t)lane : end - 1];
        Seg g;
        pos += (uint64_t)wave_segments(pr.x, pr.y, has, g);
        const uint32_t slot = g.act ? g.val : 0u;
        const HaloRec &h = F.halos[slot];
        const int32_t k = k1 + (g.act ? g.row : 0);
        /* the row's columns that may lie in the disc, a hundredth of a
         * pixel wider than it */
        const double phip = -hf + ((double)k - 0.5) * F.dpix, dphi = phip - h.ph, d2 = dphi * dphi;
        const double r2 = h.dtheta * h.dtheta, rem = r2 - d2;
        const double half = f64_sqrt(__builtin_fmax(rem, 1e-300)) * inv_dpix * (1.0 + 1e-9) + 0.01;
        const double jc = (h.th + hf) * inv_dpix + 0.5;
        const int32_t lo = (int32_t)__builtin_fmax(__builtin_ceil(jc - half), (double)max(h.jmin, j1));
        const int32_t hi = (int32_t)__builtin_fmin(__builtin_floor(jc + half), (double)min(h.jmax, j1 + (1 << FS_LOG2C) - 1));
        const int32_t len = g.act && !(rem < -1e-12 * r2) && hi >= lo ? hi - lo + 1 : 0;
        const uint32_t incl = wave_incl_scan((uint32_t)len), start = incl - (uint32_t)len;
        const uint32_t P = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        const unsigned long long some = __ballot(len > 0);
        wave_lds_fence();
        if (len > 0) {
            const int s = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(some >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)some, 0u));
            const bool slow = h.chi_out || !(r2 < F64_SMALL_Q) || !(h.chi_r > 1e-30);
            const double gm = 1.0 - h.fm, gc = 1.0 - h.fc;
            fw->th[s] = h.th; fw->dphi2[s] = d2;
            fw->edge[s] = r2 * (1.0 + EDGE_BAND);
            fw->chi2[s] = slow ? 1.0 : h.chi_r * h.chi_r;
            fw->w00[s] = h.vh * (gc * gm); fw->w10[s] = h.vh * (h.fc * gm);
            fw->w01[s] = h.vh * (gc * h.fm); fw->w11[s] = h.vh * (h.fc * h.fm);
            fw->qoff[s] = (g.row << FS_LOG2C) + (lo - j1) - (int32_t)start;
            fw->colbase[s] = A.g.nrt * ((h.imh - 1) + A.g.nmht * (h.ichi - 1));
            fw->slot[s] = slot | (slow ? SLOW : 0u);
        }
        /* at most WSEG segments of a row each: all in one window of start bits */
        const unsigned long long sb = start_bits(fw->bits, 0u, start, len > 0);
        uint32_t before = 0;
        for (uint32_t p0 = 0; p0 < P; p0 += 64) {
            const int ch = (int)(p0 >> 6);
            const uint32_t mlo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)sb, ch);
            const uint32_t mhi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(sb >> 32), ch);
            const int s = (int)__builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, before));
            before += (uint32_t)(__builtin_popcount(mlo) + __builtin_popcount(mhi));
            const uint32_t p = p0 + (uint32_t)lane;
            const bool in = p < P;
            const uint32_t sl = fw->slot[s];
            const int o = in ? (int)p + fw->qoff[s] : 0;
            const bool far = (int32_t)sl >= 0;                 /* not SLOW */
            const double thetap = -hf + ((double)(j1 + (o & ((1 << FS_LOG2C) - 1))) - 0.5) * F.dpix;
            const double dth = thetap - fw->th[s], edge = fw->edge[s];
            const double q = fw->dphi2[s] + dth * dth;
            const double lr = __builtin_fma(0.5, f64_log(q * fw->chi2[s]), f64_lntan_angle(q));
            const double u = (lr - A.g.lr0) * A.inv_drt;
            const double ub = __builtin_fmin(__builtin_fmax(u, 0.0), A.u_max64);
            const bool cand = in & !(far & (q > edge));
            const bool plain = cand & far & (q < edge * (1.0 - 2.0 * EDGE_BAND)) & (q > 1e-60) &
                               (__builtin_fabs(u - __builtin_rint(ub)) > A.band64);
            bool taken = plain;
            if (plain) quad_value<NM>(A, tab, *fw, s, lr, u, ub, [&](int m, double v) { atomicAdd(&acc[m * W + o], v); });
            if (__ballot(cand & !plain)) {
                if (cand & !plain) {
                    /* the reference's arithmetic */
                    const HaloRec &hr = F.halos[sl & ~SLOW];
                    const double angle = p2m_sqrt(q);
                    if (angle < hr.dtheta) {
                        taken = true;
                        for (int m = 0; m < NM; ++m) {
                            const __amdgpu_buffer_rsrc_t tr =
                                __builtin_amdgcn_make_buffer_rsrc((void *)A.tab_flat[m], (short)0, (int)(A.n_flat * 4), 0x00020000);
                            atomicAdd(&acc[m * W + o], hr.vh * interp_staged(hr.chi_out, hr.chi_r, hr.fc, hr.fm, hr.imh, hr.ichi,
                                                                             A.g, tr, A.profile, angle));
                        }
                    }
                }
            }
            upd += taken;
            if (F.count && taken) {
                const int64_t pix = (int64_t)(j1 - 1 + (o & ((1 << FS_LOG2C) - 1))) + (int64_t)F.npix * (k1 - 1 + (o >> FS_LOG2C));
                atomicAdd(&F.count[pix], 1u);
                atomicAdd(&F.hash[pix], (unsigned long long)halo_hash(F.halos[sl & ~SLOW].cat));
            }
        }
    }
    block_count(&F.counters[2], upd, lds16);           /* its barriers order the sums before the stores too */
    for (int p = tid; p < W; p += blockDim.x) {
        const int64_t j = j1 - 1 + (p & ((1 << FS_LOG2C) - 1)), k = k1 - 1 + (p >> FS_LOG2C);
        if (j >= F.npix || k >= F.npix) continue;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const double v = acc[m * W + p];
            if (v != 0.0) {
                if (F.slices > 1) atomicAdd(&F.map[m][j + F.npix * k], v);
                else F.map[m][j + F.npix * k] += v;
            }
        }
    }
}

int64_t p2m_flat_tiles(int32_t npix, int32_t *nj)
{
    const int64_t c = ((int64_t)npix + (1 << FS_LOG2C) - 1) >> FS_LOG2C, r = ((int64_t)npix + (1 << FS_LOG2R) - 1) >> FS_LOG2R;
    *nj = (int32_t)c;
    return c * r;
}

/* A map of few tiles has each tile's pairs in several slices, a workgroup
 * each: 2048 workgroups fill the GPU, of at least 8 pairs so that a tile's
 * clearing and adding up pays (32 is up to 1.6 times slower, 4 no faster),
 * and the slices' counters keep the listing's atomics apart (6e4 halos on
 * 200 x 200 pixels, 52 tiles: in one list per tile 307 us, 44 us in 39).  The
 * fewer the tiles, the more slices each (1e5 halos on 64 x 64 pixels, 4 tiles: 64
 * slices a tile 150 us, 128 84, 256 54, 512 42; on 16 x 16, one tile: 64 850 us,
 * 2048 60). */
int p2m_flat_slices(int64_t n_tiles, int64_t n_pairs)
{
    const int64_t s = std::min<int64_t>(2048 / n_tiles, n_pairs / (8 * n_tiles));
    return (int)std::max<int64_t>(1, s);
}

void p2m_launch_flat_pairs(const FlatArgs &f, int emit, hipStream_t s)
{
    /* few halos: a wave each, so that wide boxes are spread out */
    int64_t per = f.n_list / 8192 + 1;
    if (per > 64) per = 64;
    const int64_t waves = (f.n_list + per - 1) / per;
    const dim3 grid((unsigned)((waves + 3) / 4));
    if (emit) hipLaunchKernelGGL((k_fs_pairs<true>), grid, dim3(256), 0, s, f, (int)per);
    else hipLaunchKernelGGL((k_fs_pairs<false>), grid, dim3(256), 0, s, f, (int)per);
}

int p2m_launch_flat_paint(const TileArgs &a, const FlatArgs &f, hipStream_t s)
{
    const dim3 grid((unsigned)(f.n_tiles * f.slices));
    const size_t lds = (size_t)a.n_maps * (sizeof(double) << (FS_LOG2C + FS_LOG2R)) + 4 * sizeof(FlatWave);
#define P2M_FS(NMv) case NMv: hipLaunchKernelGGL((k_fs_paint<NMv>), grid, dim3(256), lds, s, a, f); break;
    switch (a.n_maps) { P2M_FS(1) P2M_FS(2) P2M_FS(3) P2M_FS(4) P2M_FS(5) P2M_FS(6) default: return -1; }
#undef P2M_FS
    return 0;
}

/* --------------------------------------------------------------------- */
/* FP32 tiled painter                                                      */
/*                                                                         */
/* Per pixel: the azimuth offset from the halo centre,                     */
/* then FP32: chord^2 = A + B sin^2(dphi/2) with the per-(halo,ring)       */
/* constants A = (z-z0)^2 + (sth-s0)^2, B = 4 sth s0 staged in LDS;        */
/* tan^2(theta) = 4h(1-h)/(1-2h)^2 with h = chord^2/4; the cell coordinate */
/* u = (ln r - ln rmin)/drt from log2(r^2); fr = ln(r/r_node) from         */
/* log1p(r^2/r_node^2 - 1); a lerp of the 4 bracketing radial columns.    */
/* Values are summed in an FP64 LDS tile.  Pixels whose                    */
/* chord^2 lies within band_c of the disc edge, or whose u lies within     */
/* `band` of a cell boundary, the r cut-off or the r clamp, are deferred   */
/* to k_fallback, which decides them with the exact FP64 arithmetic of the */
/* reference.                                                              */
/*                                                                         */
/* The waves of a workgroup share the tile's accumulator and nothing else: */
/* each takes its part of the tile's pairs and works through them alone,   */
/* staging up to 64 (halo, row) segments at a time in LDS of its own (their */
/* runs, a bitmap of where each starts, then the pixels), with no barrier   */
/* between the tile's first and its last.                                  */
/*                                                                         */
/* Bound: VALU issue (80% busy at six waves a SIMD).  A pixel takes about   */
/* 90 instructions, a batch of 64 segments about 250 before them (the       */
/* runs, which the binning no longer computes).  2e7 halos at nside 4096:   */
/* 1.25 ms -> 1.45 ms for 1.35 -> 0.33 ms of binning; 2e7 heavy halos at    */
/* nside 2048 3.1 -> 2.5 ms; 4e7 at nside 4096 14.7 -> 12.9 ms.  Rows by    */
/* columns of a tile: 8 x 128 instead of 16 x 64 takes 0.1 ms off the first  */
/* and adds as much to its binning, and is 2% slower on the last two.       */
/* --------------------------------------------------------------------- */

/* One array per constant: a wave's pixels read a few consecutive segments,
 * and 4-byte reads of one array (paired by the compiler into read2)
 * broadcast in one pass, where 16-byte reads of a struct keep the LDS unit
 * several times busier. */
struct FastWave {
    unsigned long long bits[WPIX / 64];   /* segment starts */
    float A[WSEG], B[WSEG], thr_hi[WSEG], chi2[WSEG];   /* chord^2 = A + B sin^2(x); its band top; chi^2 */
    float w00[WSEG], w10[WSEG], w01[WSEG], w11[WSEG];   /* corner weights times the velocity factor */
    float xc[WSEG], hphi[WSEG];    /* azimuth origin x_c; x step per pixel along the ring */
    int32_t cidx[WSEG];            /* wave's pixel number of the azimuth origin: p - cidx = ip - ip_c */
    int32_t colbase[WSEG];
    uint32_t slot[WSEG];           /* halo; ASK_RUN: its deferred pixels must lie in the exact run */
    int16_t qoff[WSEG];            /* in-tile pixel minus the wave's pixel number (-64 * 128 .. 2047) */
};
static_assert(WSEG * 128 <= 32768, "qoff: 64 segments of at most a row of the widest tile");

/* sin^2(x) for |x| <= 2: the odd Taylor polynomial of sin to x^15 (the
 * next term is below 3e-10 there, 6e-12 at pi/2), squared; one branch-free
 * sequence */
__device__ static inline float sin2f(float x)
{
    const float z = x * x;
    float p = __builtin_fmaf(z, -7.6471637e-13f, 1.6059044e-10f);
    p = __builtin_fmaf(z, p, -2.5052108e-8f);
    p = __builtin_fmaf(z, p, 2.7557319e-6f);
    p = __builtin_fmaf(z, p, -1.9841270e-4f);
    p = __builtin_fmaf(z, p, 8.3333333e-3f);
    p = __builtin_fmaf(z, p, -1.6666667e-1f);
    const float sn = __builtin_fmaf(x * z, p, x);
    return sn * sn;
}

template <int NM, bool SLICES>
__device__ static __forceinline__ void paint_fast(const TileArgs &A, const TileDesc *__restrict__ tdesc,
                                                  const unsigned long long *__restrict__ toff, const RingDesc *__restrict__ rdesc)
{
    extern __shared__ unsigned char smem_raw[];
    const int W = 1 << A.log2w, log2c = A.shape.log2c;
    /* LDS: acc (NM*W doubles) | hash (W u64) count (W u32) if membership | TileCtl | FastWave per wave |
     * hashes (WSEG u64 per wave) if membership | 1/r_node^2 (nrt+2 floats) */
    double *acc = (double *)smem_raw;
    const size_t acc_bytes = (size_t)NM * W * 8;
    unsigned long long *lhash = (unsigned long long *)(smem_raw + acc_bytes);
    uint32_t *lcount = (uint32_t *)(smem_raw + acc_bytes + (A.count ? (size_t)W * 8 : 0));
    const size_t mem_bytes = A.count ? (size_t)W * 12 : 0;
    TileCtl *ctl = (TileCtl *)(smem_raw + ((acc_bytes + mem_bytes + 15) & ~(size_t)15));
    const int tid = threadIdx.x, lane = __lane_id(), wv = tid >> 6, nwv = (int)(blockDim.x >> 6);
    FastWave *fw = (FastWave *)(ctl + 1) + wv;
    unsigned long long *hh = (unsigned long long *)((FastWave *)(ctl + 1) + nwv) + wv * WSEG;
    float *invn = (float *)((unsigned long long *)((FastWave *)(ctl + 1) + nwv) + (A.count ? nwv * WSEG : 0));
    /* inner edge of the deferral band, relative to the outer one */
    const float lo_band = (float)((1.0 - (double)A.band_c) / (1.0 + (double)A.band_c));
    const float u_zero = A.u_max + A.band;
    /* constants of the pixel loop that an instruction needs in a vector
     * register (a second scalar operand, a select), pinned there once */
    float v_k0 = A.u_k0, v_frc = A.fr_clamp;
    int v_irc = A.ir_clamp - 1;
    asm volatile("" : "+v"(v_k0), "+v"(v_frc), "+v"(v_irc));

    const int nrt = A.g.nrt;
    /* the corner-quad table as a raw buffer: a 32-bit byte offset per pixel,
     * reads past its end return 0 */
    const __amdgpu_buffer_rsrc_t trs =
        __builtin_amdgcn_make_buffer_rsrc((void *)A.tab_q, (short)0, (int)(A.n_quad * 4), 0x00020000);
    uint32_t n_upd = 0, n_fb = 0, n_list = 0, n_seg = 0, n_err = 0;     /* this thread's, see flush below */
    const int64_t fbs = A.fb_cap / P2M_SHARDS;
    unsigned long long *const fbc = A.fb_count + (blockIdx.x % P2M_SHARDS) * P2M_CTR_STRIDE;
    uint4 *const fbr = A.fb + (blockIdx.x % P2M_SHARDS) * fbs;
    const std::conditional_t<SLICES, SliceQueue, TileQueue> q(A);
    if (tid == 0) {
        ctl->nfb[0] = ctl->nfb[1] = 0; ctl->lost[0] = ctl->lost[1] = 0;
        ctl->next_tile[0] = q.first();
        ctl->next_tile[1] = SLICES ? NO_UNIT : q.claim();
    }
    for (int k = tid; k < nrt + 2; k += blockDim.x) invn[k] = A.inv_node2f[k];
    for (int p = tid; p < W; p += blockDim.x) {
        for (int m = 0; m < NM; ++m) acc[m * W + p] = 0.0;
        if (A.count) { lcount[p] = 0; lhash[p] = 0ULL; }
    }
    lds_barrier();

    /* A tile's descriptor, pair range and first pairs are loaded, and its
     * rows staged, while the tile before it is painted: every thread reads
     * the same tile, so the descriptor and range are scalar loads.  Tile k
     * uses slot par = k & 1 of the rows and control words, and next_tile[par ^ 1]
     * is the tile after it.  Between tile k's two barriers the waves paint;
     * after the second every thread writes out and clears its own pixels.  The
     * next tile's rows and words go to the other slot, whose readers of tile
     * k-1 were done at tile k's first barrier. */
    for (;;) {                     /* once, or slice by slice */
    int64_t unit = (int64_t)__builtin_amdgcn_readfirstlane(ctl->next_tile[0]);
    if (unit >= q.xe) break;
    PaintUnit U = paint_unit<SLICES>(A, toff, unit);
    TileDesc G = tdesc[U.t];
    /* not painted: a split tile here, where its slices are painted, and in
     * the repaint pass a tile that lost no pixels */
    auto skipped = [&]() { return (!SLICES && A.split.above && U.cnt > A.split.above) || (A.redo && !A.lost[U.t]); };
    bool skip = skipped();
    if (tid < G.rows) stage_row(ctl->rows[0][tid], rdesc[G.ring0 - 1 + tid], G.K, G.k);
    uint32_t key = 0, val = 0;
    auto load_pairs = [&](uint64_t base, uint32_t i, uint32_t e) {
        if (i >= e) return;
        const uint64_t at = base + (i + (uint32_t)lane < e ? i + (uint32_t)lane : e - 1);
        key = A.keys[at]; val = A.vals[at];
    };
    const int wv_u = __builtin_amdgcn_readfirstlane(wv);
    auto wave_from = [&](uint32_t n, int w) { return wave_share(n, w, nwv); };
    load_pairs(U.sbeg, wave_from(U.cnt, wv_u), wave_from(U.cnt, wv_u + 1));
    for (int par = 0;; par ^= 1) {
        lds_barrier();
        const int64_t tn = (int64_t)__builtin_amdgcn_readfirstlane(ctl->next_tile[par ^ 1]);
        const bool more = tn < q.xe;
        int32_t after = NO_UNIT;
        if (!SLICES && tid == 0) after = q.claim();
        const int64_t t = U.t;
        const uint64_t sbeg = U.sbeg;
        const uint32_t cnt = U.cnt;
        const PaintUnit Un = paint_unit<SLICES>(A, toff, more ? tn : unit);
        const TileDesc Gn = tdesc[Un.t];
        const uint64_t sbeg_n = Un.sbeg;
        const uint32_t cnt_n = Un.cnt;
        const TileRow *rows = ctl->rows[par];
        uint32_t tu = 0, tf = 0, tl = 0, ts = 0;     /* this tile's updates, deferrals, listed, segments */
        uint32_t i = wave_from(cnt, wv_u);
        const uint32_t e = skip ? i : wave_from(cnt, wv_u + 1);
        bool fetched = false;
        while (i < e) {
            Seg g;
            i += (uint32_t)wave_segments(key, val, i + (uint32_t)lane < e, g);
            uint32_t slot = g.val;
            /* a pair must name a record and rows of the tile; one that does
             * not is counted as an error and painted empty */
            if (g.act && !((uint64_t)slot < (uint64_t)A.n_halo && g.row < G.rows)) { n_err++; g.act = false; }
            if (!g.act) { slot = 0; g.row = 0; }
            const TileHalo &h = A.hot[slot];
            /* the record's fields, all requested before the first is used
             * (one memory round trip; the empty asm keeps them together) */
            const double zz0 = h.zz0, s0 = h.s0, phi0 = h.phi0, thr = h.thr;
            const float thr_h = h.thr_hi, chi2 = h.chi2, w00h = h.w00, w10h = h.w10, w01h = h.w01, w11h = h.w11;
            const int32_t colbase = h.colbase;
            /* the next pairs (the next tile's after the last of this one) */
            if (i < e) load_pairs(sbeg, i, e);
            else if (more) { load_pairs(sbeg_n, wave_from(cnt_n, wv_u), wave_from(cnt_n, wv_u + 1)); fetched = true; }
            asm volatile("" :: "v"(zz0), "v"(s0), "v"(phi0), "v"(thr), "v"(thr_h), "v"(chi2), "v"(w00h), "v"(w10h), "v"(w01h), "v"(w11h), "v"(colbase));
            const TileRow R = rows[g.row];
            const double off = (double)R.off, ik = R.ik();
            const double dz = R.zr - zz0, ds = R.sth - s0, chA = dz * dz + ds * ds;
            const float chB = (float)((4.0 * R.sth) * s0);
            /* azimuth origin: the ring pixel ip_c nearest the halo centre's
             * azimuth, with x_c = ((ip_c + off) kphi - phi0) / 2
             * (|x_c| <= kphi / 4) in FP64; a pixel's x is then x_c plus
             * n = ip - ip_c steps of kphi / 2 in FP32.  n may move by npr
             * (x by pi: sin^2 has period pi): the segment's middle step is
             * moved into [-npr/2, npr/2] here, and a segment is at most a
             * quarter of its ring, so every n of it is within 5/8 npr and
             * |x| <= pi/2 + pi/8 + kphi/4.  So the FP32 error of x stays
             * relative to x. */
            const double ipcd = __builtin_rint(phi0 * ik - off);
            const float xc = (float)(0.5 * ((ipcd + off) * R.kphi - phi0));
            int32_t ipc = (int32_t)ipcd;
            if (ipc < 0) ipc += R.npr;
            if (ipc >= R.npr) ipc -= R.npr;
            /* the halo's run on this ring.  Where that is left open, every
             * pixel that may belong to it is deferred (B = 0, its chord^2 the
             * disc edge's) for k_fallback to ask the exact run, and to count.
             * A row that the run leaves and comes back to is tested whole,
             * and its deferred pixels are asked the exact run too. */
            int32_t lo = 0, np = 0, np_max = 0, a = 0, len = 0, c = 0, d = 0;
            if (g.act) np = disc_ring_run_chord(thr, chA, chB, R.e_row, xc, (float)(2.0 * ik), ipc, R.npr, lo, np_max);
            const int32_t in_row = np != 0 && np_max > 0 ? clip_run(lo, np_max, R, a, len, c, d) : 0;
            const bool open = np < 0;
            if (!open) tl += (uint32_t)in_row;
            ts += len > 0;
            const uint32_t incl = wave_incl_scan((uint32_t)len), start = incl - (uint32_t)len;
            const uint32_t P = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            const unsigned long long some = __ballot(len > 0);
            wave_lds_fence();
            if (len > 0) {
                const int k = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(some >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)some, 0u));
                const int32_t half_npr = R.npr >> 1;
                fw->slot[k] = slot | (open || d > c ? ASK_RUN : 0u);
                fw->qoff[k] = (int16_t)((g.row << log2c) + a - (int32_t)start);
                fw->A[k] = open ? (float)thr : (float)chA;
                fw->B[k] = open ? 0.0f : chB;
                fw->thr_hi[k] = thr_h;
                fw->chi2[k] = chi2;
                fw->w00[k] = w00h; fw->w10[k] = w10h; fw->w01[k] = w01h; fw->w11[k] = w11h;
                fw->colbase[k] = colbase;
                fw->xc[k] = xc;
                fw->hphi[k] = (float)(0.5 * R.kphi);
                const int32_t nmid = (int32_t)R.ip0 + a + (len >> 1) - ipc;
                fw->cidx[k] = ipc - (int32_t)R.ip0 - (a - (int32_t)start) +
                              (nmid > half_npr ? R.npr : (nmid < -half_npr ? -R.npr : 0));
                if (A.count) hh[k] = halo_hash(A.halos[slot].cat);
            }
            uint32_t before = 0;
            for (uint32_t base = 0; base < P; base += WPIX) {
                const unsigned long long sb = start_bits(fw->bits, base, start, len > 0);
                const uint32_t pe = P - base < WPIX ? P : base + WPIX;
                for (uint32_t p0 = base; p0 < pe; p0 += 64) {
                    const int ch = (int)((p0 - base) >> 6);
                    const uint32_t mlo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)sb, ch);
                    const uint32_t mhi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(sb >> 32), ch);
                    const int s = (int)__builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, before));
                    before += (uint32_t)(__builtin_popcount(mlo) + __builtin_popcount(mhi));
                    const uint32_t p = p0 + (uint32_t)lane;
                    if (p >= pe) continue;
                    /* every per-segment constant the accepted path needs is read
                     * here, in one round of LDS reads: the empty asm below keeps
                     * the compiler from moving the later ones behind the disc test,
                     * where each would cost a round trip of its own */
                    const int cix = fw->cidx[s];
                    const float xcs = fw->xc[s], hphi = fw->hphi[s], As = fw->A[s], Bs = fw->B[s], thr_hi = fw->thr_hi[s];
                    const float chi2s = fw->chi2[s];
                    const int qo = fw->qoff[s], cb = fw->colbase[s];
                    const int n = (int)p - cix;
                    const float x = __builtin_fmaf((float)n, hphi, xcs);
                    const float s2 = sin2f(x);
                    const float c2 = __builtin_fmaf(Bs, s2, As);
                    asm volatile("" :: "v"(chi2s), "v"(qo), "v"(cb));
                    if (!(c2 < thr_hi)) continue;                     /* outside the disc */
                    const int o = (int)p + qo;
                    /* tan^2(theta) = 4h(1-h)/(1-2h)^2 with h = chord^2/4 */
                    const float dd = __builtin_fmaf(c2, -0.5f, 1.0f);
                    const float rd = __builtin_amdgcn_rcpf(dd);
                    const float t2 = __builtin_fmaf(-0.25f * c2, c2, c2) * (rd * rd);
                    const float r2 = chi2s * t2;
                    const float u = __builtin_fmaf(__builtin_amdgcn_logf(r2), A.u_k1, -v_k0);
                    const bool zero = u > u_zero;                     /* r > rmaxt: value 0 */
                    /* deferred: near the disc edge, a degenerate chord, or u within
                     * the band of a cell boundary 0..u_max (u clamped to that range,
                     * then its nearest boundary) */
                    const float ub = __builtin_amdgcn_fmed3f(u, 0.0f, A.u_max);
                    const bool defer = (c2 > thr_hi * lo_band) | !(dd > 1e-3f) | (__builtin_fabsf(u - __builtin_rintf(ub)) <= A.band);
                    if (defer) {
                        const uint32_t at = atomicAdd(&ctl->nfb[par], 1u);
                        const bool is_open = Bs == 0.0f;
                        const uint4 e = make_uint4((uint32_t)(o >> log2c) | (is_open ? COUNT_LISTED : 0u),
                                                   (uint32_t)(o & ((1 << log2c) - 1)), fw->slot[s], (uint32_t)t);
                        if (at < FB_LDS) ctl->fb[at] = e;
                        else {
                            const unsigned long long gs = atomicAdd(fbc, 1ULL);
                            if (gs < (unsigned long long)fbs) fbr[gs] = e;
                            else ctl->lost[par] = 1u;
                        }
                        tf += !is_open;
                        continue;
                    }
                    const bool clampr = u < 0.0f;                     /* r < rmint: r = rmint + 1e-5 */
                    /* cell floor(u) clamped to [0, nrt-2] (u >= 0 here unless clamped:
                     * truncation is floor); a clamped r (r = rmint + 1e-5) has the cell
                     * and fraction the host computed for it */
                    const int cell = clampr ? v_irc : min((int)ub, nrt - 2);
                    /* nodes `cell` and cell + 1: 4 corners of every map each,
                     * 32 NM contiguous bytes, requested before the radial fraction
                     * so that their latency covers its LDS read and log */
                    const int vo = (cb + cell) * (16 * NM);
                    float tq[8 * NM];
                    load_floats<8 * NM>(trs, vo, 0, tq);
                    const float w00 = fw->w00[s], w10 = fw->w10[s], w01 = fw->w01[s], w11 = fw->w11[s];
                    /* fr = ln(r / r_node) = (ln 2 / 2) log2(r^2 / r_node^2): the ratio is
                     * in [1, 1.08), where the hardware log2 is within one ulp
                     * (7e-9); both sides evaluated, then selected */
                    float fr_in = 0.34657359f * __builtin_amdgcn_logf(r2 * invn[cell]);
                    asm volatile("" : "+v"(fr_in));   /* computed on every lane: a select, not a branch */
                    const float fr = clampr ? v_frc : fr_in;
                    tu++;
#pragma unroll
                    for (int m = 0; m < NM; ++m) {
                        const float *c0v = tq + 4 * m, *c1v = tq + 4 * (NM + m);
                        /* the corners combined at each node, then one lerp in r */
                        float v0 = w00 * c0v[0];
                        v0 = __builtin_fmaf(w10, c0v[1], v0);
                        v0 = __builtin_fmaf(w01, c0v[2], v0);
                        v0 = __builtin_fmaf(w11, c0v[3], v0);
                        float v1 = w00 * c1v[0];
                        v1 = __builtin_fmaf(w10, c1v[1], v1);
                        v1 = __builtin_fmaf(w01, c1v[2], v1);
                        v1 = __builtin_fmaf(w11, c1v[3], v1);
                        const float fv = __builtin_fmaf(fr, v1 - v0, v0);
                        atomicAdd(&acc[m * W + o], (double)(zero ? 0.0f : fv));
                    }
                    if (A.count) {
                        atomicAdd(&lcount[o], 1u);
                        atomicAdd(&lhash[o], hh[s]);
                    }
                }
            }
        }
        if (!fetched && more) load_pairs(sbeg_n, wave_from(cnt_n, wv_u), wave_from(cnt_n, wv_u + 1));
        if (more && wv == nwv - 1 && lane < Gn.rows)
            stage_row(ctl->rows[par ^ 1][lane], rdesc[Gn.ring0 - 1 + lane], Gn.K, Gn.k);
        if (tid == 0) ctl->next_tile[par] = after;
        lds_barrier();
        /* the tile's deferred pixels still in LDS join the list before the
         * tile is written: a tile whose deferred pixels do not all fit in the
         * list writes nothing and is marked for the repaint pass */
        const uint32_t nfb = ctl->nfb[par];
        const uint32_t nfl = nfb < FB_LDS ? nfb : FB_LDS;
        if (nfl) {
            if (tid == 0) ctl->fb_base = atomicAdd(fbc, (unsigned long long)nfl);
            lds_barrier();
            for (uint32_t k = tid; k < nfl; k += blockDim.x)
                if (ctl->fb_base + k < (unsigned long long)fbs) fbr[ctl->fb_base + k] = ctl->fb[k];
        }
        bool lost = ctl->lost[par] != 0u || (nfl && ctl->fb_base + nfl > (unsigned long long)fbs);
        bool write = !skip;
        if constexpr (SLICES) {
            if (!skip) {
                /* the slice's counts go to the tile's, which the last slice adds
                 * up unless one was lost */
                unsigned long long *st = A.split.state[A.split.units[unit].part].stat;
                if (tid < 4) ctl->stat[tid] = 0;
                lds_barrier();
                atomicAdd(&ctl->stat[0], tl); atomicAdd(&ctl->stat[1], tu);
                atomicAdd(&ctl->stat[2], ts); atomicAdd(&ctl->stat[3], tf);
                lds_barrier();
                if (tid < 4) atomicAdd(&st[tid], (unsigned long long)ctl->stat[tid]);
                const uint32_t r = join_slice<NM>(A, ctl, unit, G.rows << log2c, lost, acc, lhash, lcount);
                write = (r & SLICE_LAST) != 0u;
                lost = (r & SLICE_LOST) != 0u;
                if (write && tid < 4) {
                    const unsigned long long v = atomicExch(&st[tid], 0ULL);
                    const int at = tid < 2 ? tid : tid + 2;           /* counters 0, 1, 4, 5 */
                    if (!lost) atomicAdd(&A.counters[at + (blockIdx.x % P2M_SHARDS) * P2M_CTR_STRIDE], v);
                }
            }
            tu = tf = tl = ts = 0;
        }
        if (tid == 0 && write) {
            if (lost) { A.lost[t] = 1; atomicAdd(A.n_lost + (blockIdx.x % P2M_SHARDS) * P2M_CTR_STRIDE, 1ULL); }
            else if (A.redo) A.lost[t] = 0;
        }
        if (!lost) { n_upd += tu; n_fb += tf; n_list += tl; n_seg += ts; }
        const bool keep = lost || !write;
        /* the branch on accumulate is taken outside the loops: a select
         * inside lets the compiler load the map speculatively (a map read and
         * a wait on it per tile) even when the tile only stores */
        const int npx = G.rows << log2c;
        auto out = [&](auto add) {
            for (int p = tid; p < npx; p += blockDim.x) {
                const TileRow &R = rows[p >> log2c];
                const int col = p & ((1 << log2c) - 1);
                if (col < (int)R.width && !keep) {
                    const int64_t pix = R.pix0 + col;
                    for (int m = 0; m < NM; ++m) {
                        float *dst = A.map32[m] + pix;
                        if constexpr (decltype(add)::value) *dst = (float)((double)*dst + acc[m * W + p]);
                        else __builtin_nontemporal_store((float)acc[m * W + p], dst);    /* not read again in the pass */
                    }
                    if (A.count) {
                        if constexpr (decltype(add)::value) { A.count[pix] += lcount[p]; A.hash[pix] += lhash[p]; }
                        else { A.count[pix] = lcount[p]; A.hash[pix] = lhash[p]; }
                    }
                }
                for (int m = 0; m < NM; ++m) acc[m * W + p] = 0.0;
                if (A.count) { lcount[p] = 0; lhash[p] = 0ULL; }
            }
        };
        if (A.accumulate) out(std::true_type{}); else out(std::false_type{});
        if (tid == 0) { ctl->nfb[par ^ 1] = 0; ctl->lost[par ^ 1] = 0; }   /* the next tile's slot */
        if (!more) break;
        /* the thread's 32-bit counts go out long before they could wrap (a
         * tile adds at most its pairs' pixels over the lanes) */
        if (n_upd >= 1u << 30 || n_list >= 1u << 30) {
            atomicAdd(&A.counters[0], (unsigned long long)n_list); n_list = 0;
            atomicAdd(&A.counters[1], (unsigned long long)n_upd); n_upd = 0;
        }
        unit = tn; U = Un; G = Gn;
        skip = skipped();
    }
    if constexpr (!SLICES) break;
    lds_barrier();
    if (tid == 0) {
        ctl->nfb[0] = 0; ctl->lost[0] = 0;
        ctl->next_tile[0] = q.claim();
        ctl->next_tile[1] = NO_UNIT;
    }
    lds_barrier();
    }
    lds_barrier();
    /* the deferred pixels' buffer is free: its space takes the block sums (the
     * kernel has no static LDS, so its occupancy is what its launch asks) */
    unsigned long long *red = (unsigned long long *)ctl->fb;
    block_count(&A.counters[0], n_list, red);
    block_count(&A.counters[1], n_upd, red);
    block_count(&A.counters[4], n_seg, red);
    block_count(&A.counters[5], n_fb, red);
    block_count(A.err, n_err, red);
}

/* The tiles, then the slices of split ones: a loop of their own, since in
 * the tiles' loop a tile's descriptor would be two loads behind its number (2e7
 * halos at nside 4096 1.45 -> 1.52 ms), and in the same launch, since an empty
 * one of as many workgroups takes 20 us. */
template <int NM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NM == 1 ? 6 : 1))) k_tile_fast(TileArgs A, const TileDesc *__restrict__ tdesc,
                                                   const unsigned long long *__restrict__ toff,
                                                   const RingDesc *__restrict__ rdesc)
{
    paint_fast<NM, false>(A, tdesc, toff, rdesc);
    const TileArgs &B = launch_args();
    if (B.split.above && *B.split.n != 0u) paint_fast<NM, true>(B, B.desc, B.tile_off, B.ring);
}

/* Deferred pixels of k_tile_fast -- (row, in-row pixel, halo, tile) --
 * decided and valued with the exact FP64 arithmetic of the reference
 * (pix2vec_ring, angdist, interpolate_table), added to the FP32 map with one
 * atomic each; ASK_RUN, COUNT_LISTED: see k_tile_fast. */
__global__ void __launch_bounds__(256) k_fallback(FallbackArgs A)
{
    __shared__ unsigned long long lds16[16];
    /* blockIdx.y: shard of the deferred list */
    const unsigned long long fbs = (unsigned long long)(A.fb_cap / P2M_SHARDS);
    unsigned long long n = A.fb_count[blockIdx.y * P2M_CTR_STRIDE];
    if (n > fbs) n = fbs;
    const uint4 *fbr = A.fb + blockIdx.y * fbs;
    unsigned long long n_upd = 0, n_list = 0, n_err = 0;
    for (unsigned long long i = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; i < n;
         i += (unsigned long long)gridDim.x * blockDim.x) {
        const uint4 e = fbr[i];
        const uint32_t slot = e.z & ~ASK_RUN, row = e.x & ~COUNT_LISTED;
        if (!(slot < (uint64_t)A.n_halo && e.w < (uint64_t)A.n_tiles && row < MAXROWS)) { n_err++; continue; }
        /* the entries of a tile that lost some of its deferred pixels: the
         * repaint pass decides that tile again */
        if (A.lost[e.w]) continue;
        const TileDesc G = A.desc[e.w];
        if ((int32_t)row >= G.rows) { n_err++; continue; }
        const int32_t ring = G.ring0 + (int32_t)row;
        /* bytes [0, 32), [80, 112) and [128, 160) of the record: the fields
         * of the exact test and value, requested before the ring geometry */
        const uint4 *hs = reinterpret_cast<const uint4 *>(A.halos + slot);
        const uint4 c0 = hs[0], c1 = hs[1], c5 = hs[5], c6 = hs[6], c8 = hs[8], c9 = hs[9];
        int32_t npr, kshift; int64_t first;
        ring_info(A.nside, ring, npr, kshift, first);
        const int32_t ip = sector_start(npr, G.K, G.k) + (int32_t)e.y;
        double zr, sth, off, den;
        ring_zsth(A.nside, ring, zr, sth);
        ring_phi_param(A.nside, ring, off, den);
        const double phi = (((double)ip + off) * HPX_HALFPI) / den;
        double sn, cs;
        p2m_sincos(phi, &sn, &cs);
        pin4(c0); pin4(c1); pin4(c5); pin4(c6); pin4(c8); pin4(c9);
        const double hx = dbl_of(c0.x, c0.y), hy = dbl_of(c0.z, c0.w), hz = dbl_of(c1.x, c1.y);
        const double dtheta = dbl_of(c1.z, c1.w);
        const double chi_r = dbl_of(c5.x, c5.y), fc = dbl_of(c5.z, c5.w), fm = dbl_of(c6.x, c6.y);
        const double vh = dbl_of(c6.z, c6.w);
        const int64_t cat = (int64_t)(((unsigned long long)c8.y << 32) | c8.x);
        const int32_t ichi = (int32_t)c8.z, imh = (int32_t)c8.w, chi_out = (int32_t)c9.z;
        const double angle = angdist(hx, hy, hz, sth * cs, sth * sn, zr);
        if (e.z & ASK_RUN) {
            int32_t lo = 0;
            const int32_t np = disc_ring_run_z(disc_rec(A.halos[slot]), ring2z(A.nside, ring), npr, kshift, lo);
            int32_t rel = ip - lo;
            if (rel < 0) rel += npr;
            if (rel >= np) continue;
            n_list += (e.x & COUNT_LISTED) != 0u;
        }
        if (!(angle < dtheta)) continue;
        n_upd++;
        const int64_t pix = first + ip;
        for (int m = 0; m < A.n_maps; ++m) {
            /* built from the kernel argument inside the loop, so that the
             * resource stays in scalar registers */
            const __amdgpu_buffer_rsrc_t tr =
                __builtin_amdgcn_make_buffer_rsrc((void *)A.tab_flat[m], (short)0, (int)(A.n_flat * 4), 0x00020000);
            double v = vh * interp_staged(chi_out, chi_r, fc, fm, imh, ichi, A.g, tr, A.profile, angle);
            atomicAdd(A.map32[m] + pix, (float)v);
        }
        if (A.count) {
            atomicAdd(&A.count[pix], 1u);
            atomicAdd(&A.hash[pix], (unsigned long long)halo_hash(cat));
        }
    }
    block_count(&A.counters[0], n_list, lds16);
    block_count(&A.counters[1], n_upd, lds16);
    block_count(A.err, n_err, lds16);
}

int p2m_launch_fallback(const FallbackArgs &a, int64_t n_max, hipStream_t s)
{
    int64_t g = (n_max / P2M_SHARDS + 255) / 256;
    if (g < 1) g = 1;
    if (g > 64) g = 64;
    hipLaunchKernelGGL(k_fallback, dim3((unsigned)g, P2M_SHARDS), dim3(256), 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* The tiled painters' table: for every (mass, chi) cell and radial node k,
 * the values of the four corners the pixel weights combine -- (imh, ichi),
 * (imh+1, ichi), (imh, ichi+1), (imh+1, ichi+1) -- for every map, so that a
 * pixel's two nodes k = ir-1, ir are 32 NM contiguous bytes:
 *   quad[((cell * nrt + k) * n_maps + m) * 4 + corner],
 *   cell = (imh-1) + nmht (ichi-1).
 * Corner values come from the (zero-padded) table by the reference's flat index
 * (maptable.f90:204-212), so the aliasing past the upper mass or chi edge
 * (Q6) reads the next column or the zero padding as the flat table does. */
__global__ void k_build_quad(const float *flat, int64_t n_flat, int32_t profile, int32_t nrt, int32_t nmht, int32_t nchit,
                             int32_t n_maps, int32_t slot, float *quad)
{
    const int64_t n = (int64_t)nrt * nmht * nchit;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        const int32_t k = (int32_t)(e % nrt);
        const int64_t cell = e / nrt;
        const int32_t imh0 = (int32_t)(cell % nmht), ichi0 = (int32_t)(cell / nmht);   /* 0-based */
        float v[4];
        for (int cr = 0; cr < 4; ++cr) {
            const int64_t idx = (int64_t)k + (int64_t)nrt * ((int64_t)(imh0 + (cr & 1)) + (int64_t)nmht * (ichi0 + (cr >> 1)));
            const int64_t at = 2 * idx + (profile - 1);
            v[cr] = at < n_flat ? flat[at] : 0.0f;
        }
        float *q = quad + (e * n_maps + slot) * 4;
        q[0] = v[0]; q[1] = v[1]; q[2] = v[2]; q[3] = v[3];
    }
}

void p2m_launch_build_quad(const float *flat, int64_t n_flat, int32_t profile, int32_t nrt, int32_t nmht, int32_t nchit,
                           int32_t n_maps, int32_t slot, float *quad, hipStream_t s)
{
    const int64_t n = (int64_t)nrt * nmht * nchit;
    if (n <= 0) return;
    int64_t g = (n + 255) / 256;
    if (g > 16384) g = 16384;
    hipLaunchKernelGGL(k_build_quad, dim3((unsigned)g), dim3(256), 0, s, flat, n_flat, profile, nrt, nmht, nchit, n_maps,
                       slot, quad);
}

/* widest tile the painters take (in-tile pixel numbers and the wave's
 * 64 segments of at most a row, 128 pixels, must fit 16 bits) */
int p2m_tile_max_log2w(void) { return 11; }

/* Whether the FP64 painter keeps a tile's pixel vectors in LDS: not where
 * fewer waves than asked, and than four, fit beside them. */
int p2m_exact_vectors(int n_maps, int log2w, int membership, int wg)
{
    const size_t W = (size_t)1 << log2w, b = (size_t)n_maps * W * 8 + (membership ? W * 12 : 0) + sizeof(TileCtl) + 2 * W * 8;
    const int waves = b > 160 * 1024 ? 0 : (int)((160 * 1024 - b) / sizeof(ExactWave));
    return waves >= std::min(wg / 64, 4);
}

size_t p2m_tile_lds_bytes(int mode, int n_maps, int log2w, int membership, int nrt, int wg)
{
    const size_t W = (size_t)1 << log2w, nw = (size_t)(wg / 64);
    size_t b = (size_t)n_maps * W * 8;
    if (membership) b += W * 12;
    b = ((b + 15) & ~(size_t)15) + sizeof(TileCtl);
    if (mode == 2) b += nw * (sizeof(FastWave) + (membership ? 8 * WSEG : 0)) + sizeof(float) * (size_t)(nrt + 2);
    else b += (p2m_exact_vectors(n_maps, log2w, membership, wg) ? 2 * W * sizeof(double) : 0) + nw * sizeof(ExactWave);
    return b;
}

/* The workgroup size to launch for an asked one: every wave has its own
 * staging, so a wide tile of many maps takes fewer waves than asked where all
 * of them do not fit the CU's 160 KB of LDS. */
int p2m_tile_wg(int mode, int n_maps, int log2w, int membership, int nrt, int wg)
{
    while (wg > 64 && p2m_tile_lds_bytes(mode, n_maps, log2w, membership, nrt, wg) > 160 * 1024) wg -= 64;
    return wg;
}

/* workgroups of the tile painter resident per CU at this shape (0 on error) */
int p2m_tile_occupancy(int mode, int n_maps, int wg, size_t lds)
{
    int nb = 0;
    hipError_t e = hipErrorInvalidValue;
#define P2M_OC(K) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, K, wg, lds)
    switch (mode * 8 + n_maps) {
    case 9: P2M_OC((k_tile_exact<1, false>)); break;   case 10: P2M_OC((k_tile_exact<2, false>)); break;
    case 11: P2M_OC((k_tile_exact<3, false>)); break;  case 12: P2M_OC((k_tile_exact<4, false>)); break;
    case 13: P2M_OC((k_tile_exact<5, false>)); break;  case 14: P2M_OC((k_tile_exact<6, false>)); break;
    case 17: P2M_OC(k_tile_fast<1>); break;   case 18: P2M_OC(k_tile_fast<2>); break;
    case 19: P2M_OC(k_tile_fast<3>); break;   case 20: P2M_OC(k_tile_fast<4>); break;
    case 21: P2M_OC(k_tile_fast<5>); break;   case 22: P2M_OC(k_tile_fast<6>); break;
    default: break;
    }
#undef P2M_OC
    return e == hipSuccess ? nb : 0;
}

int p2m_launch_tile_paint(const TileArgs &a, int mode, int n_maps, int grid, int wg, hipStream_t s)
{
    size_t lds = p2m_tile_lds_bytes(mode, n_maps, a.log2w, a.count != nullptr, a.g.nrt, wg);
    if (lds > 160 * 1024 || wg > 512 || (mode == 2 && wg > 256)) return -1;
    if (!a.tile_next || grid > P2M_TQ_MAX) return -1;
    /* the queues' counters (the slices' between the first two of the tiles') */
    p2m_launch_fill_u32(a.tile_next, (grid >= a.n_tiles ? std::max(grid, 8) : 8) * P2M_TQ_STRIDE, 0u, s);
#define P2M_TE(NMv) \
    case NMv: \
        if (a.wide || !a.vectors) hipLaunchKernelGGL((k_tile_exact<NMv, true>), dim3(grid), dim3(wg), lds, s, a, a.desc, a.tile_off, a.ring); \
        else hipLaunchKernelGGL((k_tile_exact<NMv, false>), dim3(grid), dim3(wg), lds, s, a, a.desc, a.tile_off, a.ring); \
        break;
#define P2M_TF(NMv) case NMv: hipLaunchKernelGGL((k_tile_fast<NMv>), dim3(grid), dim3(wg), lds, s, a, a.desc, a.tile_off, a.ring); break;
    if (mode == 1) {
        switch (n_maps) { P2M_TE(1) P2M_TE(2) P2M_TE(3) P2M_TE(4) P2M_TE(5) P2M_TE(6) default: return -1; }
    } else {
        switch (n_maps) { P2M_TF(1) P2M_TF(2) P2M_TF(3) P2M_TF(4) P2M_TF(5) P2M_TF(6) default: return -1; }
    }
#undef P2M_TE
#undef P2M_TF
    return 0;
}

/* ===================================================================== */
/* products: moments, RMS, dP/dy (pks2map.f90:321-357)                    */
/* ===================================================================== */

/* One read of the map: the sums of x, x^2 and x^3, the sum of squares about
 * the mean, and (HIST) the dP/dy histogram, m = int(hpmap(i)/dpdy_dy)+1 in
 * FP32 (pks2map.f90:344).  Each workgroup takes one contiguous chunk and
 * writes P2M_MOM_PART doubles: the three sums, its mean and its sum of
 * squares about that mean, which the host joins (Chan's update).  The
 * squares are summed about a pivot near the chunk's mean (the mean of the
 * chunk's first values), so that nothing cancels.
 *
 * Bound: reading the map, and the FP64 sums beside it.  The histogram is
 * kept in LDS (nb 32-bit bins, 40 KB) and the first bin, which takes every
 * pixel no halo reaches, in a register: with one global atomic per pixel
 * most of the map's updates met on that one address, and the two passes took
 * 1390 ms for a nside-4096 map of 2e7 halos of which a tenth are painted
 * (0.23 ms now, 3.5 TB/s). */
#define MOM_WG 1024

__device__ static inline double wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

template <typename T, bool HIST>
__global__ void __launch_bounds__(MOM_WG) k_moments(const T *__restrict__ map, int64_t n, int64_t chunk, double *part,
                                                    unsigned long long *hist, int nb, float dy)
{
    extern __shared__ uint32_t bins[];
    __shared__ double red[5][MOM_WG / 64];
    const int tid = threadIdx.x, lane = __lane_id(), wv = tid >> 6;
    const int64_t i0 = (int64_t)blockIdx.x * chunk, i1 = i0 + chunk < n ? i0 + chunk : n;
    if (HIST) for (int k = tid; k < nb; k += MOM_WG) bins[k] = 0u;
    /* pivot: the mean of the chunk's first values */
    const int64_t np = i1 - i0 < MOM_WG ? i1 - i0 : MOM_WG;
    {
        const double v = wave_sum(tid < np ? (double)(float)map[i0 + tid] : 0.0);
        if (lane == 0) red[0][wv] = v;
    }
    __syncthreads();
    double piv = 0.0;
    for (int k = 0; k < MOM_WG / 64; ++k) piv += red[0][k];
    piv /= (double)np;
    __syncthreads();
    double s1 = 0, s2 = 0, s3 = 0, d1 = 0, d2 = 0;
    uint32_t zero = 0;
    auto take = [&](T raw) {
        const float xf = (float)raw;
        const double x = (double)xf, xx = x * x, d = x - piv;
        s1 += x; s2 += xx; s3 = __builtin_fma(xx, x, s3);
        d1 += d; d2 = __builtin_fma(d, d, d2);
        if (HIST) {
            const float u = xf / dy;
            if (u > -1.0f && u < (float)nb) {
                const int mb = (int)u;
                if (mb == 0) ++zero;
                else atomicAdd(&bins[mb], 1u);
            }
        }
    };
    /* four consecutive values per thread and round (a chunk starts at a
     * multiple of 4), then the rest one by one */
    struct alignas(sizeof(T) * 4) Four { T v[4]; };
    const Four *m4 = reinterpret_cast<const Four *>(map + i0);
    const int64_t n4 = (i1 - i0) >> 2;
#pragma unroll 2
    for (int64_t k = tid; k < n4; k += MOM_WG) {
        const Four q = m4[k];
        take(q.v[0]); take(q.v[1]); take(q.v[2]); take(q.v[3]);
    }
    for (int64_t i = i0 + 4 * n4 + tid; i < i1; i += MOM_WG) take(map[i]);
    s1 = wave_sum(s1); s2 = wave_sum(s2); s3 = wave_sum(s3); d1 = wave_sum(d1); d2 = wave_sum(d2);
    if (lane == 0) { red[0][wv] = s1; red[1][wv] = s2; red[2][wv] = s3; red[3][wv] = d1; red[4][wv] = d2; }
    if (HIST) {
        for (int o = 32; o > 0; o >>= 1) zero += __shfl_xor(zero, o);
        if (lane == 0 && zero) atomicAdd(&bins[0], zero);
    }
    __syncthreads();
    if (tid == 0) {
        double t[5] = {0, 0, 0, 0, 0};
        for (int j = 0; j < 5; ++j)
            for (int k = 0; k < MOM_WG / 64; ++k) t[j] += red[j][k];
        const double cnt = (double)(i1 - i0), off = t[3] / cnt;
        double *p = part + (int64_t)blockIdx.x * P2M_MOM_PART;
        p[0] = t[0]; p[1] = t[1]; p[2] = t[2];
        p[3] = piv + off;                       /* the chunk's mean */
        p[4] = t[4] - off * t[3];               /* squares about it */
    }
    if (HIST) {
        /* every workgroup starts its flush elsewhere, so that they do not
         * all meet on the same bins */
        const int k0 = (int)(((int64_t)blockIdx.x * nb) / gridDim.x);
        for (int k = tid; k < nb; k += MOM_WG) {
            const int bin = k + k0 < nb ? k + k0 : k + k0 - nb;
            const uint32_t v = bins[bin];
            if (v) atomicAdd(&hist[bin], (unsigned long long)v);
        }
    }
}

/* chunks of a map of n values: one per workgroup, a multiple of 4 values,
 * at least 4096, at most P2M_MOM_BLOCKS of them (one 1024-lane workgroup per
 * CU, enough loads in flight to stream the map) */
int64_t p2m_moments_chunk(int64_t n)
{
    int64_t c = (n + P2M_MOM_BLOCKS - 1) / P2M_MOM_BLOCKS;
    if (c < 4096) c = 4096;
    return (c + 3) & ~(int64_t)3;
}

/* m32 or m64 is read; hist NULL: no histogram */
void p2m_launch_moments(const float *m32, const double *m64, int64_t n, double *part, unsigned long long *hist, int nb,
                        float dy, hipStream_t s)
{
    if (n <= 0) return;
    const int64_t chunk = p2m_moments_chunk(n);
    const dim3 g((unsigned)((n + chunk - 1) / chunk)), wg(MOM_WG);
    const size_t lds = sizeof(uint32_t) * (size_t)nb;
    if (m32 && hist) hipLaunchKernelGGL((k_moments<float, true>), g, wg, lds, s, m32, n, chunk, part, hist, nb, dy);
    else if (m32) hipLaunchKernelGGL((k_moments<float, false>), g, wg, 0, s, m32, n, chunk, part, hist, nb, dy);
    else if (hist) hipLaunchKernelGGL((k_moments<double, true>), g, wg, lds, s, m64, n, chunk, part, hist, nb, dy);
    else hipLaunchKernelGGL((k_moments<double, false>), g, wg, 0, s, m64, n, chunk, part, hist, nb, dy);
}

__global__ void k_f64_to_f32(const double *in, float *out, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) out[i] = (float)in[i];
}
__global__ void k_f32_to_f64(const float *in, double *out, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) out[i] = (double)in[i];
}
void p2m_launch_f64_to_f32(const double *in, float *out, int64_t n, hipStream_t s) { if (n > 0) hipLaunchKernelGGL(k_f64_to_f32, dim3(fill_grid(n)), dim3(256), 0, s, in, out, n); }
void p2m_launch_f32_to_f64(const float *in, double *out, int64_t n, hipStream_t s) { if (n > 0) hipLaunchKernelGGL(k_f32_to_f64, dim3(fill_grid(n)), dim3(256), 0, s, in, out, n); }

/* ===================================================================== */
/* diagnostic: portable math on the device                                */
/* ===================================================================== */

__global__ void k_selftest_math(int op, const double *x, const double *y, double *out, int64_t n)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double a = x[i], b = y ? y[i] : 0.0, r = 0.0;
    switch (op) {
    case 0: r = p2m_sqrt(a); break;
    case 1: r = p2m_sin(a); break;
    case 2: r = p2m_cos(a); break;
    case 3: r = p2m_tan(a); break;
    case 4: r = p2m_asin(a); break;
    case 5: r = p2m_acos(a); break;
    case 6: r = p2m_atan2(a, b); break;
    case 7: r = p2m_log(a); break;
    case 8: r = p2m_exp(a); break;
    case 9: r = p2m_pow(a, b); break;
    default: r = 0.0; break;
    }
    out[i] = r;
}

int p2m_launch_selftest_math(int op, const double *x, const double *y, double *out, int64_t n, hipStream_t s)
{
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_selftest_math, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, op, x, y, out, n);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* plain streaming copy, 16 B per lane per iteration: the known-traffic
 * kernel that calibrates HBM byte counters and measures copy bandwidth */
__global__ void __launch_bounds__(256) k_copy_calib(const float4 *__restrict__ src, float4 *__restrict__ dst, int64_t n4)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

int p2m_launch_copy_calib(const void *src, void *dst, int64_t n4, hipStream_t s)
{
    if (n4 <= 0) return 0;
    int64_t g = (n4 + 255) / 256;
    if (g > 8192) g = 8192;
    hipLaunchKernelGGL(k_copy_calib, dim3((unsigned)g), dim3(256), 0, s, (const float4 *)src, (float4 *)dst, n4);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
