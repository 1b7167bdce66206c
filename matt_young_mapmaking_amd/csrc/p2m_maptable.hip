/*
 * p2m_maptable.hip -- make_maptable on the GPU: the projected Battaglia et
 * al. (2012) tSZ y (times G(x) at frequency nu) and tau profiles on the
 * (chi, M, r) grid of maptable.f90:25-146, one work item per grid node.
 *
 * FP64 arithmetic after maptable.f90, integrate_profiles.f90:12-95 and
 * bbps_profile.f90:60-180; named constants keep the reference's values
 * (real(4) literals rounded to float where the reference declares them so).
 * What depends on (chi, M) or (chi, r) alone is computed once per pair, with
 * the portable functions of p2m_math.h; the line-of-sight sums of the
 * reference (401 points of spacing 0.01) are evaluated through Gauss rules
 * for sums over equidistant points, see k_make_maptable.
 */
#include <hip/hip_runtime.h>

#include <vector>

#include "../../include/pks2map_gpu.h"
#include "p2m_kernels.h"
#include "p2m_fast64.h"

namespace {

/* bbps_profile.f90:9-40 (real(4) parameter arrays) */
struct BBPS {
    float P0_Am[3], P0_alpham[3], P0_alphaz[3];
    float xc_Am[3], xc_alpham[3], xc_alphaz[3];
    float beta_Am[3], beta_alpham[3], beta_alphaz[3];
    float P0_Am_rho[3], P0_alpham_rho[3], P0_alphaz_rho[3];
    float alpha_Am_rho[3], alpha_alpham_rho[3], alpha_alphaz_rho[3];
    float beta_Am_rho[3], beta_alpham_rho[3], beta_alphaz_rho[3];
};

const BBPS kBBPS = {
    {18.100f, 7.490f, 20.7f}, {0.154f, 0.226f, -0.074f}, {-0.758f, -0.957f, -0.743f},
    {0.497f, 0.710f, 0.438f}, {-0.00865f, -0.0833f, 0.011f}, {0.731f, 0.853f, 1.01f},
    {4.35f, 4.19f, 3.82f}, {0.0393f, 0.048f, 0.0375f}, {0.415f, 0.615f, 0.535f},
    {1.9e-5f, 9.1e-05f, 1.5e-4f}, {0.29f, 0.10f, 0.14f}, {-0.67f, -0.92f, -1.32f},
    {0.88f, 0.69f, 0.68f}, {-0.03f, -0.02f, -0.02f}, {0.20f, 0.27f, 0.29f},
    {3.83f, 4.43f, 6.4f}, {0.044f, 0.0035f, 0.028f}, {-0.025f, 0.037f, -0.25f}};

/* What a node needs from its (chi, M) pair. */
struct CellCM {
    double P0, ixc, gl, beta;    /* y integrand: P0 exp(gl + gamma ln x - beta ln(1 + x ixc)) */
    double P0r, alr, er;         /* rho integrand: P0r exp(-0.2 l + er ln(1 + exp(alr l))), l = ln(x / 0.5) */
    double rvir, cy, ctau, Gx;
};

struct MTArgs {
    BBPS b;
    int32_t mi, nchit, nmht, nrt;
    double nu, alpha_cmb, Delta, y0, tau0, x0const;
    double omegam, omegal, rhocrit_0;
    double chimint, mhmint, rmint, dchit, dmht, drt;
    const double *rofz, *zofr;
    CellCM *cm;                  /* nchit * nmht */
    double *proj;                /* chi sin(theta): nchit * nrt */
    double *rules;               /* the Gauss rules (k_gram_rules) */
    float *table;
};

}  // namespace

#define MT_DS ((double)1e-2f)            /* integrate_profiles.f90:8 */
#define MT_GAMMA ((double)-0.3f)         /* bbps_profile.f90:25 */
#define MT_GAMMA_RHO ((double)0.2f)      /* bbps_profile.f90:40 */

/* a wave-uniform double, in scalar registers */
__device__ static inline double dbl_uniform(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ static inline double mt_lookup(const double *t, double dt, double x)
{
    double u = (x - 0.0) / dt + 1.0;
    if (u < 1.0) return t[0];
    if (u >= 10000.0) return t[9999];
    int itab = (int)u;
    double fint = ((x - (double)(itab - 1) * dt) - 0.0) / dt;
    return (1.0 - fint) * t[itab - 1] + fint * t[itab];
}

__device__ static inline double mt_fit(float A0, float am, float az, double mh, double z)
{
    return ((double)A0 * p2m_pow(mh / 1e14, (double)am)) * p2m_pow(1.0 + z, (double)az);
}

/* ------------------------------------------------------------ sums */

/* The reference adds f(s_q), s_q = (q - 1/2) ds, over q = 1..N, one by one.
 * f is analytic in s for Re s > 0 (x = sqrt(s^2 + b^2), powers of x and of
 * 1 + x^a, a < 2), with its singular points at s = +-i b.  For a sum of N
 * equidistant values there is a Gauss rule, as there is for an integral: the
 * roots of the polynomial of degree n that is orthogonal over the points
 * (Gram's discrete Chebyshev polynomials) and positive weights adding to N
 * give the sum of every polynomial of degree 2n - 1 exactly.  Over points
 * [p, 2p) or part of them the singular points lie outside the ellipse of
 * parameter 5.8, so MT_N = 11 nodes leave an error below 6e-17 of the block's
 * sum.  The first block [0, S) is summed point by point (S = 16) where b is
 * small; where S ds <= b/2, the values mirrored at s = 0 are 2S points
 * whose rule of 2 MT_M nodes is symmetric, so MT_M = 8 evaluations do.
 * Against sums in extended precision over b in (0.002, 4) and the profiles'
 * ranges of exponents both agree to 1e-15.  The rest of the last block, of
 * any length, has a rule of its own length (of at most MT_N points every
 * point itself).
 *
 * Layout: rule N (1..MT_MAXN) holds MT_N pairs (t, w): t = q - 1/2 counted
 * from the block's start; then the half rules of S = 16 * 2^j, MT_M pairs
 * each.  b is at most MT_RMAX, so S at most 128; the blocks are then of 16 to
 * 128 points, and the last one starts at 256. */
#define MT_N 11
#define MT_M 8
#define MT_MAXN 145
#define MT_S0 16
#define MT_NSTART 4
#define MT_RMAX 4.0                      /* in virial radii, integrate_profiles.f90:12-95 */
static_assert((MT_S0 << MT_NSTART) * MT_DS > 0.5 * MT_RMAX, "a larger start block than the rules hold");
static_assert((int)(MT_RMAX / MT_DS) + 1 - 256 <= MT_MAXN && MT_MAXN >= 128, "a longer block than the rules hold");
#define MT_RULE_DOUBLES (2 * (MT_MAXN * MT_N + MT_NSTART * MT_M))

__device__ static inline double gram_b2(double k, double N)      /* squared off-diagonal of the Jacobi matrix */
{
    return (k * k) * (N * N - k * k) / (4.0 * (4.0 * k * k - 1.0));
}

/* one work item per node: its root by bisection on the Sturm count, its
 * weight as Christoffel's number */
__global__ void __launch_bounds__(64) k_gram_rules(double *rules)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= MT_RULE_DOUBLES / 2) return;
    int N, n, j;
    const bool half = i >= MT_MAXN * MT_N;
    if (half) { N = 2 * (MT_S0 << ((i - MT_MAXN * MT_N) / MT_M)); n = 2 * MT_M; j = MT_M + (i - MT_MAXN * MT_N) % MT_M; }
    else { N = i / MT_N + 1; n = N < MT_N ? N : MT_N; j = i % MT_N; }
    double t = 0.5, w = 0.0;                      /* beyond a short rule's points: weight 0 */
    if (N <= n) {
        if (j < N) { t = (double)j + 0.5; w = 1.0; }
    } else {
        /* root j (from below) in centred coordinates: the values of the
         * monic polynomials at x agree in sign with their predecessors as
         * often as there are roots below x (no quotients: a chain of
         * 64 x 15 divisions took 109 us) */
        const double dN = (double)N;
        double lo = -0.5 * dN, hi = 0.5 * dN, bb[2 * MT_M];
#pragma unroll
        for (int k = 1; k < 2 * MT_M; ++k) bb[k] = gram_b2((double)k, dN);
        for (int it = 0; it < 64; ++it) {
            const double x = 0.5 * (lo + hi);
            double p0 = 1.0, p1 = x;
            int below = x > 0.0;
#pragma unroll
            for (int k = 1; k < 2 * MT_M; ++k) {
                const double p2 = __builtin_fma(x, p1, -bb[k] * p0);
                below += k < n && (p2 > 0.0) == (p1 > 0.0);
                p0 = p1; p1 = p2;
            }
            if (below > j) hi = x; else lo = x;
        }
        const double x = 0.5 * (lo + hi);
        double pm = 0.0, p = 1.0 / p2m_sqrt(dN), sum = p * p, bm = 0.0;
        for (int k = 1; k < n; ++k) {
            const double bk = p2m_sqrt(gram_b2((double)k, dN));
            const double q = (x * p - bm * pm) / bk;
            pm = p; p = q; bm = bk;
            sum += p * p;
        }
        w = 1.0 / sum;
        t = half ? x : x + 0.5 * dN;
    }
    rules[2 * i] = t;
    rules[2 * i + 1] = w;
}

/* per (chi, M): the fit parameters and prefactors; per (chi, r): chi times
 * the sine of the angle.  One work item each. */
__global__ void __launch_bounds__(64) k_maptable_cells(MTArgs A)
{
    const int64_t item = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t ncm = (int64_t)A.nchit * A.nmht;
    if (item >= ncm + (int64_t)A.nchit * A.nrt) return;
    const bool is_cm = item < ncm;
    const int per = is_cm ? A.nmht : A.nrt;
    const int64_t at = is_cm ? item : item - ncm;
    const int i = (int)(at / per) + 1, j = (int)(at % per) + 1;
    const double dz_r = 6.0 / 9999.0, dr_z = 1.3e4 / 9999.0;
    const double chit = p2m_exp(p2m_log(A.chimint) + (double)(i - 1) * A.dchit);
    const double z = mt_lookup(A.zofr, dr_z, chit);
    if (!is_cm) {
        const double chi = mt_lookup(A.rofz, dz_r, z);
        const double rt = p2m_exp(p2m_log(A.rmint) + (double)(j - 1) * A.drt);
        const double theta = p2m_atan(rt / chit);
        A.proj[at] = chi * p2m_sin(theta);
        return;
    }
    double z1 = 1.0 + z;
    double zc = (z1 * z1) * z1;
    double zfacy = A.omegam * zc + A.omegal;
    double rhoc = (A.rhocrit_0 * (A.omegam * zc + A.omegal)) / zc;
    double zfact = (1.0 / (1.0 + z)) / p2m_pow(rhoc, 1.0 / 3.0);
    CellCM c;
    c.Gx = 0.0;
    if (A.nu > 0.0) {
        double x0new = A.x0const * p2m_pow(1.0 + z, A.alpha_cmb);
        double ex = p2m_exp(x0new);
        c.Gx = ((x0new * (ex + 1.0)) / (ex - 1.0)) - 4.0;
    }
    double mht = p2m_exp(p2m_log(A.mhmint) + (double)(j - 1) * A.dmht);
    double mht3 = p2m_pow(mht, 1.0 / 3.0);
    const int mi = A.mi;
    c.P0 = mt_fit(A.b.P0_Am[mi], A.b.P0_alpham[mi], A.b.P0_alphaz[mi], mht, z);
    const double xc = mt_fit(A.b.xc_Am[mi], A.b.xc_alpham[mi], A.b.xc_alphaz[mi], mht, z);
    c.ixc = 1.0 / xc;
    c.gl = -MT_GAMMA * p2m_log(xc);
    c.beta = mt_fit(A.b.beta_Am[mi], A.b.beta_alpham[mi], A.b.beta_alphaz[mi], mht, z);
    c.P0r = mt_fit(A.b.P0_Am_rho[mi], A.b.P0_alpham_rho[mi], A.b.P0_alphaz_rho[mi], mht, z);
    c.alr = mt_fit(A.b.alpha_Am_rho[mi], A.b.alpha_alpham_rho[mi], A.b.alpha_alphaz_rho[mi], mht, z);
    const double betar = mt_fit(A.b.beta_Am_rho[mi], A.b.beta_alpham_rho[mi], A.b.beta_alphaz_rho[mi], mht, z);
    c.er = (-1.0 * (betar - MT_GAMMA_RHO)) / c.alr;
    c.rvir = p2m_pow(((((3.0 * mht) / 4.0) / COSMO_PI) / A.Delta) / rhoc, 1.0 / 3.0);
    c.cy = (A.y0 * mht) * zfacy;
    c.ctau = (A.tau0 * mht3) * zfact;
    A.cm[at] = c;
}

/* One work item per node, r fastest.  Bound: FP64 VALU.  The reference's
 * two sums take up to 401 points each and five powers a point; here both
 * share their nodes (one square root, three logarithms and three exponentials
 * a node for both) and take 30 to 71 nodes for y, by the start block, and 11
 * more for the rest of rho's sum.  A wave takes the start block that its smallest b allows.
 * 100 x 100 x 200 nodes: 0.98 ms (15.9 ms point by point). */
__global__ void __launch_bounds__(256) k_make_maptable(MTArgs A)
{
    const int64_t total = (int64_t)A.nchit * A.nmht * A.nrt;
    const int64_t node = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t nd = node < total ? node : total - 1;
    const int k = (int)(nd % A.nrt);
    const int64_t cmi = nd / A.nrt;
    const CellCM c = A.cm[cmi];
    const double b = A.proj[(cmi / A.nmht) * A.nrt + k] / c.rvir;
    const double rmaxp = MT_RMAX;
    const bool in = !(b > rmaxp);
    double bmin = in ? b : rmaxp;
    for (int o = 32; o > 0; o >>= 1) bmin = fmin(bmin, __shfl_xor(bmin, o));
    bmin = dbl_uniform(bmin);
    /* start block: 16 points, or the largest S with S ds <= bmin / 2 */
    int sj = 0;
    while (sj + 1 < MT_NSTART && (double)(MT_S0 << (sj + 1)) * MT_DS <= 0.5 * bmin) ++sj;
    const int S = MT_S0 << sj;
    const bool sym = (double)S * MT_DS <= 0.5 * bmin;
    const double b2 = b * b;
    const int ny = (int)(rmaxp / MT_DS) + 1;
    const int nr = in ? (int)(p2m_sqrt(rmaxp * rmaxp - b2) / MT_DS) + 1 : 0;
    const double lhalf = 0x1.62e42fefa39efp-1;       /* ln 2 = -ln 0.5 */
    double ysum = 0.0, rsum = 0.0;
    auto rho = [&](double lx) {
        const double l = lx + lhalf;
        return f64_exp(__builtin_fma(c.er, f64_log(1.0 + f64_exp(c.alr * l)), -MT_GAMMA_RHO * l));
    };
    /* both integrands at s = (pos + t) ds with weights wy and wr */
    auto both = [&](double q, double wy, double wr) {
        const double s = q * MT_DS;
        const double s2 = __builtin_fma(s, s, b2);
        const double lx = 0.5 * f64_log(s2), x = f64_sqrt(s2);
        const double y = f64_exp(__builtin_fma(MT_GAMMA, lx, c.gl) - c.beta * f64_log(__builtin_fma(x, c.ixc, 1.0)));
        ysum = __builtin_fma(wy, y, ysum);
        rsum = __builtin_fma(wr, rho(lx), rsum);
    };
    const double first = nr >= S ? 1.0 : 0.0;
    if (sym) {
        const double *h = A.rules + 2 * (MT_MAXN * MT_N + sj * MT_M);
        for (int j = 0; j < MT_M; ++j) both(h[2 * j], h[2 * j + 1], first * h[2 * j + 1]);
    } else {
        for (int q = 0; q < S; ++q) both((double)q + 0.5, 1.0, first);
    }
    int edge = nr >= S ? S : 0;                      /* where rho's last, partial block starts */
    for (int pos = S; pos < ny; pos *= 2) {
        const int len = ny - pos < pos ? ny - pos : pos;
        const bool full = nr >= 2 * pos;
        const double *h = A.rules + 2 * MT_N * (len - 1);
        for (int j = 0; j < MT_N; ++j) both((double)pos + h[2 * j], h[2 * j + 1], full ? h[2 * j + 1] : 0.0);
        if (full) edge = 2 * pos;
    }
    const int rest = nr - edge;
    if (rest > 0) {
        const double *h = A.rules + 2 * MT_N * (rest - 1);
        for (int j = 0; j < MT_N; ++j) {
            const double s = ((double)edge + h[2 * j]) * MT_DS;
            rsum = __builtin_fma(h[2 * j + 1], rho(0.5 * f64_log(__builtin_fma(s, s, b2))), rsum);
        }
    }
    const double yint = in ? (c.P0 * ysum) * MT_DS : 0.0;
    const double rint = in ? 2.0 * ((c.P0r * rsum) * MT_DS) : 0.0;
    double y = c.cy * yint;
    if (A.nu > 0.0) y = y * c.Gx;
    const double tau = c.ctau * rint;
    if (node < total) reinterpret_cast<float2 *>(A.table)[node] = make_float2((float)y, (float)tau);
}

static double mt_dzdr(double h, double om, double z)
{
    double z1 = 1.0 + z;
    return ((h * 100.0) / (2.99792458e10 / 1e5)) * p2m_sqrt((om * ((z1 * z1) * z1) + 1.0) - om);
}

extern "C" int p2m_make_maptable(int32_t device, int32_t model, double nu, double alpha_cmb,
                                 int32_t nchit, int32_t nmht, int32_t nrt,
                                 int32_t hdr_i[3], float hdr_f[6], float *table, int64_t n_table)
{
    if (!hdr_i || !hdr_f || !table) return P2M_E_INVALID;
    if (model < 1 || model > 3 || nchit < 2 || nmht < 2 || nrt < 2) return P2M_E_INVALID;
    if (n_table != 2LL * nchit * nmht * nrt) return P2M_E_SIZE;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) { (void)hipGetLastError(); return P2M_E_NODEVICE; }
    if (device < 0 || device >= ndev) return P2M_E_INVALID;
    if (hipSetDevice(device) != hipSuccess) return P2M_E_HIP;
    /* make_maptable.f90:33-43 */
    const double omegam = 0.25, omegab = 0.043, omegal = 0.75, h = 0.7;
    const double fb = omegab / omegam;
    const int n = 10000;
    /* maptable.f90:56-64 and the cosmology.f90:13-33 parameters */
    const double sigmat = 6.65246e-25, me = 9.109383e-28, mue = (double)1.136f, mp = (double)1.67e-24f;
    const double msun = 1.9891e33, mpc2km = 3.08567758e19, mpc = 3.08567758e24, kpc = 3.08567758e21;
    const double cc = 2.99792458e10, h100 = 100.0 / mpc2km;
    MTArgs A;
    A.b = kBBPS;
    A.mi = model - 1;
    A.nchit = nchit; A.nmht = nmht; A.nrt = nrt;
    A.nu = nu; A.alpha_cmb = alpha_cmb;
    A.Delta = model == 2 ? 500.0 : 200.0;
    const double m2rfac = p2m_pow(((3.0 / 4.0) / COSMO_PI) / A.Delta, 1.0 / 3.0);
    const double ypermass = ((((((3.0 * sigmat) * (h100 * h100)) / 8.0) / COSMO_PI) / me) / (cc * cc)) * msun / (double)1.932f;
    const double taupersigma = ((((sigmat / mue) / mp) * msun) / (kpc * kpc * kpc)) * mpc * 1e10;
    A.y0 = ((fb * A.Delta) * (h * h)) * ypermass;
    A.tau0 = (taupersigma * (h * h)) * m2rfac;
    A.x0const = 0.017612 * nu;
    A.omegam = omegam; A.omegal = omegal; A.rhocrit_0 = 2.775e11 * (0.7 * 0.7);
    /* maptable.f90:69-87; bounds as the float32 values of the header */
    const double chimint = (double)1e2f, chimaxt = (double)7e3f, mhmint = (double)1e13f, mhmaxt = (double)1e16f;
    const double rmint = (double)1e-2f, rmaxt = (double)10.0f;
    A.chimint = chimint; A.mhmint = mhmint; A.rmint = rmint;
    A.dchit = (p2m_log(chimaxt) - p2m_log(chimint)) / (double)(nchit - 1);
    A.dmht = (p2m_log(mhmaxt) - p2m_log(mhmint)) / (double)(nmht - 1);
    A.drt = (p2m_log(rmaxt) - p2m_log(rmint)) / (double)(nrt - 1);
    hdr_i[0] = nchit; hdr_i[1] = nmht; hdr_i[2] = nrt;
    hdr_f[0] = (float)chimint; hdr_f[1] = (float)chimaxt; hdr_f[2] = (float)mhmint;
    hdr_f[3] = (float)mhmaxt; hdr_f[4] = (float)rmint; hdr_f[5] = (float)rmaxt;
    /* one block of device memory: the distance tables, the rules, the
     * per-pair values and the table */
    const int64_t ncm = (int64_t)nchit * nmht, nproj = (int64_t)nchit * nrt, total = ncm * nrt;
    const size_t o_z = sizeof(double) * n, o_rule = o_z + sizeof(double) * n,
                 o_proj = o_rule + sizeof(double) * MT_RULE_DOUBLES, o_cm = o_proj + sizeof(double) * nproj,
                 o_tab = o_cm + sizeof(CellCM) * ncm;
    char *d = nullptr;
    int rc = 0;
    if (hipMalloc((void **)&d, o_tab + sizeof(float) * n_table) != hipSuccess) rc = P2M_E_NOMEM;
    /* the rules are made while the host sums the distance tables */
    if (!rc) {
        A.rules = (double *)(d + o_rule);
        hipLaunchKernelGGL(k_gram_rules, dim3((MT_RULE_DOUBLES / 2 + 63) / 64), dim3(64), 0, 0, A.rules);
    }
    std::vector<double> rofz(n, 0.0), zofr(n, 0.0);
    double dz = 6.0 / (double)(n - 1), dr = 1.3e4 / (double)(n - 1);
    for (int i = 2; i <= n; ++i) rofz[i - 1] = rofz[i - 2] + (1.0 / mt_dzdr(h, omegam, (double)(i - 1) * dz + 0.0)) * dz;
    for (int i = 2; i <= n; ++i) zofr[i - 1] = zofr[i - 2] + mt_dzdr(h, omegam, zofr[i - 2]) * dr;
    if (!rc && (hipMemcpy(d, rofz.data(), sizeof(double) * n, hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(d + o_z, zofr.data(), sizeof(double) * n, hipMemcpyHostToDevice) != hipSuccess))
        rc = P2M_E_HIP;
    if (!rc) {
        A.rofz = (const double *)d; A.zofr = (const double *)(d + o_z);
        A.proj = (double *)(d + o_proj); A.cm = (CellCM *)(d + o_cm); A.table = (float *)(d + o_tab);
        hipLaunchKernelGGL(k_maptable_cells, dim3((unsigned)((ncm + nproj + 63) / 64)), dim3(64), 0, 0, A);
        /* fewer nodes than 512 workgroups of 256: single waves, spread over the CUs */
        const int wg = total < 512 * 256 ? 64 : 256;
        hipLaunchKernelGGL(k_make_maptable, dim3((unsigned)((total + wg - 1) / wg)), dim3(wg), 0, 0, A);
        if (hipGetLastError() != hipSuccess) rc = P2M_E_HIP;
    }
    if (!rc && hipMemcpy(table, d + o_tab, sizeof(float) * n_table, hipMemcpyDeviceToHost) != hipSuccess) rc = P2M_E_HIP;
    if (d) (void)hipFree(d);
    (void)hipGetLastError();
    return rc;
}
