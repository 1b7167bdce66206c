"""The radial fraction of the FP64 painters (fr = ln r - ln r_node, maptable
f90:200) to the rounding that its terms carry, HEALPix and flat sky.

The table is 1 on the odd radial nodes and 0 on the even ones for every mass
and distance, so that in the cells from an even node to an odd one a pixel
of a single halo holds fr itself; the oracle's map holds the reference's.
Both sides round ln r (|ln r| < 4 over the table's range 0.02 .. 50) and the
same node value is taken from it.  In units of 1e-16, against exact numbers:
the oracle's argument of the logarithm is a root (1.1), an arc tangent (2 ulp,
4.4), a tangent (2 ulp, 4.4) and a product (1.1), its logarithm 2 ulp (8.9);
the painter's is two products under the root (1.1 together), its half
logarithm 2 ulp (8.9) and a sum (2.2).  That is 32 in the worst case and,
independent errors uniform within their bounds, at most 8.3 rms."""
import numpy as np
import pytest

import p2mo
from matt_young_mapmaking_amd import abi

pytestmark = pytest.mark.gpu

WORST, RMS = 3.2e-15, 8.3e-16


def table():
    hi = np.array([5, 6, 200], np.int32)
    hf = np.array([100, 7000, 1e13, 1e16, 0.02, 50], np.float32)
    t = np.zeros((5, 6, 200, 2), np.float32)
    t[:, :, ::2, :] = 1.0                     # nodes 1, 3, ... counted from 1
    return hi, hf, t.ravel()


def halos(n=300):
    """Halos that do not overlap much, 250 to 3000 Mpc away, some in the flat-sky field."""
    rng = np.random.default_rng(11)
    mu, ph = 2 * rng.random(n) - 1, 2 * np.pi * rng.random(n)
    s = np.sqrt(1 - mu * mu)
    u = np.stack([s * np.cos(ph), s * np.sin(ph), mu], 1)
    a = (rng.random((n // 3, 2)) - 0.5) * 0.17
    u[:n // 3] = np.stack([np.sqrt(1 - a[:, 0] ** 2 - a[:, 1] ** 2), a[:, 0], a[:, 1]], 1)
    r = np.exp(rng.uniform(np.log(250), np.log(3000), n))
    h = np.zeros((n, 7), np.float32)
    h[:, :3] = u * r[:, None]
    h[:, 6] = rng.uniform(8, 25, n)
    return h


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32_COMP])
def test_radial_fraction(prec):
    print(f"\n[gpu radial] precision={prec}", flush=True)
    h, t = halos(), table()
    nside, npix = (1024 if prec == abi.PREC_FP64 else 0), 1500
    with abi.Painter(nside=nside, npix_fs=npix, precision=prec, membership=True) as p:
        p.set_run()
        p.load_table(0, *t)
        p.set_tile(1024, 256)
        p.paint(h)
        hc, _, fc, _ = p.membership()
        hp, fs = p.maps()
    ref = p2mo.Oracle(*t).paint(h, nside=nside, npix=npix, nthreads=8)
    for what, got, want, cnt in (("healpix", hp, ref["hp"], hc), ("flat", fs, ref["fs"], fc)):
        if got is None:
            continue
        one = (cnt == 1) & (want < 0.5) & (want > 0)
        d = got[one] - want[one]
        rms = np.sqrt(np.mean(d * d))
        print(f"[gpu radial] {what}: {one.sum()} pixels, largest {np.abs(d).max():.2e}, rms {rms:.2e}", flush=True)
        assert one.sum() > 20000
        assert np.abs(d).max() <= WORST
        assert rms <= RMS
