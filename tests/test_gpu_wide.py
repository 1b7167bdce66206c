"""Catalogues of wide discs (nearby halos), whose (halo, tile) pairs are
mostly whole tiles, hundreds a halo: both tiled precisions against the oracle
at small and large tiles, one wave to eight a workgroup, discs over the poles
and over the azimuth's wrap among small ones; and the time of the binning
against as many pairs of small discs."""
import numpy as np
import pytest

import p2mo
from matt_young_mapmaking_amd import abi, catalog, devmem

pytestmark = pytest.mark.gpu


def halos(n, small=0):
    """n halos 25 to 60 Mpc away (discs of about 0.1 to 0.4 rad), the first few over the poles and the wrap."""
    rng = np.random.default_rng(5)
    mu, ph = 2 * rng.random(n) - 1, 2 * np.pi * rng.random(n)
    s = np.sqrt(1 - mu * mu)
    u = np.stack([s * np.cos(ph), s * np.sin(ph), mu], 1)
    u[:4] = [[0, 0, 1], [0, 0, -1], [-1, 0, 0], [-1, 1e-3, 0.2]]
    u /= np.sqrt((u * u).sum(1))[:, None]
    r = rng.uniform(25, 60, n)
    h = np.zeros((n, 7), np.float32)
    h[:, :3] = u * r[:, None]
    h[:, 6] = rng.uniform(15, 25, n)
    return np.concatenate([h, catalog.make_catalog(small, mlo=1e13, mhi=1e15)]) if small else h


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32_COMP])
@pytest.mark.parametrize("nside,small,w,wg,n_maps", [
    (128, 0, 1024, 256, 1), (256, 0, 64, 256, 1), (512, 0, 2048, 128, 2), (256, 500, 1024, 192, 1), (64, 0, 512, 64, 6),
    (1024, 0, 256, 256, 1)])
def test_wide_discs(nside, small, w, wg, n_maps, prec):
    print(f"\n[gpu wide] nside={nside} small={small} tile={w} threads={wg} maps={n_maps} precision={prec}", flush=True)
    tabs = [abi.make_maptable(model=1 + k % 3, nchit=12, nmht=9, nrt=37) for k in range(n_maps)]
    h = halos(40, small)
    with abi.Painter(nside=nside, n_maps=n_maps, precision=prec, membership=True) as p:
        p.set_run(zmin=0.0)
        for k, t in enumerate(tabs):
            p.load_table(k, *t)
        p.set_tile(w, wg)
        p.paint(h)
        s = p.stats()
        hc, hh, _, _ = p.membership()
        for k, t in enumerate(tabs):
            ref = p2mo.Oracle(*t).paint(h, nside=nside, nthreads=8, zmin=0.0)
            if k == 0:
                assert ref["stats"]["n_painted"] >= 40 and hc.max() > 1
                assert np.array_equal(hc, ref["hp_count"]) and np.array_equal(hh, ref["hp_hash"])
                assert (s["n_listed_hp"], s["n_upd_hp"]) == (ref["stats"]["n_listed_hp"], ref["stats"]["n_upd_hp"])
            hp, _ = p.maps(slot=k)
            nz = ref["hp"] != 0
            assert np.array_equal(hp != 0, nz)
            assert np.max(np.abs(hp[nz] / ref["hp"][nz] - 1)) <= (1e-12 if prec == abi.PREC_FP64 else 1e-6)


def test_wide_discs_are_binned_as_fast_as_small_ones():
    """The binning of 100 discs over some 400 tiles each within twice that of
    40000 halos of about one tile each (by one lane a halo it is more than
    three times)."""
    ms = {}
    for name, h in (("wide", halos(100)), ("small", catalog.make_catalog(40000, mlo=1e13, mhi=1e15))):
        d = devmem.DeviceArray(h)
        with abi.Painter(nside=1024) as p:
            p.set_run(zmin=0.0)
            p.load_table(0, *abi.make_maptable(nchit=40, nmht=40, nrt=200))
            p.set_tile(1024, 256)
            t = []
            for _ in range(8):
                p.clear()
                p.paint_device(d.address, len(h))
                t.append(p.stats()["ms_bin"])
            ms[name] = min(t)
    print(f"\n[gpu wide] {ms}", flush=True)
    assert ms["wide"] <= 2 * ms["small"]
