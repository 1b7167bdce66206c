"""Tiles of many pairs, painted in slices by several workgroups: catalogues of
a small field against the oracle, in both tiled precisions, with one to six
maps, small and large tiles, at the equator and at a pole; two catalogues
into one map; deferred pixels that do not fit their list, so that split tiles
lose slices and are painted again; and the time of a field against an even
sky's."""
import numpy as np
import pytest

import p2mo
from matt_young_mapmaking_amd import abi, catalog, devmem

pytestmark = pytest.mark.gpu


def halos(n, deg, pole=False):
    h = catalog.make_catalog(n, geom="patch", mlo=1e13, mhi=1e15, patch_deg=deg)
    return np.ascontiguousarray(h[:, [2, 1, 0, 3, 4, 5, 6]]) if pole else h


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32_COMP])
@pytest.mark.parametrize("nside,deg,pole,w,wg,n_maps,fb_cap", [
    (64, 3.0, False, 1024, 256, 1, 0), (256, 1.0, False, 1024, 256, 2, 0), (512, 2.0, True, 2048, 256, 1, 0),
    (128, 4.0, False, 64, 64, 6, 0), (1024, 0.5, False, 1024, 256, 3, 0), (2048, 0.5, False, 1024, 256, 1, 64),
    (2048, 0.5, True, 512, 128, 1, 64)])
def test_split_tiles(nside, deg, pole, w, wg, n_maps, fb_cap, prec, monkeypatch):
    print(f"\n[gpu split] nside={nside} field={deg} pole={pole} tile={w} threads={wg} maps={n_maps} list={fb_cap} "
          f"precision={prec}", flush=True)
    if fb_cap:
        monkeypatch.setenv("P2M_FB_CAP", str(fb_cap))
    tabs = [abi.make_maptable(model=1 + k % 3, nu=(148.0, 100.0, 353.0)[k % 3], nchit=12, nmht=9, nrt=37)
            for k in range(n_maps)]
    h = halos(24000, deg, pole)
    parts = ((0, len(h)),) if n_maps > 1 else ((0, 15000), (15000, len(h)))
    with abi.Painter(nside=nside, n_maps=n_maps, precision=prec, membership=True) as p:
        p.set_run()
        for k, t in enumerate(tabs):
            p.load_table(k, *t)
        p.set_tile(w, wg)
        listed = upd = redo = 0
        for lo, hi in parts:
            p.paint(h[lo:hi], index_base=lo)
            s = p.stats()
            listed += s["n_listed_hp"]
            upd += s["n_upd_hp"]
            redo += s["n_redo_tiles"]
        assert (redo > 0) == bool(fb_cap and prec == abi.PREC_FP32_COMP)
        hc, hh, _, _ = p.membership()
        for k, t in enumerate(tabs):
            ref = p2mo.Oracle(*t).paint(h, nside=nside, nthreads=8)
            if k == 0:
                assert np.array_equal(hc, ref["hp_count"]) and np.array_equal(hh, ref["hp_hash"])
                assert upd == hc.astype(np.int64).sum() == ref["stats"]["n_upd_hp"]
                assert listed == ref["stats"]["n_listed_hp"]
            hp, _ = p.maps(slot=k)
            nz = ref["hp"] != 0
            assert nz.any() and np.array_equal(hp != 0, nz)
            assert np.max(np.abs(hp[nz] / ref["hp"][nz] - 1)) <= (1e-12 if prec == abi.PREC_FP64 else 1e-6)


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32_COMP])
def test_field_takes_no_longer_than_a_sky(prec):
    """As many halos in a 10 x 10 degree field as over the sky keep the GPU as
    busy: the tile painter within four times the sky's time (in one workgroup
    per tile it is 10 times and more)."""
    ms = {}
    for geom in ("sky", "patch"):
        d = devmem.DeviceArray(catalog.make_catalog(1000000, geom=geom, mlo=1e13, mhi=1e15))
        with abi.Painter(nside=512, precision=prec) as p:
            p.set_run()
            p.load_table(0, *abi.make_maptable(nchit=40, nmht=40, nrt=200))
            p.set_tile(1024, 256)
            t = []
            for _ in range(8):
                p.clear()
                p.paint_device(d.address, 1000000)
                t.append(p.stats()["ms_tile"])
            ms[geom] = min(t)
    print(f"\n[gpu split] precision={prec} {ms}", flush=True)
    assert ms["patch"] <= 4 * ms["sky"]
