"""The flat-sky painter on maps of one to a few tiles under many halos, where
a tile's pairs go to hundreds of lists: membership equal to the oracle's and
values within 1e-12 of it, in both tiled precisions; and the time on one tile
against a map of many tiles."""
import numpy as np
import pytest

import p2mo
from matt_young_mapmaking_amd import abi, catalog, devmem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32_COMP])
@pytest.mark.parametrize("npix,n_maps", [(3, 1), (16, 2), (64, 1), (65, 6)])
def test_many_halos_on_few_tiles(npix, n_maps, prec):
    print(f"\n[gpu flat small] npix={npix} maps={n_maps} precision={prec}", flush=True)
    tabs = [abi.make_maptable(nu=(148.0, 100.0, 353.0)[k % 3], nchit=12, nmht=9, nrt=37) for k in range(n_maps)]
    h = catalog.make_catalog(60000, geom="patch", mlo=1e13, mhi=3e15)
    with abi.Painter(npix_fs=npix, n_maps=n_maps, precision=prec, membership=True) as p:
        p.set_run()
        for k, t in enumerate(tabs):
            p.load_table(k, *t)
        p.paint(h)
        _, _, fc, fh = p.membership()
        assert p.stats()["n_upd_fs"] == fc.astype(np.int64).sum()
        for k, t in enumerate(tabs):
            ref = p2mo.Oracle(*t).paint(h, nside=0, npix=npix, nthreads=8)
            if k == 0:
                assert fc.any()
                assert np.array_equal(fc, ref["fs_count"]) and np.array_equal(fh, ref["fs_hash"])
            _, fs = p.maps(slot=k)
            nz = ref["fs"] != 0
            assert np.array_equal(fs != 0, nz)
            assert np.max(np.abs(fs[nz] / ref["fs"][nz] - 1), initial=0) <= 1e-12


def test_one_tile_takes_no_longer_than_many():
    """1e5 halos on 16 x 16 pixels (one tile) within five times their time on
    200 x 200 (52 tiles, more updates): in 64 lists it is nineteen times."""
    d = devmem.DeviceArray(catalog.make_catalog(100000, geom="patch", mlo=1e13, mhi=1e15))
    ms = {}
    for npix in (16, 200):
        with abi.Painter(npix_fs=npix) as p:
            p.set_run()
            p.load_table(0, *abi.make_maptable(nchit=40, nmht=40, nrt=200))
            t = []
            for _ in range(8):
                p.clear()
                p.paint_device(d.address, 100000)
                t.append(p.stats()["ms_finish"])
            ms[npix] = min(t)
    print(f"\n[gpu flat small] {ms}", flush=True)
    assert ms[16] <= 5 * ms[200]
