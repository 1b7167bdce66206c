"""The FP64 painter on tiles of many pixels and maps, where the LDS holds few
waves beside the tile's sums and pixel vectors: six maps with the membership
arrays on 2048-pixel tiles, over wide discs, small ones and a dense field
(tiles painted in slices), against the oracle; and as many waves as fit, by
the time."""
import numpy as np
import pytest

import p2mo
from matt_young_mapmaking_amd import abi, catalog, devmem
from test_gpu_wide import halos

pytestmark = pytest.mark.gpu

TABS = [dict(model=1 + k % 3, nu=(148.0, 100.0, 353.0)[k % 3], nchit=12, nmht=9, nrt=37) for k in range(6)]


@pytest.mark.parametrize("n_maps,w,wg", [(6, 2048, 512), (6, 2048, 256), (5, 2048, 512), (6, 2048, 64)])
@pytest.mark.parametrize("what", ["wide", "small", "field"])
def test_tiles_of_many_maps(what, n_maps, w, wg):
    print(f"\n[gpu tile waves] {what} maps={n_maps} tile={w} threads={wg}", flush=True)
    h = {"wide": lambda: halos(30, 20), "small": lambda: catalog.make_catalog(3000, mlo=1e13, mhi=3e15),
         "field": lambda: catalog.make_catalog(8000, geom="patch", mlo=1e13, mhi=3e15, patch_deg=2.0)}[what]()
    tabs = [abi.make_maptable(**t) for t in TABS[:n_maps]]
    with abi.Painter(nside=256, n_maps=n_maps, precision=abi.PREC_FP64, membership=True) as p:
        p.set_run(zmin=0.0)
        for k, t in enumerate(tabs):
            p.load_table(k, *t)
        p.set_tile(w, wg)
        p.paint(h)
        hc, hh, _, _ = p.membership()
        for k, t in enumerate(tabs):
            ref = p2mo.Oracle(*t).paint(h, nside=256, nthreads=8, zmin=0.0)
            if k == 0:
                assert hc.any() and np.array_equal(hc, ref["hp_count"]) and np.array_equal(hh, ref["hp_hash"])
            hp, _ = p.maps(slot=k)
            nz = ref["hp"] != 0
            assert np.array_equal(hp != 0, nz)
            assert np.max(np.abs(hp[nz] / ref["hp"][nz] - 1)) <= 1e-12


def test_more_waves_take_less_time():
    """Eight waves asked for and one: as many as fit beside each other take at
    most 0.6 of one wave's time (with the pixel vectors in LDS one fits)."""
    d = devmem.DeviceArray(catalog.make_catalog(1000000, mlo=1e13, mhi=1e15))
    ms = {}
    for wg in (64, 512):
        with abi.Painter(nside=1024, n_maps=6, precision=abi.PREC_FP64, membership=True) as p:
            p.set_run()
            t = abi.make_maptable(nchit=40, nmht=40, nrt=200)
            for k in range(6):
                p.load_table(k, *t)
            p.set_tile(2048, wg)
            times = []
            for _ in range(5):
                p.clear()
                p.paint_device(d.address, 1000000)
                times.append(p.stats()["ms_tile"])
            ms[wg] = min(times)
    print(f"\n[gpu tile waves] {ms}", flush=True)
    assert ms[512] <= 0.6 * ms[64]
