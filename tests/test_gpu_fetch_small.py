"""p2m_fetch_maps in the other precision around the size from which the
device converts (256 KB of the map as held): values as the map's own, and a
small map without the time of a launch."""
import ctypes as C
import time

import numpy as np
import pytest

from matt_young_mapmaking_amd import abi, catalog

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [abi.PREC_FP32_COMP, abi.PREC_FP64])
@pytest.mark.parametrize("nside,npix", [(1, 3), (32, 180), (64, 181), (64, 182), (128, 256), (64, 257)])
def test_values_on_both_sides(prec, nside, npix):
    h = catalog.make_catalog(2000, geom="patch", mlo=1e13, mhi=1e15)
    with abi.Painter(nside=nside, npix_fs=npix, precision=prec) as p:
        p.set_run()
        p.load_table(0, *abi.make_maptable(nchit=10, nmht=10, nrt=40))
        p.paint(h)
        (hp64, fs64), (hp32, fs32) = p.maps(dtype=np.float64), p.maps(dtype=np.float32)
        assert np.array_equal(hp32, hp64.astype(np.float32)) and np.array_equal(fs32, fs64.astype(np.float32))
        if prec == abi.PREC_FP32_COMP:
            assert np.array_equal(hp64, hp32.astype(np.float64))
        assert fs64.any()


def test_small_maps_are_not_converted_by_a_launch():
    """768 values in the other precision within 6 us of the same map in its
    own (least of 400 each): a launch and its wait take some 10."""
    with abi.Painter(nside=8, precision=abi.PREC_FP64) as p:
        p.clear()
        f32, f64 = np.zeros(768, np.float32), np.zeros(768)
        us = {"own": [], "other": []}
        args = {"own": (None, abi._p(f64, C.c_double), None, None), "other": (abi._p(f32, C.c_float), None, None, None)}
        for _ in range(400):
            for name, a in args.items():
                t0 = time.perf_counter()
                assert p.L.p2m_fetch_maps(p.ctx, 0, *a) == 0
                us[name].append(1e6 * (time.perf_counter() - t0))
        us = {k: min(v) for k, v in us.items()}
        print(f"\n[gpu fetch] {us}", flush=True)
        assert us["other"] <= us["own"] + 6
