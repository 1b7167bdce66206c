"""p2m_fetch_maps in both precisions, the one the map is held in and the
other (converted on the device piece by piece): the float32 values are the
rounded float64 ones, the float64 values the float32 ones exactly, for maps
shorter than, equal to and longer than a piece of 2^24 values, HEALPix and
flat, into pageable and page-locked memory."""
import ctypes as C

import numpy as np
import pytest

from matt_young_mapmaking_amd import abi, catalog

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [abi.PREC_FP32_COMP, abi.PREC_FP64, abi.PREC_PLAIN_FP64])
@pytest.mark.parametrize("nside,npix", [(1, 1), (64, 129), (0, 4096), (0, 4099), (2048, 0)])
def test_both_precisions_agree(prec, nside, npix):
    print(f"\n[gpu fetch] precision={prec} nside={nside} npix={npix}", flush=True)
    h = catalog.make_catalog(3000, geom="patch", mlo=1e13, mhi=1e15)
    with abi.Painter(nside=nside, npix_fs=npix, precision=prec) as p:
        p.set_run()
        p.load_table(0, *abi.make_maptable(nchit=10, nmht=10, nrt=40))
        p.paint(h)
        for k, (m64, m32) in enumerate(zip(p.maps(dtype=np.float64), p.maps(dtype=np.float32))):
            if m64 is None:
                continue
            assert np.array_equal(m32, m64.astype(np.float32))
            if k == 0 and prec == abi.PREC_FP32_COMP:
                assert np.array_equal(m64, m32.astype(np.float64))
            assert nside == 1 or m64.any()
            # page-locked memory, both at once
            pin = p.host_array((3 * m64.size + 6) // 7 + 1).reshape(-1)
            a = pin[:m64.size]
            o = (m64.size + 1) // 2 * 2
            b = pin[o:o + 2 * m64.size].view(np.float64)
            f32, f64 = a.ctypes.data_as(C.POINTER(C.c_float)), b.ctypes.data_as(C.POINTER(C.c_double))
            args = (f32, f64, None, None) if k == 0 else (None, None, f32, f64)
            assert p.L.p2m_fetch_maps(p.ctx, 0, *args) == 0
            assert np.array_equal(a, m32) and np.array_equal(b, m64)
