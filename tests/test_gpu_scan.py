"""Catalogues whose (halo, tile) pair counts fill the one-workgroup scan's
threads, leave a remainder, and lie on either side of its largest size, in one
block and in several: membership equal to the oracle's."""
import numpy as np
import pytest

import p2mo
from matt_young_mapmaking_amd import abi, catalog

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,block", [(1, 1), (1022, 1022), (1023, 500), (1024, 1024), (5000, 4999), (16382, 16382),
                                     (16383, 8192), (16384, 16384), (20001, 20000)])
def test_pair_scan_sizes(n, block):
    print(f"\n[gpu scan] n={n} block={block}", flush=True)
    h = catalog.make_catalog(n, mlo=1e14, mhi=1e15)
    tab = abi.make_maptable(nchit=10, nmht=10, nrt=40)
    with abi.Painter(nside=256, npix_fs=64, membership=True) as p:
        p.set_run()
        p.load_table(0, *tab)
        p.stream_begin(n)
        for i in range(0, n, block):
            p.stream_push(h[i:i + block], index_base=i)
        p.stream_finish()
        assert p.stats()["n_painted"] == n
        hc, hh, fc, fh = p.membership()
    ref = p2mo.Oracle(*tab).paint(h, nside=256, npix=64, nthreads=8)
    assert np.array_equal(hc, ref["hp_count"]) and np.array_equal(hh, ref["hp_hash"])
    assert np.array_equal(fc, ref["fs_count"]) and np.array_equal(fh, ref["fs_hash"])
