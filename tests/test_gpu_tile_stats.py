"""p2m_stats reports the workgroup that painted: the one set, or as many waves
as fit a CU's 160 KB of LDS beside the tile (six maps with the membership
arrays: 2048 pixels of 60 bytes leave room for six of the FP64 painter's 6 KB
waves); an autotuned call reports one of its trials'."""
import pytest

from matt_young_mapmaking_amd import abi, catalog

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,n_maps,mem,w,wg,launched", [
    (abi.PREC_FP64, 6, True, 2048, 512, 384), (abi.PREC_FP64, 6, True, 2048, 320, 320), (abi.PREC_FP64, 1, False, 1024, 256, 256),
    (abi.PREC_FP32_COMP, 1, False, 1024, 256, 256), (abi.PREC_FP32_COMP, 6, True, 2048, 128, 128)])
def test_launched_workgroup(prec, n_maps, mem, w, wg, launched):
    t = abi.make_maptable(nchit=12, nmht=9, nrt=37)
    with abi.Painter(nside=64, n_maps=n_maps, precision=prec, membership=mem) as p:
        p.set_run()
        for k in range(n_maps):
            p.load_table(k, *t)
        p.set_tile(w, wg)
        p.paint(catalog.make_catalog(500, mlo=1e13, mhi=1e15))
        s = p.stats()
        assert (s["tile_w"], s["tile_wg"]) == (w, launched)


def test_autotuned_workgroup():
    t = abi.make_maptable(nchit=12, nmht=9, nrt=37)
    with abi.Painter(nside=256, n_maps=6, precision=abi.PREC_FP64, membership=True) as p:
        p.set_run()
        for k in range(6):
            p.load_table(k, *t)
        p.paint(catalog.make_catalog(300000, mlo=1e13, mhi=1e15))
        s = p.stats()
        assert s["tile_w"] in (512, 1024, 2048) and s["tile_wg"] in (128, 256)
