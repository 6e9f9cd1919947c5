"""The column sweep with its strips cut into parts (launches of few strips)
against the tile kernel: the same bits, whatever the split."""
import numpy as np
import pytest

from lensed_amd import workloads as W
from lensed_amd._lib import LENSED_GRAPH, LENSED_TABLE
from lensed_amd.lensed import Context, SystemSpec

pytestmark = pytest.mark.gpu

NAMES = ("x", "y", "r", "t", "q", "pa", "g1", "g2", "x", "y", "sigma", "mag", "q", "pa")


# one strip and many; one block of rows, a last block of 1 and of 7 rows; the
# smallest PSFs that are taken apart into two passes, the largest of the sweep,
# even and odd sides; whole strips (1100 candidates of four strips) down to a
# part per block.  PSFs too small to gain from two passes take no sweep.
@pytest.mark.parametrize("shape,psf,n", [((8, 40), (3, 3), 1), ((9, 64), (21, 1), 3), ((57, 65), (1, 21), 2),
                                         ((257, 130), (21, 21), 1), ((512, 70), (4, 21), 5),
                                         ((63, 200), (20, 7), 300), ((40, 256), (21, 21), 1100),
                                         ((8, 40), (4, 4), 1), ((9, 64), (21, 3), 3), ((57, 65), (3, 21), 2)])
@pytest.mark.parametrize("flags", [LENSED_GRAPH, LENSED_GRAPH | LENSED_TABLE])
def test_parts_equal_tiles(shape, psf, n, flags):
    h, w = shape
    r = max(3.0, min(h, w) / 6)
    span = {"x": ((w + 1) / 2 - 2, (w + 1) / 2 + 2), "y": ((h + 1) / 2 - 2, (h + 1) / 2 + 2), "r": (0.7 * r, r),
            "t": (0.6, 1.4), "q": (0.5, 0.95), "pa": (0, 180), "g1": (-0.05, 0.05), "g2": (-0.05, 0.05),
            "sigma": (0.2, 0.7), "mag": (-3, 3)}
    ids = ["%s.%s" % ("lens" if i < 8 else "source", p) for i, p in enumerate(NAMES)]
    pri = {k: "unif %g %g" % span[k.split(".")[1]] for k in ids}
    side = max(psf)
    taps = W.gaussian_psf(side, 2.0)[(side - psf[0]) // 2:(side - psf[0]) // 2 + psf[0],
                                     (side - psf[1]) // 2:(side - psf[1]) // 2 + psf[1]].copy()
    rng = np.random.default_rng(h + w)
    image = rng.normal(0, 0.05, shape).astype(np.float32)
    spec = SystemSpec([("lens", "epl_plus_shear"), ("source", "gauss")], pri, image,
                      np.full(shape, 400.0, np.float32), psf=taps / taps.sum())
    cubes = rng.random((n, 14))
    got = []
    with Context(spec, max_batch=n, flags=flags) as ctx:
        for rows in (1, 8, 2):
            ctx.set_tuning(conv_rows=rows)
            lnew, phys = ctx.loglike_batch(cubes)
            if rows != 1 or psf[0] * psf[1] >= 2 * sum(psf):
                assert ctx.tuning()["conv_rows"] == rows
            p = np.zeros(14)
            p[ctx.pmap()] = phys[0]
            got.append((lnew, ctx.render(p)))
    for lnew, planes in got[1:]:
        assert np.all(np.isfinite(lnew)) and np.array_equal(lnew, got[0][0])
        for k in planes:
            assert np.array_equal(planes[k], got[0][1][k]), k
