"""The 64-row convolution tile, whose taps are held in vector registers, and
the rule that picks a launch's tile, against the 8-row tile: the same bits."""
import numpy as np
import pytest

from lensed_amd import workloads as W
from lensed_amd._lib import LENSED_GRAPH
from lensed_amd.lensed import Context, SystemSpec

pytestmark = pytest.mark.gpu


# direct (Moffat, and PSFs too small for two passes) and two passes, up to and
# beyond the 21 taps whose column pass holds them; sides of one tile and more,
# 1, 63 and 65 rows; launches on both sides of each line of the rule
@pytest.mark.parametrize("shape,psf,kind,n,rows", [
    ((65, 64), (31, 31), "moffat", 300, 16), ((63, 129), (9, 31), "moffat", 200, 16), ((1, 70), (3, 3), "gauss", 600, 16),
    ((64, 64), (21, 21), "gauss", 512, 16), ((130, 61), (31, 31), "gauss", 256, 16), ((33, 65), (22, 8), "gauss", 300, 16),
    ((65, 64), (31, 31), "moffat", 250, 8), ((64, 64), (21, 21), "gauss", 256, 8), ((65, 64), (31, 31), "moffat", 3, 2),
    ((70, 64), (63, 63), "gauss", 300, 8)])
def test_tall_tile_equals_short(shape, psf, kind, n, rows):
    h, w = shape
    side = max(psf)
    taps = W.gaussian_psf(side, 3.0) if kind == "gauss" else W.moffat_psf(side, 3.0, 3.0)
    taps = taps[(side - psf[0]) // 2:(side - psf[0]) // 2 + psf[0], (side - psf[1]) // 2:(side - psf[1]) // 2 + psf[1]]
    rng = np.random.default_rng(h * w)
    spec = SystemSpec([("lens", "sie"), ("source", "exponential")],
                      {"lens.x": f"unif {w / 2 - 2} {w / 2 + 2}", "lens.y": f"unif {h / 2 - 2} {h / 2 + 2}",
                       "lens.r": "unif 5 9", "lens.q": "unif 0.5 0.95", "lens.pa": "unif 0 180",
                       "source.x": f"unif {w / 2 - 3} {w / 2 + 3}", "source.y": f"unif {h / 2 - 3} {h / 2 + 3}",
                       "source.rs": "unif 0.5 2", "source.mag": "unif -3 3", "source.q": "unif 0.4 1",
                       "source.pa": "unif 0 180"}, rng.normal(0, 0.05, shape).astype(np.float32),
                      np.full(shape, 400.0, np.float32), psf=taps / taps.sum(), rule="sub2")
    cubes = rng.random((n, 11))
    with Context(spec, max_batch=n, flags=LENSED_GRAPH) as ctx:
        lnew, phys = ctx.loglike_batch(cubes)
        assert ctx.tuning()["conv_rows"] == rows  # (on 256 CUs)
        p = np.zeros(11)
        p[ctx.pmap()] = phys[n // 2]
        for r in (2, 16):
            ctx.set_tuning(conv_rows=r)
            other, _ = ctx.loglike_batch(cubes)
            planes = ctx.render(p)
            if r == 2:
                first = planes
            assert np.all(np.isfinite(other)) and np.array_equal(other, lnew), r
            for k in planes:
                assert np.array_equal(planes[k], first[k]), (r, k)
