"""Launches of few pixels: the render that shares a pixel's rays among the
waves of a block, and launches without the cull pass, against the same
candidates in launches that take the other routes: the same bits."""
import numpy as np
import pytest

from lensed_amd import workloads as W
from lensed_amd._lib import LENSED_GRAPH, LENSED_NO_CULL, LENSED_TABLE
from lensed_amd.lensed import Context, SystemSpec

pytestmark = pytest.mark.gpu

LENS = {"sie": ("x", "y", "r", "q", "pa"), "epl_plus_shear": ("x", "y", "r", "t", "q", "pa", "g1", "g2")}
SOURCE = {"gauss": ("x", "y", "sigma", "mag", "q", "pa"), "sersic": ("x", "y", "r", "mag", "n", "q", "pa")}


def make_spec(lens, source, shape, psf, rule, seed):
    h, w = shape
    r = max(2.0, min(h, w) / 8)
    cx, cy = (w + 1) / 2, (h + 1) / 2
    span = {"lens.x": (cx - 2, cx + 2), "lens.y": (cy - 2, cy + 2), "lens.r": (0.7 * r, 1.3 * r), "lens.t": (0.5, 1.5),
            "lens.q": (0.4, 0.95), "lens.pa": (0, 180), "lens.g1": (-0.1, 0.1), "lens.g2": (-0.1, 0.1),
            "source.x": (cx - 3, cx + 3), "source.y": (cy - 3, cy + 3), "source.sigma": (0.1 * r, 0.2 * r),
            "source.r": (0.2 * r, 0.4 * r), "source.mag": (-4, 4), "source.n": (1, 3), "source.q": (0.4, 1),
            "source.pa": (0, 180)}
    ids = [f"lens.{p}" for p in LENS[lens]] + [f"source.{p}" for p in SOURCE[source]]
    rng = np.random.default_rng(seed)
    return SystemSpec([("lens", lens), ("source", source)], {k: "unif %g %g" % span[k] for k in ids},
                      rng.normal(0, 0.05, shape).astype(np.float32), np.full(shape, 400.0, np.float32),
                      psf=W.gaussian_psf(psf, 2.0) if psf else None, rule=rule)


# one square and fewer pixels than one; odd sizes; every count of rays per
# wave (4 and 1 rays: not shared; 16 and 17; 225: with the table too much
# LDS); counts that cull with a wave per square, cull with shared rays, and
# share without a cull pass
@pytest.mark.parametrize("lens,source,shape,psf,rule,flags", [
    ("sie", "sersic", (100, 100), 0, "g3k7", 0), ("sie", "sersic", (5, 3), 0, "gm75", 0),
    ("epl_plus_shear", "gauss", (97, 131), 7, "g3k7", 0), ("epl_plus_shear", "gauss", (64, 200), 21, "g3k7", LENSED_TABLE),
    ("epl_plus_shear", "sersic", (33, 65), 5, "g5k11", LENSED_TABLE), ("epl_plus_shear", "gauss", (40, 24), 0, "g7k15", LENSED_TABLE),
    ("epl_plus_shear", "gauss", (40, 24), 0, "g7k15", 0), ("sie", "gauss", (48, 48), 9, "sub4", 0),
    ("sie", "gauss", (48, 48), 9, "sub2", 0), ("epl_plus_shear", "gauss", (70, 33), 5, "point", LENSED_TABLE)])
def test_small_launches_keep_the_bits(lens, source, shape, psf, rule, flags):
    spec = make_spec(lens, source, shape, psf, rule, 7)
    squares = 4 * ((shape[0] + 15) // 16) * ((shape[1] + 15) // 16)
    n = 40000 // squares  # more than any rule's line
    cubes = np.random.default_rng(8).random((n, len(LENS[lens]) + len(SOURCE[source])))
    with Context(spec, max_batch=n, flags=flags | LENSED_GRAPH) as ctx:
        full, _ = ctx.loglike_batch(cubes)
        assert np.all(np.isfinite(full))
        for k in sorted({1, 2, max(1, 1000 // squares), max(1, 2500 // squares), max(1, 6000 // squares),
                         max(1, 12000 // squares)}):
            part, _ = ctx.loglike_batch(cubes[n // 2:n // 2 + k])
            assert np.array_equal(part, full[n // 2:n // 2 + k]), k
        again, phys = ctx.loglike_batch(cubes)  # the cull after launches that left every pixel written
        assert np.array_equal(again, full)
        p = np.zeros(ctx.npars())
        p[ctx.pmap()] = phys[3]
        planes = ctx.render(p)
        assert ctx.loglike(cubes[3])[0] == full[3]
    with Context(spec, max_batch=n, flags=flags | LENSED_GRAPH | LENSED_NO_CULL) as ctx:
        every, _ = ctx.loglike_batch(cubes)
        assert np.array_equal(every, full)
        assert np.array_equal(ctx.render(p)["error"], planes["error"])


def test_shared_rays_beside_a_large_system():
    """Three candidates with the rays shared (a system alone) and with a wave
    per square (the same system beside a large one, whose squares alone pass
    the line)."""
    small = make_spec("sie", "sersic", (61, 77), 7, "g3k7", 3)
    big = make_spec("sie", "sersic", (512, 512), 7, "g3k7", 4)
    rng = np.random.default_rng(5)
    with Context(small, max_batch=3, flags=LENSED_GRAPH) as ctx:
        alone, phys = ctx.loglike_batch(rng.random((3, 12)))
    with Context([small, big], max_batch=3, flags=LENSED_GRAPH) as ctx:
        both = [np.zeros((3, 12)), np.zeros((3, 12))]
        both[0][:, ctx.pmap(0)] = phys
        both[1][:, ctx.pmap(1)] = ctx.loglike_batch(rng.random((3, 12)), 1)[1]
        together = ctx.loglike_phys(both)
    assert np.array_equal(together[0], alone)
