"""A deflection is rounded to FP32 before it is subtracted from the ray's
position: a lens whose deflection ends in a product, and a source that gives
the ray's x, against the two operations in numpy."""
import numpy as np
import pytest

from lensed_amd._lib import LENSED_GRAPH
from lensed_amd.lensed import Context, SystemSpec

pytestmark = pytest.mark.gpu

LENS = """type = LENS;
params { { "x", POSITION_X }, { "y", POSITION_Y }, { "k", PARAMETER } };
data { float2 c; float k; };
static float2 deflection(local data* this, float2 x) { return this->k*(x - this->c); }
static void set(local data* this, float x, float y, float k) { this->c = (float2)(x, y); this->k = k; }
"""
SOURCE = """type = SOURCE;
params { { "s", PARAMETER } };
data { float s; };
static float brightness(local data* this, float2 x) { return this->s*x.%s; }
static void set(local data* this, float s) { this->s = s; }
"""


@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("n", [1, 40, 3000])  # a wave per 64 pixels and rays shared
def test_deflection_is_rounded_before_the_subtraction(tmp_path, monkeypatch, axis, n):
    (tmp_path / "linear.cl").write_text(LENS)
    (tmp_path / "position.cl").write_text(SOURCE % axis)
    monkeypatch.setenv("LENSED_OBJECTS_PATH", str(tmp_path))
    shape = (40, 56)
    ks = np.float32([0.1, 0.3, 0.7, 1.3, -0.37])
    spec = SystemSpec([("l", "linear"), ("s", "position")],
                      {"l.x": "unif 0 40", "l.y": "unif 0 40", "l.k": "unif -2 2", "s.s": "1"},
                      np.zeros(shape, np.float32), np.ones(shape, np.float32), rule="point")
    c = np.float32([20.3, 17.7])
    with Context(spec, max_batch=n, flags=LENSED_GRAPH) as ctx:
        for k in ks:
            phys = np.tile(np.array([c[0], c[1], k, 1.0]), (n, 1))
            py, px = np.mgrid[1:shape[0] + 1, 1:shape[1] + 1].astype(np.float32)
            x, centre = (px, c[0]) if axis == "x" else (py, c[1])
            want = x - k * (x - centre)
            assert want.dtype == np.float32
            assert np.array_equal(ctx.render(phys[0])["value"], want), k
            # (data of 0 and a weight of 1: chi^2 is the sum of the squares, summed
            # with compensation in FP32 over blocks of 512 pixels)
            logl = ctx.loglike_phys(phys)
            ref = -0.5 * np.sum((want * want).astype(np.float64))
            assert np.all(np.abs(logl - ref) <= 512 * 2.0 ** -47 * abs(ref)), k
