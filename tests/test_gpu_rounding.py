"""Which products the ray loop fuses with the sum that follows, against the
same operations one by one on the host: logL has the bits of these pairings."""
from fractions import Fraction

import numpy as np
import pytest

from lensed_amd._lib import LENSED_GRAPH, LENSED_TABLE
from lensed_amd.lensed import Context, SystemSpec

pytestmark = pytest.mark.gpu

LENS = """type = LENS;
params { { "x", POSITION_X }, { "y", POSITION_Y }, { "k", PARAMETER } };
data { float2 c; float k; };
static float2 deflection(local data* this, float2 x)
{
    return %s;
}
static void set(local data* this, float x, float y, float k) { this->c = (float2)(x, y); this->k = k; }
"""
SOURCE = """type = SOURCE;
params { { "s", PARAMETER } };
data { float s; };
static float brightness(local data* this, float2 x) { return this->s*x.%s; }
static void set(local data* this, float s) { this->s = s; }
"""


def fma(a, b, c):
    return np.float32(float(Fraction(float(a)) * Fraction(float(b)) + Fraction(float(c))))


# a lens whose deflection ends in a product, and a source that gives the ray's
# position: the deflection is rounded before it is subtracted
@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("form", ["this->k*(x - this->c)", "mv22((mat22)(1, 0, 0, 1), x - this->c)*this->k",
                                  "mv22((mat22)(1, 0, 0, 1), this->k*(x - this->c))"])
@pytest.mark.parametrize("n", [1, 40, 3000])  # a wave per 64 pixels and rays shared
def test_deflection_is_rounded_before_the_subtraction(tmp_path, monkeypatch, axis, form, n):
    (tmp_path / "linear.cl").write_text(LENS % form)
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


# a sky with a gradient behind nothing, a lens and a tabulated lens (dark
# sources: what they add is 0): level + fma(gx, x - 1, gy (y - 1)), and the
# level alone without a gradient
@pytest.mark.parametrize("objects,flags", [(["sky"], 0), (["sie", "sersic", "sky"], 0), (["epl", "sersic", "sky"], LENSED_TABLE),
                                           (["epl_plus_shear", "gauss", "gauss", "sky"], LENSED_TABLE)])
@pytest.mark.parametrize("grad", [(0.0, 0.0), (1.3e-3, -7.7e-4), (0.0, 3.1e-4)])
def test_sky_gradient_is_one_fma(objects, flags, grad):
    shape, level = (33, 50), np.float32(0.0173)
    gx, gy = np.float32(grad)
    values = {"x": 25.2, "y": 16.4, "r": 5.0, "t": 1.1, "q": 0.7, "pa": 40.0, "g1": 0.02, "g2": -0.03, "sigma": 0.01,
              "n": 1.0, "mag": 400.0, "bg": float(level), "dx": float(gx), "dy": float(gy)}
    params = {"sky": "bg dx dy", "sie": "x y r q pa", "epl": "x y r t q pa", "epl_plus_shear": "x y r t q pa g1 g2",
              "sersic": "x y r mag n q pa", "gauss": "x y sigma mag q pa"}
    pri = {f"o{i}.{p}": repr(values[p]) for i, n in enumerate(objects) for p in params[n].split()}
    spec = SystemSpec([(f"o{i}", n) for i, n in enumerate(objects)], pri, np.zeros(shape, np.float32),
                      np.ones(shape, np.float32), rule="point")
    with Context(spec, flags=flags) as ctx:
        got = ctx.render([values[p] for n in objects for p in params[n].split()])["value"]
    want = np.array([[level + fma(gx, np.float32(j), gy * np.float32(i)) for j in range(shape[1])]
                     for i in range(shape[0])], np.float32)
    assert np.array_equal(got, want)


PRODUCT = """type = SOURCE;
params { { "x", POSITION_X }, { "y", POSITION_Y }, { "s", PARAMETER } };
data { float2 c; float s; };
static float brightness(local data* this, float2 x) { return this->s*exp(%s); }
static void set(local data* this, float x, float y, float s) { this->c = (float2)(x, y); this->s = s; }
"""


# two products with exp(), the first behind a longer chain: the second product
# is fused with the sum in either order, the first is rounded (each exponential
# is read off with a factor of 1)
@pytest.mark.parametrize("lens", ["sis", "sie"])
@pytest.mark.parametrize("order", ["deep shallow", "shallow deep"])
def test_the_shallower_of_two_products_is_fused(tmp_path, monkeypatch, lens, order):
    (tmp_path / "deep.cl").write_text(PRODUCT % "-3.3f*sqrt(sqrt(length(x - this->c)/7))")
    (tmp_path / "shallow.cl").write_text(PRODUCT % "-length(x - this->c)/9")
    monkeypatch.setenv("LENSED_OBJECTS_PATH", str(tmp_path))
    shape = (33, 50)
    values = {"x": 25.3, "y": 16.4, "r": 5.0, "q": 0.7, "pa": 40.0}
    lp = {"sis": "x y r", "sie": "x y r q pa"}[lens].split()
    names = order.split()
    pri = {f"l.{p}": repr(values[p]) for p in lp}
    pri.update({f"{n}.{p}": "unif 0 60" for n in names for p in ("x", "y", "s")})
    spec = SystemSpec([("l", lens)] + [(n, n) for n in names], pri, np.zeros(shape, np.float32),
                      np.ones(shape, np.float32), rule="point")
    centre = {"deep": (20.1, 18.2), "shallow": (27.7, 13.9)}
    with Context(spec) as ctx:
        def value(**s):
            return ctx.render([values[p] for p in lp] + [v for n in names for v in (*centre[n], s.get(n, 0.0))])["value"]
        e = {n: value(**{n: 1.0}) for n in names}
        for s in (0.37, 1.7):
            s = {"deep": np.float32(s), "shallow": np.float32(1 / s)}
            got = value(**s)
            want = [[fma(s["shallow"], e["shallow"][i, j], s["deep"] * e["deep"][i, j]) for j in range(shape[1])]
                    for i in range(shape[0])]
            assert np.array_equal(got, np.array(want, np.float32)), s
