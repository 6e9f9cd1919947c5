"""The host's launch code on the CPU: a child process with a HIP runtime
without a device preloaded (hip_stub.cpp), whose kernels do nothing."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
sys.path[:0] = [%r, %r]
import numpy as np
from lensed_amd import _lib as L
from lensed_amd.lensed import Context, LensedError, SystemSpec
stub = ctypes.CDLL(None)
stub.stub_log.restype = ctypes.c_char_p

def launches():
    lines = [s.split() for s in stub.stub_log().decode().splitlines()]
    stub.stub_clear()
    return {name: (int(blocks), int(lds)) for name, blocks, lds in lines}

def spec(lens, source, shape, psf=None):
    params = {"sie": "x y r q pa", "epl_plus_shear": "x y r t q pa g1 g2", "gauss": "x y sigma mag q pa",
              "sersic": "x y r mag n q pa"}
    pri = {f"{o}.{p}": "unif 0.5 1" for o, n in (("lens", lens), ("source", source)) for p in params[n].split()}
    return SystemSpec([("lens", lens), ("source", source)], pri, np.zeros(shape, np.float32),
                      np.ones(shape, np.float32), psf=psf)

def noalloc(ctx, n):
    DP = ctypes.POINTER(ctypes.c_double)
    cubes, out = np.full((n, ctx.ndims()), 0.5), np.zeros(n)
    rc = L.load().lensed_loglike_batch_noalloc(ctypes.c_void_p(ctx.ptr), 0, cubes.ctypes.data_as(DP), n, None,
                                               out.ctypes.data_as(DP))
    return rc, launches()
""" % (ROOT, HERE)


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("stub")
    so = str(d / "hip_stub.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", "-o", so,
                           os.path.join(HERE, "hip_stub.cpp")])

    def call(code):
        preload = ":".join(p for p in (so, os.environ.get("LD_PRELOAD")) if p)
        env = dict(os.environ, LD_PRELOAD=preload, LENSED_CACHE_DIR=str(d))
        r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code)], env=env, capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0, (r.returncode, r.stderr[-3000:])
        return r.stdout
    return call


@pytest.mark.parametrize("lens", ["sie", "epl_plus_shear"])
def test_a_launch_without_candidates_is_an_error(run, lens):
    run(f"""
    with Context([spec({lens!r}, "gauss", (20, 30)), spec("sie", "sersic", (16, 16))], max_batch=4) as ctx:
        for counts in ([0, 0], [5, 0], [0, 1 << 62]):
            out = np.zeros(8)
            DP = ctypes.POINTER(ctypes.c_double)
            p = np.zeros(200)
            rc = L.load().lensed_loglike_systems(ctypes.c_void_p(ctx.ptr), (DP * 2)(*[p.ctypes.data_as(DP)] * 2),
                                                 (ctypes.c_size_t * 2)(*counts), (DP * 2)(*[out.ctypes.data_as(DP)] * 2))
            assert rc != 0 and ("no candidates" if not any(counts) else "max_batch") in L.last_error(), L.last_error()
        try:
            ctx.loglike_phys([np.zeros((0, ctx.npars(0))), np.zeros((0, ctx.npars(1)))])
            raise SystemExit("no error")
        except LensedError as e:
            assert "no candidates" in str(e)
        assert ctx.loglike_phys([np.zeros((0, ctx.npars(0))), np.full((2, ctx.npars(1)), 0.7)])[1].shape == (2,)
    """)


@pytest.mark.parametrize("lens,source,psf,flags", [("sie", "gauss", 21, 0), ("sie", "sersic", 5, 0),
                                                   ("epl_plus_shear", "gauss", 21, 4), ("epl_plus_shear", "gauss", 0, 4)])
def test_the_entry_that_allocates_nothing_launches_as_the_batch(run, lens, source, psf, flags):
    """For every count the same kernels and grids as lensed_loglike_batch,
    whatever the context's largest."""
    run(f"""
    from lensed_amd import workloads as W
    with Context(spec({lens!r}, {source!r}, (100, 120), W.gaussian_psf({psf}, 2.0) if {psf} else None), flags={flags},
                 max_batch=2000) as ctx:
        seen = set()
        for n in (2000, 1, 2, 16, 300, 2000, 7):
            launches()
            ctx.loglike_batch(np.full((n, ctx.ndims()), 0.5))
            batch = launches()
            rc, got = noalloc(ctx, n)
            assert rc == 0, L.last_error()
            assert got == batch, (n, got, batch)
            seen.add(tuple(got))
        assert len(seen) > 2, seen
    """)


@pytest.mark.parametrize("shape", [(48, 48), (40, 72), (64, 100)])
def test_scratch_holds_as_many_candidates_with_the_cull(run, shape):
    """Culled without a table: the cull's constants do not push a count out
    of the scratch that fits it without them."""
    run(f"""
    h, w = {shape}
    s = spec("sie", "gauss", (h, w))
    words, npar = sum(o.obj.size for o in s.objects), sum(o.obj.npars for o in s.objects)
    items = -(-h // 16) * -(-w // 16)
    up = lambda n: -(-n // 256) * 256
    def need(n):  # descriptor, parameters, blocks, two unused, model, partials, flags, list, record, owner
        parts = [512, n * npar * 4, (n * words + 256) * 4, 16, 16, n * h * w * 4, n * -(-h // 8) * -(-w // 64) * 8,
                 n * items * 16, 4 * (1 + 16 * n * items + 16 * n * -(-items // 64)), n * items * 16, 8]
        return sum(up(p) for p in parts)
    n = (128 << 20) // (need(1000) // 1000)
    while need(n) > 128 << 20:
        n -= 1
    with Context(s, max_batch=n + n // 8) as ctx:
        rc, got = noalloc(ctx, n)
        assert rc == 0, L.last_error()
        assert "lensed_cull" not in got, got
        rc, got = noalloc(ctx, n - n // 8)
        assert rc == 0 and "lensed_cull" in got, (L.last_error(), got)
        rc, got = noalloc(ctx, n + n // 8)
        assert rc != 0 and "static scratch" in L.last_error() and not got
    """)


@pytest.mark.parametrize("psf", [0, 7, 13, 31])
def test_tall_tiles_only_where_the_images_fill_them(run, psf):
    """64-row tiles for images whose rows they hold with little left over,
    whatever the number of candidates."""
    run(f"""
    from lensed_amd import workloads as W
    def kernel(h, n):
        with Context(spec("sie", "sersic", (h, 64), W.moffat_psf({psf}, 3.0, 2.5) if {psf} else None), max_batch=n) as ctx:
            launches()
            ctx.loglike_batch(np.full((n, ctx.ndims()), 0.5))
            return next(k for k in launches() if k.startswith("lensed_conv"))
    for h in (5, 20, 32, 65, 80, 96):
        tall = h > 32 and {psf} == 31  # (direct)
        assert kernel(h, 8192) == "lensed_conv_chi2" + ("_tall" if tall else ""), h
    for h in (33, 64, 97, 128, 200, 256):
        assert kernel(h, 4096) == "lensed_conv_chi2_tall", h
    assert kernel(160, 4096) == ("lensed_conv_chi2" if {psf} in (7, 13) else "lensed_conv_chi2_tall")
    assert kernel(64, 600) == ("lensed_conv_chi2_tall" if {psf} > 14 else "lensed_conv_chi2")
    assert kernel(64, 100) == "lensed_conv_chi2_small"
    """)


def test_cull_pass_only_where_it_can_skip_enough(run):
    """Without a table: by squares of 64 pixels per SIMD, and not for images of
    a few 16 x 16 blocks."""
    run("""
    def culled(lens, shape, n):
        with Context(spec(lens, "gauss", shape), max_batch=n) as ctx:
            launches()
            ctx.loglike_batch(np.full((n, ctx.ndims()), 0.5))
            return "lensed_cull" in launches()
    assert not culled("epl_plus_shear", (128, 128), 16) and culled("epl_plus_shear", (128, 128), 17)
    assert not culled("sie", (128, 128), 11) and culled("sie", (128, 128), 12)
    assert not culled("epl_plus_shear", (32, 32), 4000) and culled("epl_plus_shear", (40, 40), 4000)
    assert not culled("sie", (16, 48), 4000) and culled("sie", (24, 24), 4000)
    """)
