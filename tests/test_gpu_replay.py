"""Captured launches replayed with other parameters each time, against a
context that captures nothing: the kernels of a graph read the parameters of
the call, whether they are copied or (up to 4 KiB) lie in pinned host memory."""
import numpy as np
import pytest

from lensed_amd._lib import LENSED_GRAPH, LENSED_TABLE
from lensed_amd.lensed import Context
from test_gpu_small_launches import make_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,source,flags", [("sie", "sersic", 0), ("epl_plus_shear", "gauss", LENSED_TABLE),
                                               ("epl_plus_shear", "gauss", 0)])
def test_replays_take_the_call_s_parameters(lens, source, flags):
    spec = make_spec(lens, source, (70, 90), 7, "g3k7", 21)
    rng = np.random.default_rng(22)
    with Context(spec, max_batch=200, flags=flags) as eager, Context(spec, max_batch=200, flags=flags | LENSED_GRAPH) as ctx:
        for n in (2, 64, 73, 74, 200) * 2:  # (14 parameters: 4 KiB end at 73 candidates)
            for _ in range(4):
                cubes = rng.random((n, ctx.ndims()))
                got, phys = ctx.loglike_batch(cubes)
                want, same = eager.loglike_batch(cubes)
                assert np.array_equal(phys, same)
                assert np.all(np.isfinite(got)) and np.array_equal(got, want), n
                assert np.unique(got).size == n
