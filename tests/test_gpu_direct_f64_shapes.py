"""The FP64 direct sum's kernel shapes and its in-range square root / division,
bit for bit against the oracle: around the target counts where the shape
changes (1024, 2048, 4096; the wide form from 3/5 of a round of 16384, whole
rounds with a remainder in the narrow form), operands outside the range the
fast sequence takes, and coincident particles."""
import numpy as np
import pytest

from grav_sim_amd import _abi, ic
from grav_sim_amd import lib as L
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1024, 1025, 2048, 2049, 4096, 4097, 9830, 9831, 16384, 16700])
def test_shapes_bitwise(n):
    x, v, m = ic.plummer(n, n)
    m[n // 3::3] = 0.0
    for method, ref in ((1, O.pairwise), (2, O.massless)):
        assert np.array_equal(L.acceleration(x, m, method, G=0.9, eps=1e-3), ref(x, m, G=0.9, eps=1e-3)), method


@pytest.mark.parametrize("n", [130, 9900])
@pytest.mark.parametrize("scale,G", [(1e-70, 1.0), (1e-55, 1e-30), (1e60, 1.0), (1.0, 1e-120), (1.0, 0.0), (1.0, -2.0)])
def test_operands_outside_the_fast_range(n, scale, G):
    x, v, m = ic.plummer(n, 5)
    x = x * scale
    assert np.array_equal(L.acceleration(x, m, 1, G=G, eps=0.0), O.pairwise(x, m, G=G, eps=0.0))


@pytest.mark.parametrize("n", [66, 9900])
def test_coincident_and_non_finite_positions(n):
    x, v, m = ic.plummer(n, 6)
    x[n // 2] = x[3]
    assert np.array_equal(L.acceleration(x, m, 1, eps=0.0), O.pairwise(x, m, eps=0.0), equal_nan=True)
    x[7, 1] = np.inf
    assert np.array_equal(L.acceleration(x, m, 1, eps=0.0), O.pairwise(x, m, eps=0.0), equal_nan=True)


@pytest.mark.parametrize("n,method", [(1030, 1), (10000, 1), (10000, 2), (17000, 1)])
def test_leapfrog_step_shapes_bitwise(n, method):
    x, v, m = ic.plummer(n, 9)
    m[n // 2:] = 0.0 if method == 2 else m[0]
    dt = 2.0 ** -9
    ids, xg, vg, mg, steps = L.launch_simulation(x, v, m, 1.0, _abi.INTEGRATOR_LEAPFROG, dt, 6 * dt, method=method,
                                                 eps=1e-2)
    xo, vo, so = O.leapfrog(x, v, m, 1.0, dt, 6 * dt, eps=1e-2, method=method)
    assert steps == so == 6
    assert np.array_equal(xg, xo) and np.array_equal(vg, vo)
