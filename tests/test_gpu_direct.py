"""GPU parity of the direct-sum kernels, called through the C-ABI.

FP64 (methods 1, 2): bitwise equal to the oracle and to the reference's
golden outputs.  FP32 split (methods 16, 17): relative error against the
FP64 direct sum, median <= 1e-6 (the north-star bound at N = 2^17) and
max <= 1e-4 per particle.
"""
import numpy as np
import pytest

from grav_sim_amd import ic
from grav_sim_amd import lib as L
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rel_err(a, b):
    return np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)


def test_fp64_pairwise_golden_bitwise(golden):
    f = golden("f1_pairwise.npz")
    assert np.array_equal(L.acceleration(f["x"], f["m"], 1, eps=0.0), f["a_eps0"])
    assert np.array_equal(L.acceleration(f["x"], f["m"], 1, eps=1e-3), f["a_eps1e3"])


@pytest.mark.parametrize("n", [1, 2, 3, 63, 255, 256, 257, 1000])
def test_fp64_pairwise_oracle_bitwise_ragged(n):
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, 3)) * 3.0
    m = rng.uniform(0.1, 2.0, n)
    for eps in (0.0, 0.01):
        got = L.acceleration(x, m, 1, G=0.7, eps=eps)
        assert np.array_equal(got, O.pairwise(x, m, G=0.7, eps=eps)), (n, eps)


def test_fp64_massless_golden_and_oracle(golden):
    f = golden("f2_massless.npz")
    assert np.array_equal(L.acceleration(f["x"], f["m"], 2, eps=0.0), f["a_eps0"])
    assert np.array_equal(L.acceleration(f["x"], f["m"], 2, eps=1e-2), f["a_eps1e2"])
    # massive particles not first: physics-correct masses (oracle), interleaved
    rng = np.random.default_rng(4)
    x = rng.normal(size=(300, 3))
    m = np.where(rng.uniform(size=300) < 0.3, rng.uniform(0.5, 1.0, 300), 0.0)
    assert np.array_equal(L.acceleration(x, m, 2, eps=0.0), O.massless(x, m, eps=0.0))


def test_fp64_massless_coincident_massless_particles():
    # two massless particles at the same point: the massless method never pairs them
    x = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [1.0, 0.0, 0.0]])
    m = np.array([1.0, 0.0, 0.0])
    a = L.acceleration(x, m, 2)
    assert np.all(np.isfinite(a))
    assert np.array_equal(a, O.massless(x, m))


@pytest.mark.parametrize("n,eps", [(1000, 0.0), (1000, 1e-3), (4097, 1e-2)])
def test_fp32_split_vs_fp64_small(n, eps):
    x, v, m = ic.plummer(n, 7)
    a32 = L.acceleration(x, m, 16, eps=eps)
    a64 = O.pairwise(x, m, eps=eps)
    e = rel_err(a32, a64)
    assert np.median(e) <= 1e-6 and e.max() <= 1e-4, (np.median(e), e.max())


def test_fp32_split_plummer_2e17_error_bound():
    """north-star accuracy bound: N=2^17 Plummer, eps=1e-3, median <= 1e-6 vs the FP64 GPU oracle."""
    x, v, m = ic.plummer(1 << 17, 2)
    sim = L.Sim(x, v, m, 1.0)
    med, p99, mx = sim.accel_error(L.param(16, eps=1e-3), samples=8192)
    print(f"fp32 split N=2^17: median {med:.3e} p99 {p99:.3e} max {mx:.3e}")
    assert med <= 1e-6
    assert p99 <= 1e-5
    sim.close()


def test_fp32_massless_sources():
    off, X, V, M = ic.ensemble(2, 5, max_test=500)
    x, m = X[off[0]:off[1]], M[off[0]:off[1]]
    a32 = L.acceleration(x, m, 17, eps=0.0)
    a64 = O.massless(x, m, eps=0.0)
    e = rel_err(a32, a64)
    assert np.median(e) <= 1e-6 and e.max() <= 1e-4


def test_energy_matches_oracle(golden):
    f = golden("f5_leapfrog.npz")
    import ctypes as C
    from grav_sim_amd import _abi
    s = _abi.make_system(f["x"], f["v"], f["m"], 1.0)
    e = L.load().compute_energy(C.byref(s))
    assert abs(e - float(f["e0"])) <= 1e-12 * abs(float(f["e0"]))


@pytest.mark.parametrize("block,ipt", [(4, 1), (8, 1), (16, 1), (0, 1), (0, 2), (0, 4), (256, 1), (256, 2), (256, 4), (128, 2),
                                       (128, 4), (512, 1), (512, 2)])
@pytest.mark.parametrize("split", [0, 3, 5, 12])
def test_fp32_every_shape_vs_oracle(block, ipt, split):
    """Each kernel shape the autotuner may pick gives the same accuracy (ragged N)."""
    x, v, m = ic.plummer(3001, 13)
    saved = L.get_fp32_config()
    try:
        L.set_fp32_config(block, ipt, split)
        a32 = L.acceleration(x, m, 16, eps=1e-3)
    finally:
        L.set_fp32_config(*saved)
    a64 = O.pairwise(x, m, eps=1e-3)
    e = rel_err(a32, a64)
    assert np.median(e) <= 1e-6 and e.max() <= 1e-4, (np.median(e), e.max())


def test_autotuner_picks_a_valid_shape_that_meets_the_error_bound():
    """gs_autotune_fp32 times every candidate shape and keeps the fastest; the
    shape it keeps is one of the parity-tested ones and later evaluations with
    it meet the FP32 bound against the oracle."""
    saved = L.get_fp32_config()
    try:
        block, ipt, split = L.autotune_fp32(1 << 14)
        assert (block, ipt) in {(4, 1), (8, 1), (16, 1), (0, 1), (0, 2), (0, 4), (256, 1), (256, 2), (256, 4),
                                (128, 2), (128, 4), (512, 1), (512, 2)}
        assert split in (0, 4, 8, 16, 32, 64)
        assert L.get_fp32_config() == (block, ipt, split)
        x, v, m = ic.plummer(3001, 17)
        a32 = L.acceleration(x, m, 16, eps=1e-3)
    finally:
        L.set_fp32_config(*saved)
    e = rel_err(a32, O.pairwise(x, m, eps=1e-3))
    assert np.median(e) <= 1e-6 and e.max() <= 1e-4, (block, ipt, split, np.median(e), e.max())


def test_issue_rate_probe_is_plausible():
    """The FP32 issue-rate probe behind the bench's instruction-mix ceiling: every
    form takes at least one cycle per wave64 instruction per SIMD, the FMA at
    least as long as the MUL, the transcendental v_rsq_f32 longer than the MUL."""
    r = L.issue_rates()
    print("issue rates (cycles per wave64 instruction):", r)
    assert 1.0 <= r["mul"] <= 1.1 * r["fma"] and r["rsq"] > r["mul"]


@pytest.mark.parametrize("n", [15, 16, 17, 64, 65, 1000, 2047, 5000, 11585, 16384, 23200])
def test_fp32_source_units_vs_fp64(n):
    """The automatic division of the sources (16-source units for the fewest targets, whole tiles from about 11 600
    particles, 1, 2 or 4 tiles per wavefront) against the FP64 sum, with the file's error bounds."""
    x, v, m = ic.plummer(n, 19)
    ref = L.acceleration(x, m, 1, G=1.3, eps=1e-2)  # (bitwise the oracle's)
    a32 = L.acceleration(x, m, 16, G=1.3, eps=1e-2)
    e = rel_err(a32, ref)
    assert np.median(e) <= 1e-6 and e.max() <= 1e-4, (np.median(e), e.max())


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 191, 192, 193, 1000, 3001])
def test_energy_blocks_vs_oracle(n):
    """Odd and even numbers of 64-particle blocks, ragged last blocks, a massless particle and particles at a distance
    whose square is outside the fast reciprocal root's range."""
    rng = np.random.default_rng(n)
    x, v, m = rng.normal(size=(n, 3)), rng.normal(size=(n, 3)), rng.uniform(0.1, 1.0, n)
    m[n // 2] = 0.0 if n > 2 else m[n // 2]
    for scale in (1.0, 1e-70):
        sim = L.Sim(x * scale, v, m, 0.7)
        e, ref = sim.energy(), O.energy(x * scale, v, m, 0.7)
        sim.close()
        # each term rounds to a few 2^-53; |sum of terms| / |energy| is bounded here by 1e2
        assert abs(e - ref) <= 1e-13 * abs(ref)
