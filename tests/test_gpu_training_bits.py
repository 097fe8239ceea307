"""Training the learned correction on a given sample gives the same weights, bit for bit, however the force kernels
divide their work.

Training turns a change in the last bits of its labels or walk sums into 1e-4 of the weights, so gs_learned_train takes
both in one fixed order.  The expected values (golden f12_training.npz) are this library's own at commit 909feb2; the
particles come from uniform draws and products alone, so that they are the same doubles on any host."""
import hashlib

import numpy as np
import pytest

from grav_sim_amd import lib as L

pytestmark = pytest.mark.gpu

# the sizes of two forms of the per-particle walk and of two divisions of the direct sums
CASES = [dict(n=4096, samples=4096, epochs=2, batch=512, theta=0.8, leaf=1),
         dict(n=20000, samples=5000, epochs=1, batch=512, theta=0.5, leaf=8)]


def particles(n):
    x = np.random.default_rng(n).random((n, 3))
    x = x * x * x
    x[n // 2:, 0] += 2.0
    return x, np.full(n, 1.0 / n)


def train(case):
    x, m = particles(case["n"])
    loss = L.learned_train(x, m, eps=1e-3, theta=case["theta"], leaf=case["leaf"], samples=case["samples"],
                           epochs=case["epochs"], batch=case["batch"], lr=1e-3, seed=5)
    w, mean, std, scale = L.learned_get_params()
    return {"weights": w[::16], "mean": mean, "std": std, "loss": np.array([loss, scale]),
            "sha256": np.frombuffer(hashlib.sha256(np.ascontiguousarray(w, np.float32).tobytes()).digest(), np.uint8)}


@pytest.mark.parametrize("k", range(len(CASES)))
def test_training_keeps_its_bits(golden, k):
    f = golden("f12_training.npz")
    for name, v in train(CASES[k]).items():
        assert np.array_equal(v, f[f"{name}{k}"]), name
