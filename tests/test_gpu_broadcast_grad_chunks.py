"""GPU parity of the broadcast gradient around its chunk lengths: one chunk
(written straight to the result), exactly one, and one element more.

A column's n / nb values are added in some order, so the result is within
(n / nb + 1) 2^-24 of the sum of their magnitudes.
"""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("negate", [False, True])
@pytest.mark.parametrize("nb", [1, 10, 63, 64, 65, 128, 130, 1000])
def test_chunks(hip, nb, negate):
    chunk = 64 * nb if nb >= 64 else 64 * nb * (256 // nb)
    for n in (1, nb, nb + 1, 7 * nb - 1, chunk - 1, chunk, chunk + 1, 3 * chunk + 5):
        g = rng(n + nb).standard_normal(n, dtype=np.float32)
        pad = np.zeros(-(-n // nb) * nb)
        pad[:n] = g
        cols = pad.reshape(-1, nb)
        got = hip.broadcast_grad(hip.tensor(g), nb, negate).numpy().ravel()
        want = cols.sum(axis=0) * (-1 if negate else 1)
        bound = (len(cols) + 1) * 2.0**-24 * np.abs(cols).sum(axis=0)
        assert np.all(np.abs(got - want) <= bound), (n, nb)
