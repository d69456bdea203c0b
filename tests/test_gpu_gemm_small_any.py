"""GPU parity of the small matmul path's other forms: K of any length, A at any
4-byte address, and the backward's transposed operands.

They put the vector form's values into the same registers, so the checks are
for equal bits: against the product with K padded by zeros to a multiple of
four, against the aligned copy, and against explicit transposes.  The padded
product itself is held to (K + 1) 2^-24 sum |a b|: at most one rounding per k
and per partial sum.
"""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu

# K around the groups of 16, the waves' 64 and the last wave; M, N around the
# 16 x 16 tiles, with one, two and four row blocks a workgroup
SHAPES = [(1, 1, 1), (16, 3, 16), (17, 15, 15), (33, 17, 31), (5, 63, 200), (64, 65, 10),
          (1, 127, 65), (100, 129, 37), (64, 783, 128), (250, 1023, 250), (500, 30, 200),
          (497, 66, 129), (1000, 2, 200), (400, 61, 500)]


def operands(m, k, n):
    g = rng(m + 3 * k + 7 * n)
    return [g.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (m, n))]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_any_k(hip, m, k, n):
    a, b, _ = operands(m, k, n)
    got = hip.matmul(hip.tensor(a), hip.tensor(b)).numpy()
    bound = (k + 1) * 2.0**-24 * (np.abs(a).astype(np.float64) @ np.abs(b)) + 1e-30
    assert np.all(np.abs(got - a.astype(np.float64) @ b) <= bound)
    pad = -k % 4
    ap, bp = np.pad(a, ((0, 0), (0, pad))), np.pad(b, ((0, pad), (0, 0)))
    assert np.array_equal(got, hip.matmul(hip.tensor(ap), hip.tensor(bp)).numpy())
    # what lies beyond a row's end must not reach the sums
    b[0, :] = np.inf
    a[:, 0] = 1.0
    assert np.all(np.isinf(hip.matmul(hip.tensor(a), hip.tensor(b)).numpy()))


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("m,k,n", [(33, 64, 31), (64, 783, 128), (500, 48, 200)])
def test_any_address(hip, off, m, k, n):
    a, b, _ = operands(m, k, n)
    whole = hip.tensor(np.concatenate([np.full(off, np.nan, np.float32), a.ravel()]))
    view = hip.wrap(whole.device_ptr + 4 * off, a.shape)
    want = hip.matmul(hip.tensor(a), hip.tensor(b)).numpy()
    assert np.array_equal(hip.matmul(view, hip.tensor(b)).numpy(), want)


@pytest.mark.parametrize("m,k,n", SHAPES + [(64, 784, 128), (30, 784, 128), (64, 201, 1000)])
def test_gradients_match_transposed_copies(hip, monkeypatch, m, k, n):
    a, b, dc = (hip.tensor(x) for x in operands(m, k, n))
    got = [t.numpy() for t in hip.matmul_backward(a, b, dc)]
    monkeypatch.setenv("CLOVE_GEMM_TRANSPOSED", "0")
    for x, y in zip(got, hip.matmul_backward(a, b, dc)):
        assert np.array_equal(x, y.numpy())
