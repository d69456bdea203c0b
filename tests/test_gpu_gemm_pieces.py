"""GPU parity of the matmul on the bf16 matrix cores (three bf16 pieces per
f32 value), against float64.

Every rounding of the kernel is one of f32 on a partial sum: at most four per
MFMA step of 16 k and product, six products, so 1.5 per k; and the products it
leaves out are at most 2^-24 |a b| (two pieces of 2^-8 and 2^-17 each way; the
data that reaches it is in test_same_sign_and_constant_operands).  The bound per
element is therefore (1.5 K + 1) 2^-24 sum |a b|, or half a subnormal step
(2^-150) per rounding where sums are subnormal; over a whole random matrix the
roundings add as a random walk, and the 2-norm error stays below 2.5e-8 sqrt(K)
(the FP32 MFMA kernel measures 1.8e-8 sqrt(K), this one 1.6e-8).
"""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu

TILES = ["7", "8", "9"]  # 256x128, 128x128, 128x128 with eight waves


def check64(got, a, b, what):
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    k = a.shape[1]
    want = a64 @ b64
    bound = (1.5 * k + 1) * 2.0**-24 * (np.abs(a64) @ np.abs(b64)) + 1.5 * k * 2.0**-150
    assert np.all(np.abs(got - want) <= bound), what
    return want


@pytest.mark.parametrize("cfg", TILES)
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (65, 16, 128), (128, 32, 128), (129, 33, 127),
                                   (256, 15, 129), (257, 47, 255), (300, 1030, 514),
                                   (255, 4099, 131), (512, 512, 384), (1000, 777, 1001)])
def test_tile_edges(hip, monkeypatch, cfg, m, k, n):
    """Tiles, slabs and splits that the shape ends inside, rows at any 4-byte
    alignment; a repeated call gives the same bits, and the fused bias + GELU
    the bits of the separate calls."""
    monkeypatch.setenv("CLOVE_GEMM_CFG", cfg)
    g = rng(m + 3 * k + 7 * n)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    ta, tb = hip.tensor(a), hip.tensor(b)
    got = hip.matmul(ta, tb)
    want = check64(got.numpy(), a, b, f"{cfg}: {m}x{k}x{n}")
    if m * n > 10000:
        err = np.linalg.norm(got.numpy() - want) / np.linalg.norm(want)
        assert err <= 2.5e-8 * np.sqrt(k) + 1e-7, err
    assert np.array_equal(hip.matmul(ta, tb).numpy(), got.numpy())
    bias = hip.tensor(g.standard_normal(n, dtype=np.float32))
    gr = hip.Graph()
    x, w, bi = gr.input((m, k)), gr.input((k, n)), gr.input((n,))
    model = gr.compile([gr.op("gelu", gr.op("add", gr.op("matmul", x, w), bi))])
    (fused,) = model.execute([ta, tb, bias])
    assert np.array_equal(fused.numpy(), hip.gelu(hip.add(got, bias)).numpy())


@pytest.mark.parametrize("m,k,n", [(1000, 700, 700), (2050, 1028, 3000), (777, 1001, 1003),
                                   (4096, 128, 1000)])
def test_planned_forward_and_gradients(hip, monkeypatch, m, k, n):
    """Shapes the plan sends to the bf16 matrix cores in all three products
    (plain, B transposed, A transposed), aligned or not; the gradients match
    explicit transposes bit for bit."""
    g = rng(m + k + n)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    dc = g.standard_normal((m, n), dtype=np.float32)
    ta, tb, tc = hip.tensor(a), hip.tensor(b), hip.tensor(dc)
    check64(hip.matmul(ta, tb).numpy(), a, b, "forward")
    da, db = (t.numpy() for t in hip.matmul_backward(ta, tb, tc))
    check64(da, dc, b.T, "grad a")
    check64(db, a.T, dc, "grad b")
    monkeypatch.setenv("CLOVE_GEMM_TRANSPOSED", "0")
    da0, db0 = (t.numpy() for t in hip.matmul_backward(ta, tb, tc))
    assert np.array_equal(da, da0) and np.array_equal(db, db0)


@pytest.mark.parametrize("off", [1, 2, 3])
def test_offset_operands(hip, off):
    """A and B that start `off` floats past a 16-byte boundary."""
    g = rng(off)
    a = g.standard_normal((900, 800), dtype=np.float32)
    b = g.standard_normal((800, 700), dtype=np.float32)
    bufs = [hip.tensor(np.concatenate([np.full(off, np.nan, np.float32), x.ravel()]))
            for x in (a, b)]
    ta, tb = (hip.wrap(t.device_ptr + 4 * off, x.shape) for t, x in zip(bufs, (a, b)))
    check64(hip.matmul(ta, tb).numpy(), a, b, f"offset {off}")


@pytest.mark.parametrize("cfg", TILES)
def test_pieces_hold_every_bit(hip, monkeypatch, cfg):
    """Products with the identity, a permutation and powers of two are exact:
    no bit of an operand is dropped."""
    monkeypatch.setenv("CLOVE_GEMM_CFG", cfg)
    g = rng(5)
    a = g.standard_normal((300, 256), dtype=np.float32)
    a[:, ::3] *= np.exp2(g.integers(-60, 60, (300, 1))).astype(np.float32)
    eye = np.eye(256, dtype=np.float32)
    assert np.array_equal(hip.matmul(hip.tensor(a), hip.tensor(eye)).numpy(), a)
    p = eye[g.permutation(256)] * np.exp2(g.integers(-20, 20, 256)).astype(np.float32)
    assert np.array_equal(hip.matmul(hip.tensor(a), hip.tensor(p)).numpy(), a @ p)


@pytest.mark.parametrize("cfg", TILES)
@pytest.mark.parametrize("sa,sb", [(1e-36, 1e30), (1e-33, 1e25), (1e-40, 1e36), (1e-25, 1e-20),
                                   (1e30, 1e-35), (1e18, 1e18)])
def test_far_scales(hip, monkeypatch, cfg, sa, sb):
    """Operands near the ends of f32's range: small ones in pieces of 2^24 x, and
    past 2^103, or for sums past 2^79, on the FP32 MFMA instead."""
    monkeypatch.setenv("CLOVE_GEMM_CFG", cfg)
    g = rng(9)
    a = (g.standard_normal((200, 96)) * sa).astype(np.float32)
    b = (g.standard_normal((96, 140)) * sb).astype(np.float32)
    check64(hip.matmul(hip.tensor(a), hip.tensor(b)).numpy(), a, b, f"{sa} x {sb}")


@pytest.mark.parametrize("cfg", TILES)
def test_special_values(hip, monkeypatch, cfg):
    """Infinities, NaN, the lowest f32 and single tiny entries: the results
    of f32 arithmetic, elsewhere as if they were not there."""
    monkeypatch.setenv("CLOVE_GEMM_CFG", cfg)
    g = rng(10)
    a = g.standard_normal((300, 64), dtype=np.float32)
    b = np.abs(g.standard_normal((64, 200), dtype=np.float32)) + 0.5
    a[3, 5] = np.inf
    a[7, 63] = -np.inf
    a[131, 0] = np.nan
    a[140, 2] = np.finfo(np.float32).min
    b[2, 150] = 0.0
    a[260, 9] = 1e-38
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
        want32 = want.astype(np.float32)
    got = hip.matmul(hip.tensor(a), hip.tensor(b)).numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want32))
    inf = np.isinf(want32)
    assert np.array_equal(got[inf], want32[inf])
    rest = np.isfinite(want32)
    scale = np.abs(np.nan_to_num(a.astype(np.float64), posinf=0, neginf=0)) @ np.abs(b)
    assert np.all(np.abs(got[rest] - want[rest]) <= (97 * 2.0**-24 * scale)[rest])


def test_plan_takes_special_values(hip):
    """The same through the default plan and the split-K reduce."""
    g = rng(11)
    a = g.standard_normal((700, 1500), dtype=np.float32)
    b = g.standard_normal((1500, 700), dtype=np.float32)
    a[650, 1400] = np.inf
    b[0, 0] = np.nan
    a[0, 700] = 1e-39
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    got = hip.matmul(hip.tensor(a), hip.tensor(b)).numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf].astype(np.float32))
    ok = np.isfinite(want)
    assert np.max(np.abs(got[ok] - want[ok])) < 1e-3


@pytest.mark.parametrize("cfg", TILES)
def test_small_operands_keep_every_bit(hip, monkeypatch, cfg):
    """The same down to f32's smallest: every bit of values from 2^-149 on,
    beside ordinary ones, and products of two small operands."""
    monkeypatch.setenv("CLOVE_GEMM_CFG", cfg)
    g = rng(12)
    a = g.standard_normal((300, 256)).astype(np.float32)
    a[:, 1::2] *= np.exp2(g.integers(-149, -100, (300, 128))).astype(np.float32)
    eye = np.eye(256, dtype=np.float32)
    assert np.array_equal(hip.matmul(hip.tensor(a), hip.tensor(eye)).numpy(), a)
    b = (eye[g.permutation(256)] * np.exp2(g.integers(-80, 20, 256))).astype(np.float32)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)  # rounded once
    assert np.array_equal(hip.matmul(hip.tensor(a), hip.tensor(b)).numpy(), want)


@pytest.mark.parametrize("k", [64, 1024, 4096, 16384])
def test_same_sign_and_constant_operands(hip, monkeypatch, k):
    """Data whose roundings do not cancel: values in [0, 1), held to the error of
    the FP32 MFMA tiles, and constants, whose every partial sum rounds alike: the
    one that makes the most of the products left out, and 12 others, whose
    root mean square is held to those tiles' as well."""
    g = rng(k)

    def error(a, b, cfg=None):
        if cfg:
            monkeypatch.setenv("CLOVE_GEMM_CFG", cfg)
        got = hip.matmul(hip.tensor(a), hip.tensor(b)).numpy()[:64].astype(np.float64)
        monkeypatch.delenv("CLOVE_GEMM_CFG", raising=False)
        want = a[:64].astype(np.float64) @ b.astype(np.float64)
        return np.linalg.norm(got - want) / np.linalg.norm(want)

    a, b = g.random((512, k), dtype=np.float32), g.random((k, 512), dtype=np.float32)
    assert error(a, b, "8") <= 1.1 * error(a, b, "2")
    worst = np.float32(1 + 2.0**-8 - 2.0**-17)
    # 2^-24 left out, and the roundings of sums that are half the whole on average
    chain = min(k, 1024) / 16 * 6  # 16 splits, 6 products a step of 16 k
    assert error(np.full((512, k), worst), np.full((k, 512), worst), "8") <= 2.0**-24 * (2 + chain / 2)
    pieces, fp32 = [], []
    for _ in range(12):
        x, y = (np.float32(1 + g.random()) for _ in range(2))
        a, b = np.full((512, k), x), np.full((k, 512), y)
        pieces.append(error(a, b, "8"))
        fp32.append(error(a, b, "2"))
    # (the splits differ, so the bound leaves room for a chain twice as long)
    assert np.linalg.norm(pieces) <= 2 * np.linalg.norm(fp32) + 1e-7, (pieces, fp32)


def test_outer_product_rounds_once(hip):
    """K = 1 at a size past 0.7 GFLOP: each output is its product, rounded."""
    n = 18900
    a, b = hip.empty((n, 1)).fill_normal(1), hip.empty((1, n)).fill_normal(2)
    got = hip.matmul(a, b)
    ah, bh = a.numpy(), b.numpy()
    for r in (0, 1, 127, 128, 9000, n - 1):
        assert np.array_equal(got.read(r * n, n), ah[r, 0] * bh[0]), r


def best_ms(hip, call, reps=10):
    call()
    times = []
    for _ in range(3):
        e0 = hip.event_record()
        for _ in range(reps):
            call()
        times.append(hip.event_elapsed(e0, hip.event_record()))
        hip.event_reset()
    return min(times)


# The smallest K and the fewest tiles that the plan takes, long K whose C cannot
# fill the chip, thin C whose K splits would park mostly padding.
@pytest.mark.parametrize("m,k,n", [(4096, 24, 4096), (8192, 16, 4096), (512, 192, 4096),
                                   (3000, 200, 700), (128, 32768, 128), (256, 16384, 256),
                                   (1000, 16384, 64), (40000, 256, 64)])
def test_planned_edges(hip, m, k, n):
    """Against float64, to the FP32 MFMA kernel's error: 2.3e-8 sqrt(chain) for
    the K range that one accumulator sums."""
    g = rng(m + k + n)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    got = hip.matmul(hip.tensor(a), hip.tensor(b)).numpy()
    rows = np.r_[0:min(m, 300), max(0, m - 20):m]
    want = a[rows].astype(np.float64) @ b.astype(np.float64)
    err = np.linalg.norm(got[rows] - want) / np.linalg.norm(want)
    # (64 splits at most; their sum adds one rounding of each)
    assert err <= 2.3e-8 * np.sqrt(max(k / 64, min(k, 1280))) + 1e-7, err


def test_small_operands_cost_nothing(hip):
    """A tiny value per 256 rows, as softmax and loss gradients hold them, does
    not send its tiles to a second computation (which took 2.6 times as long)."""
    n = 4096
    a, b = hip.empty((n, n)).fill_normal(1), hip.empty((n, n)).fill_normal(2)
    plain = best_ms(hip, lambda: hip.matmul(a, b))
    for r in range(0, n, 256):
        a.write(r * n + 5, np.array([1e-33, 1e-40], np.float32))
    assert best_ms(hip, lambda: hip.matmul(a, b)) <= 1.3 * plain


# Shapes on both sides of 0.7 GFLOP, where the plan first weighs the bf16 pieces:
# (below, above, most that `above` may take of `below`'s time; the work grows by
# 1.6, 1.2 and 1.6, bound by C's write in the first and last).
@pytest.mark.parametrize("below,above,most", [((8192, 10, 4096), (8192, 16, 4096), 1.35),
                                              ((512, 160, 4096), (512, 192, 4096), 1.35),
                                              ((300000, 10, 100), (300000, 16, 100), 1.4)])
def test_no_step_where_the_pieces_begin(hip, below, above, most):
    """Thin K and few tiles took 1.7 to 2 times as long past the line."""
    ms = {}
    for m, k, n in (below, above):
        a, b = hip.empty((m, k)).fill_normal(1), hip.empty((k, n)).fill_normal(2)
        ms[m, k, n] = best_ms(hip, lambda: hip.matmul(a, b), 50)
    assert ms[above] <= most * ms[below], ms
