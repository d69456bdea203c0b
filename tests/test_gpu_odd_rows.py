"""GPU parity of the row kernels at widths and addresses that are not whole
16-byte vectors: every tail length (width % 4) at the edges of each kernel
family (a wave per row up to 1027 columns, a workgroup per row up to 53248,
rows re-read past that), and tensors that start 4, 8 or 12 bytes off a
16-byte boundary.

Tolerances are those of test_gpu_rowwise.py and test_gpu_backward.py: 1e-4
relative for the rows (sums in another order than the oracle's sequential
one), 1e-9 / 1e-5 absolute for softmax / layer norm.
"""
import numpy as np
import pytest

import oracle
from conftest import assert_close, rng

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 3, 5, 255, 257, 1023, 1025, 1027, 1029, 2047, 2051, 8193, 8197, 32769, 50257,
         53249, 53251, 60001]


def check_rows(hip, view, x, t, gam, bet):
    rows, cols = x.shape
    what = f"{rows}x{cols}"
    tx, tg, tb, tt = view(x), view(gam), view(bet), hip.tensor(t)
    want = oracle.softmax(x)
    assert_close(hip.softmax(tx).numpy(), want, 1e-4, 1e-9, f"softmax {what}")
    assert_close(hip.layer_norm(tx, tg, tb).numpy(), oracle.layer_norm(x, gam, bet), 1e-4, 1e-5,
                 f"layer norm {what}")
    loss = hip.cross_entropy(tx, tt).numpy()[0, 0]
    wl = oracle.cross_entropy(x, t)[0, 0]
    assert abs(loss - wl) <= 1e-4 * abs(wl) + 1e-7, (what, loss, wl)
    grad = hip.cross_entropy_backward(tx, tt, hip.tensor(np.array([1.5], np.float32))).numpy()
    assert_close(grad, oracle.cross_entropy_backward(x, t, 1.5), 1e-4, 1.5e-6 / rows,
                 f"cross entropy backward {what}")
    # both sides take the oracle's y: its sequential row sum is off by up to
    # cols * 2^-24 relative (2e-3 at 32769 columns), which dx would show
    # where its two terms cancel.  The sum of dy y runs in another order on
    # the GPU, again up to cols * 2^-24 of its terms.
    dx = hip.softmax_backward(view(want), tx).numpy()
    wd = oracle.softmax_backward(want, x)
    slack = want * max(1e-5, cols * 2.0**-24) * np.sum(np.abs(x * want), axis=1, keepdims=True)
    assert np.all(np.abs(dx - wd) <= 1e-4 * np.abs(wd) + slack + 1e-12), f"softmax backward {what}"


@pytest.mark.parametrize("cols", EDGES)
def test_odd_widths(hip, cols):
    g = rng(cols)
    rows = 5
    x = g.normal(0, 2, (rows, cols)).astype(np.float32)
    # targets in the first and last columns and around the last whole vector
    t = np.array([0, cols - 1, max(0, cols - 3), max(0, 4 * (cols // 4) - 1), cols // 2],
                 np.float32)
    gam = g.uniform(0.5, 1.5, cols).astype(np.float32)
    bet = g.uniform(-0.1, 0.1, cols).astype(np.float32)
    check_rows(hip, hip.tensor, x, t, gam, bet)


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("cols", [64, 1000, 4096, 8200, 50256])
def test_offset_tensors(hip, cols, off):
    """Widths of whole vectors whose tensors start `off` floats past a
    16-byte boundary (borrowed views of larger buffers)."""
    g = rng(cols + off)
    rows = 3
    x = g.normal(0, 2, (rows, cols)).astype(np.float32)
    t = np.array([cols - 1, 0, cols // 3], np.float32)
    gam = g.uniform(0.5, 1.5, cols).astype(np.float32)
    bet = g.uniform(-0.1, 0.1, cols).astype(np.float32)
    keep = []

    def view(a):
        buf = hip.tensor(np.concatenate([np.full(off, np.nan, np.float32), a.ravel()]))
        keep.append(buf)
        return hip.wrap(buf.device_ptr + 4 * off, a.shape)

    check_rows(hip, view, x, t, gam, bet)


@pytest.mark.parametrize("cols", [67, 1001, 4099, 50257, 53251])
def test_odd_special_values(hip, cols):
    """Masked (-inf, the lowest f32) and huge entries, and the rows whose
    result is NaN in the reference (all -inf, a +inf, a NaN), the special
    entries in the first vector, the middle and the tail."""
    g = rng(cols)
    x = g.normal(0, 2, (9, cols)).astype(np.float32)
    x[0, ::3] = 1000.0
    x[1, :] = -1000.0
    x[1, cols - 1] = -999.0
    x[2, 1::2] = -np.inf
    x[3, ::2] = np.finfo(np.float32).min
    x[4, :] = np.finfo(np.float32).min
    x[5, :] = -np.inf
    x[6, cols - 1] = np.inf
    x[7, 0] = np.nan
    x[8, cols - 2] = np.nan
    got, want = hip.softmax(hip.tensor(x)).numpy(), oracle.softmax(x)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert_close(got[ok], want[ok], 1e-4, 1e-9, f"softmax special rows x{cols}")
    assert np.all(got[2, 1::2] == 0.0) and np.all(got[3, ::2] == 0.0)


# The close softmax: odd widths of every kernel family, and every width past
# 32768 columns (aligned ones in registers up to 53248, re-read past that).
@pytest.mark.parametrize("cols", [67, 1001, 4099, 32769, 32772, 40000, 50257, 50304, 53248, 53252])
def test_close_softmax_against_float64(hip, cols):
    """Each entry against its row's largest, which the row sum's own rounding
    leaves alone: y = y_max exp(x - x_max), x - x_max rounded to f32 as every
    form does.  close_exp is within 1.5 ulp and the two quotients within half
    of one each: 2.5 ulp of at most 2^-23."""
    g = rng(cols)
    x = g.normal(0, 4, (4, cols)).astype(np.float32)
    y = hip.softmax(hip.tensor(x)).numpy().astype(np.float64)
    top = np.arange(4), x.argmax(1)
    d = (x - x[top][:, None]).astype(np.float64)
    want = y[top][:, None] * np.exp(d)
    assert np.max(np.abs(y - want) / want) <= 2.5 * 2.0**-23
    assert np.all(np.abs(y.sum(1) - 1) <= 2.0**-24 * (cols / 512 + 16))


@pytest.mark.parametrize("cols", [7, 67, 1001, 4099, 32772, 50257, 60001])
def test_close_softmax_subnormal_entries(hip, cols):
    """Entries between 2^-149 and 2^-126 of the largest are subnormal, not 0;
    the exponential, the quotient and the largest entry round once each, by at
    most half of 2^-149 here."""
    g = rng(cols)
    x = g.uniform(-105, -80, (3, cols)).astype(np.float32)
    x[:, cols // 3] = 0.0
    x[1, cols - 1] = 1.0
    y = hip.softmax(hip.tensor(x)).numpy().astype(np.float64)
    top = np.arange(3), x.argmax(1)
    want = y[top][:, None] * np.exp((x - x[top][:, None]).astype(np.float64))
    assert np.any((want > 0) & (want < 2.0**-127))
    assert np.all(np.abs(y - want) <= 2.5 * 2.0**-23 * want + 1.5 * 2.0**-149)


# One element a lane up to 64 columns (aligned widths from an odd address too), two
# up to 128 in the softmax backward;
# the loss's wave kernel up to 1152 columns.
@pytest.mark.parametrize("cols", [4, 31, 33, 60, 63, 64, 65, 68, 127, 128, 129, 1029, 1031, 1151, 1152, 1153])
@pytest.mark.parametrize("off", [0, 1])
def test_narrow_and_loss_edges(hip, cols, off):
    g = rng(cols + off)
    rows = 6
    x = g.normal(0, 2, (rows, cols)).astype(np.float32)
    t = np.array([cols - 1, 0, cols // 3, 4 * (cols // 4) - 1, cols // 2, max(0, cols - 2)],
                 np.float32)
    gam = g.uniform(0.5, 1.5, cols).astype(np.float32)
    bet = g.uniform(-0.1, 0.1, cols).astype(np.float32)
    keep = []

    def view(a):
        buf = hip.tensor(np.concatenate([np.full(off, np.nan, np.float32), a.ravel()]))
        keep.append(buf)
        return hip.wrap(buf.device_ptr + 4 * off, a.shape)

    check_rows(hip, view, x, t, gam, bet)


def best_ms(hip, call, reps=30):
    call()
    times = []
    for _ in range(4):
        e0 = hip.event_record()
        for _ in range(reps):
            call()
        times.append(hip.event_elapsed(e0, hip.event_record()))
        hip.event_reset()
    return min(times)


@pytest.mark.parametrize("op,rows,near,cols", [("softmax_backward", 1000000, 8, 7),
                                               ("softmax_backward", 300000, 68, 65),
                                               ("cross_entropy", 60000, 1027, 1029)])
def test_no_step_at_odd_widths(hip, op, rows, near, cols):
    """Narrow odd rows take about as long as the aligned width beside them, and
    the loss no longer past the wave kernel's width than at it (they took 1.4
    and 2.7 times as long)."""
    ms = {}
    for c in (near, cols):
        x = hip.empty((rows, c)).fill_normal(1)
        t = hip.tensor(np.arange(rows, dtype=np.float32) % c)
        call = {"softmax_backward": lambda: hip.softmax_backward(x, x),
                "cross_entropy": lambda: hip.cross_entropy(x, t)}[op]
        ms[c] = best_ms(hip, call)
    assert ms[cols] <= 1.25 * ms[near], ms
