"""GPU parity of the attention prefill on the bf16 matrix cores, against
float64: head dims on and off its tile sizes, ragged blocks, keys split over
workgroups, and values its bf16 pieces cannot hold.

The bound: scores and output are f32 sums, so the relative 2-norm error over
random inputs stays within a few 1e-7 (measured 1e-7 to 6e-7; the FP32 MFMA
kernels measure 2.5e-7 to 6e-7); 2e-6 is asked.
"""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu


def attention64(q, k, v, heads, past, causal):
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    B, S, X = q.shape
    D, Sk = X // heads, k.shape[1]
    out = np.empty_like(q)
    hidden = np.arange(Sk)[None, :] > np.arange(S)[:, None] + past
    for b in range(B):
        for h in range(heads):
            c = slice(h * D, (h + 1) * D)
            s = q[b, :, c] @ k[b, :, c].T / np.sqrt(D)
            if causal:
                s[hidden] = -np.inf
            p = np.exp(s - s.max(1, keepdims=True))
            out[b, :, c] = p @ v[b, :, c] / p.sum(1, keepdims=True)
    return out


def inputs(seed, B, S, past, H, D):
    g = rng(seed)
    return [g.standard_normal((B, n, H * D), dtype=np.float32) for n in (S, S + past, S + past)]


def run(hip, q, k, v, H, past, causal):
    flags = hip.ATTN_CAUSAL if causal else 0
    return hip.flash_attention(hip.tensor(q), hip.tensor(k), hip.tensor(v), H, q_pos=past,
                               flags=flags).numpy()


def check(got, want, what):
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= 2e-6, (what, err)
    assert np.max(np.abs(got - want)) <= 2e-5 * np.abs(want).max(), what


# One query and key; blocks of 128 and 256 queries and of 32 keys that the
# lengths end inside, at and past; few queries over many keys (split), many
# queries (unsplit); every tile size with a head dim below it.
@pytest.mark.parametrize("D", [8, 32, 40, 64, 72, 96, 104, 128])
@pytest.mark.parametrize("B,S,past,H", [(1, 1, 0, 1), (1, 31, 33, 2), (2, 128, 0, 2),
                                        (1, 257, 63, 2), (3, 5, 1500, 1), (1, 600, 0, 3)])
@pytest.mark.parametrize("causal", [True, False])
def test_shapes(hip, D, B, S, past, H, causal):
    q, k, v = inputs(D + S + past, B, S, past, H, D)
    got = run(hip, q, k, v, H, past, causal)
    check(got, attention64(q, k, v, H, past, causal), f"D={D} {B}x{S}+{past}")
    assert np.array_equal(got, run(hip, q, k, v, H, past, causal))  # fixed order


@pytest.mark.parametrize("D", [64, 80, 96, 128])
@pytest.mark.parametrize("scale_q,scale_k,scale_v", [(1e-33, 1e33, 1), (1e33, 1e-33, 1),
                                                     (1, 1, 1e-36), (1, 1, 1e32)])
def test_far_scales(hip, D, scale_q, scale_k, scale_v):
    """Values near the ends of f32's range, as pieces or on the FP32 MFMA."""
    q, k, v = inputs(D, 1, 150, 40, 2, D)
    q, k, v = (x * np.float32(s) for x, s in zip((q, k, v), (scale_q, scale_k, scale_v)))
    check(run(hip, q, k, v, 2, 40, True), attention64(q, k, v, 2, 40, True), f"D={D}")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,past", [(300, 0), (40, 900)])
def test_special_values(hip, D, S, past):
    """NaN and infinite values reach the queries that see them, in one split or
    another, and no other query or dim; single tiny values change nothing else.
    (A masked key weighs 0, and 0 times an infinite v is NaN in an f32 sum: the
    infinity's own dim is only looked at where its key is visible.)"""
    q, k, v = inputs(D + S, 1, S, past, 1, D)
    q[0, 3, 1] = 1e-39
    k[0, 2, 5] = 1e-38
    k[0, past + 20, 0] = np.nan          # queries 20.. see it
    v[0, past + 30, 7] = np.inf          # queries 30.. see it, in dim 7
    keep = np.ones(D, bool)
    keep[7] = False
    got = run(hip, q, k, v, 1, past, True)[0]
    assert np.all(np.isnan(got[20:]))
    want = attention64(q, np.nan_to_num(k), np.nan_to_num(v, posinf=0.0), 1, past, True)[0]
    check(got[:20, keep], want[:20, keep], "rows before the NaN")
    k[0, past + 20, 0] = 0.0
    got = run(hip, q, k, v, 1, past, True)[0]
    assert np.all(np.isinf(got[30:, 7]))
    want = attention64(q, k, np.nan_to_num(v, posinf=0.0), 1, past, True)[0]
    check(got[:, keep], want[:, keep], "dims beside the infinity")


# Head dims of the smallest tile; and enough heads that no keys are split.
@pytest.mark.parametrize("D", [8, 24, 32])
@pytest.mark.parametrize("scale_q,scale_k,scale_v", [(1e-33, 1e33, 1), (1, 1, 1e-36), (1, 1, 1e32)])
def test_far_scales_small_tile(hip, D, scale_q, scale_k, scale_v):
    q, k, v = inputs(D, 1, 600, 40, 3, D)
    q, k, v = (x * np.float32(s) for x, s in zip((q, k, v), (scale_q, scale_k, scale_v)))
    check(run(hip, q, k, v, 3, 40, True), attention64(q, k, v, 3, 40, True), f"D={D}")


@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_unsplit_launches(hip, D, causal):
    B, S, H = 32, 600, 16
    q, k, v = inputs(D, B, S, 0, H, D)
    got = run(hip, q, k, v, H, 0, causal)
    for b, h in ((0, 0), (17, 3), (31, 15)):
        c = slice(h * D, (h + 1) * D)
        want = attention64(q[b:b + 1, :, c], k[b:b + 1, :, c], v[b:b + 1, :, c], 1, 0, causal)
        check(got[b:b + 1, :, c], want, f"D={D} b={b} h={h}")


def test_no_visible_key(hip):
    """Queries before every key get zeros, in split and unsplit launches."""
    for S, Sk in ((64, 64), (80, 80), (10, 3000)):
        g = rng(S)
        q = g.standard_normal((1, S, 256), dtype=np.float32)
        k, v = (g.standard_normal((1, Sk, 256), dtype=np.float32) for _ in range(2))
        got = hip.flash_attention(hip.tensor(q), hip.tensor(k), hip.tensor(v), 2, q_pos=0,
                                  k_pos=S - 4, flags=hip.ATTN_CAUSAL).numpy()
        assert np.all(got[0, :S - 4] == 0.0)
        assert np.array_equal(got[0, S - 4], v[0, 0])


# Up to 64 queries and keys run on the FP32 MFMA, one more of either may run on
# the bf16 pieces (as priced).
@pytest.mark.parametrize("D", [8, 64, 80, 104, 128])
@pytest.mark.parametrize("S,past", [(1, 63), (64, 0), (65, 0), (33, 31), (33, 32), (1, 64)])
def test_short_calls(hip, D, S, past):
    q, k, v = inputs(D + S, 2, S, past, 3, D)
    check(run(hip, q, k, v, 3, past, True), attention64(q, k, v, 3, past, True), f"D={D} {S}+{past}")


# Heads and keys whose k and v end just under 2 GiB, inside a block of 32 keys.
@pytest.mark.parametrize("H,D,Sk", [(7, 64, 1198372), (7, 96, 798915)])
def test_last_keys_near_2_gib(hip, H, D, Sk):
    """The last block's byte offsets stay inside 32 bits up to the largest k and
    v taken: a query that attends to the last Sk % 32 keys alone gets the mean
    of their values (equal scores, the others' weights e^-200)."""
    X, last = H * D, Sk % 32
    assert 2**31 - 32 * X * 4 < Sk * X * 4 < 2**31 < (Sk - last + 11) * X * 4
    k = hip.empty((1, Sk, X)).fill_uniform(0, 0.0, 0.0)
    k.write((Sk - last) * X, np.full(last * X, 200 / np.sqrt(D), np.float32))
    v = hip.empty((1, Sk, X)).fill_normal(7)
    q = hip.tensor(np.ones((1, 1, X), np.float32))
    got = hip.flash_attention(q, k, v, H, flags=0).numpy()[0, 0]
    want = v.read((Sk - last) * X, last * X).reshape(last, X).astype(np.float64).mean(0)
    assert np.max(np.abs(got - want)) <= 4 * 2.0**-24 * np.abs(want).max()
    del k, v
    hip.empty_cache()


@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("S,Sk", [(4, 200), (4, 3000), (300, 300)])
def test_small_weights_keep_their_bits(hip, D, S, Sk):
    """A weight of 2^-125.x of the largest on the one value that is not 0, and
    large enough to make up for it.  Its score's rounding, 126 ln 2 2^-24 of the
    weight, and that of the q . k sum bound the error: 2e-5."""
    g = rng(D + Sk)
    q = np.ones((1, S, D), np.float32)
    k = np.zeros((1, Sk, D), np.float32)
    v = np.zeros((1, Sk, D), np.float32)
    k[0, Sk // 2, 0] = -125.3 * np.log(2) * np.sqrt(D)
    v[0, Sk // 2] = g.uniform(0.5, 1, D) * 2.0**90
    got = hip.flash_attention(hip.tensor(q), hip.tensor(k), hip.tensor(v), 1, flags=0).numpy()
    want = attention64(q, k, v, 1, 0, False)
    assert np.max(np.abs(got - want) / want) <= 2e-5


def best_ms(hip, q, k, v, H, reps=10):
    times = []
    for _ in range(5):
        e0 = hip.event_record()
        for _ in range(reps):
            hip.flash_attention(q, k, v, H, flags=hip.ATTN_CAUSAL)
        times.append(hip.event_elapsed(e0, hip.event_record()))
        hip.event_reset()
    return min(times)


def test_small_operands_cost_nothing(hip):
    """Tiny values in k or v do not send their heads' queries to a second
    computation (which took 2.2 times as long)."""
    S, X = 4096, 2048
    q, k, v = (hip.empty((1, S, X)).fill_normal(i) for i in (1, 2, 3))
    plain = best_ms(hip, q, k, v, 16)
    for h in range(16):
        k.write(7 * X + 128 * h, np.array([1e-33, 1e-40], np.float32))
        v.write(9 * X + 128 * h, np.array([1e-33, 1e-40], np.float32))
    assert best_ms(hip, q, k, v, 16) <= 1.3 * plain


@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_small_values_keep_their_bits(hip, D):
    """v down to f32's smallest: a query that attends to one key alone (its
    score 200 above the others) gets that key's row, every bit of it."""
    g = rng(D)
    S = 300
    q, k = np.ones((1, S, D), np.float32), np.zeros((1, S, D), np.float32)
    k[0, 77] = 200 / np.sqrt(D)
    v = (g.standard_normal((1, S, D)) * np.exp2(g.integers(-149, -90, (1, S, D)))).astype(np.float32)
    got = hip.flash_attention(hip.tensor(q), hip.tensor(k), hip.tensor(v), 1, flags=0).numpy()
    assert np.array_equal(got[0], np.broadcast_to(v[0, 77], (S, D)))


@pytest.mark.parametrize("D,below,B,S", [(128, 124, 256, 8), (104, 100, 64, 100), (16, 12, 12, 128)])
def test_many_short_heads_take_the_faster_kernel(hip, D, below, B, S):
    """Calls of many short heads take no longer than those of a head dim just
    below, which always run on the FP32 MFMA (they took 1.2 to 1.7 times as
    long on the bf16 pieces), and give the same values as ever."""
    H, took = 32, {}
    for d in (below, D):
        q, k, v = (hip.empty((B, S, H * d)).fill_normal(i) for i in (1, 2, 3))
        took[d] = best_ms(hip, q, k, v, H, 50)
    assert took[D] <= 1.12 * took[below], took
    got = hip.flash_attention(q, k, v, H, flags=hip.ATTN_CAUSAL).read((B - 1) * S * H * D, S * H * D)
    last = [t.read((B - 1) * S * H * D, S * H * D).reshape(1, S, H * D) for t in (q, k, v)]
    check(got.reshape(1, S, H * D), attention64(*last, H, 0, True), f"D={D} {B}x{S}")


def test_more_heads_than_one_grid(hip):
    """Past 2^23 heads (of one query block each) a launch would hold 2^32
    threads: they go in several.  One key: every output row is its v."""
    B, H, D = (1 << 18) + 1, 32, 128
    q, k, v = (hip.empty((B, 1, H * D)).fill_normal(i) for i in (1, 2, 3))
    out = hip.flash_attention(q, k, v, H, flags=0)
    for b in (0, 1, (1 << 18) - 2, (1 << 18) - 1, 1 << 18):
        assert np.array_equal(out.read(b * H * D, H * D), v.read(b * H * D, H * D)), b
    del q, k, v, out
    hip.empty_cache()


@pytest.mark.parametrize("D,S,Sk,H,most", [(32, 8, 8, 600, 1.3e-7), (64, 16, 16, 600, 2.0e-7),
                                           (96, 70, 70, 512, 3.4e-7), (64, 1024, 1024, 2, 4e-7),
                                           (128, 1024, 1024, 2, 5e-7), (128, 8, 8000, 1, 6e-7)])
def test_error_stays_below_the_fp32_kernels(hip, D, S, Sk, H, most):
    """The relative 2-norm error over normal data, held to what the FP32 MFMA
    kernel measures there (1.24e-7, 1.94e-7, 3.35e-7, 6.5e-7, 6.9e-7, 16e-7; the
    pieces 0.9, 1.5, 2.7, 2.6, 3.5 and 4.2e-7)."""
    q, k, v = inputs(D + S, 1, S, Sk - S, H, D)
    got = run(hip, q, k, v, H, Sk - S, False)
    want = attention64(q, k, v, H, Sk - S, False)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) <= most


@pytest.mark.parametrize("D", [8, 16, 104, 120, 128])
def test_priced_calls_with_rope(hip, D):
    """Short calls of many heads, which the plan gives to the FP32 MFMA, with RoPE
    and a past: the result of rotating q and k first, and float64's."""
    B, S, past, H = 48, 20, 9, 16
    q, k, v = inputs(D, B, S, past, H, D)
    tq, tk, tv = (hip.tensor(x) for x in (q, k, v))
    got = hip.flash_attention(tq, tk, tv, H, q_pos=past,
                              flags=hip.ATTN_CAUSAL | hip.ATTN_ROPE).numpy()
    rq, rk = hip.rope(tq, D, past), hip.rope(tk, D, 0)
    first = hip.flash_attention(rq, rk, tv, H, q_pos=past, flags=hip.ATTN_CAUSAL).numpy()
    assert np.array_equal(got, first)
    want = attention64(rq.numpy()[-2:], rk.numpy()[-2:], v[-2:], H, past, True)
    check(got[-2:], want, f"D={D}")
