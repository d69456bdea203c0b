"""GPU parity of the paged decode's partition merge and of short partitions,
against the CPU oracle at the decode's bound (2e-3 relative, 1e-5 absolute).
"""
import numpy as np
import pytest

import oracle
from conftest import assert_close, rng
from test_gpu_paged import ATOL, RTOL, make, run

pytestmark = pytest.mark.gpu


# Partition counts at the edges of the merge: two, one lane per partition
# (64, 65), one round of weights (256) and several (up to 630); row lengths
# odd, below and past the thread groups; heads whose context fits one
# partition or is empty beside long ones.
@pytest.mark.parametrize("D,H", [(1, 2), (7, 3), (50, 1), (64, 4), (128, 5), (300, 1), (513, 1),
                                 (1024, 1)])
@pytest.mark.parametrize("ctx", [(9, 16, 0), (512, 520, 8), (2048, 2049, 1), (5040, 3, 2600)])
def test_merge_edges(hip, monkeypatch, D, H, ctx):
    monkeypatch.setenv("CLOVE_PAGED_PART", "8")
    bs, B = 8, len(ctx)
    mb = max(ctx) // bs + 1
    q, kn, vn, kv, bt, cl = make(D + max(ctx), B, H, D, bs, B * mb + 1, mb, ctx)
    want = oracle.paged_attention(q, None, None, kv, bt, cl).reshape(B, H * D)
    got = run(hip, q, None, None, kv, bt, cl)
    assert_close(got, want, RTOL, ATOL, f"D={D} ctx={ctx}")
    assert np.array_equal(got, run(hip, q, None, None, kv, bt, cl))  # fixed order


# Few heads: the plan cuts the context into 64- and 128-token partitions.
@pytest.mark.parametrize("B,H,D,bs,ctx", [(1, 1, 64, 16, 4096), (1, 8, 128, 16, 1000),
                                          (1, 12, 80, 16, 300), (2, 4, 128, 32, 129),
                                          (3, 2, 1024, 8, 700), (1, 3, 96, 100, 1500)])
def test_short_partitions_as_planned(hip, B, H, D, bs, ctx):
    mb = ctx // bs + 1
    q, kn, vn, kv, bt, cl = make(B + D + ctx, B, H, D, bs, B * mb + 1, mb,
                                 [ctx - 17 * b for b in range(B)])
    want = oracle.paged_attention(q, kn, vn, kv, bt, cl).reshape(B, H * D)
    assert_close(run(hip, q, kn, vn, kv, bt, cl), want, RTOL, ATOL, f"{B} x {H} x {D} over {ctx}")


# The longest contexts that keep one partition, and one block more.
@pytest.mark.parametrize("D,blocks", [(64, 16), (64, 17), (128, 10), (128, 11), (80, 10), (80, 11)])
def test_one_partition_edge(hip, D, blocks):
    B, H, bs = 2, 6, 16
    ctx = [blocks * bs, blocks * bs - 3]
    q, kn, vn, kv, bt, cl = make(D + blocks, B, H, D, bs, B * blocks + 1, blocks, ctx)
    want = oracle.paged_attention(q, kn, vn, kv, bt, cl).reshape(B, H * D)
    assert_close(run(hip, q, kn, vn, kv, bt, cl), want, RTOL, ATOL, f"D={D} {blocks} blocks")


def test_more_pairs_than_one_grid_side(hip):
    """2^24 (sequence, head) pairs and more, a workgroup of 256 each: long
    sequences at both ends match a call of their own, the short ones copy v."""
    B, H, D, bs, blocks = 65535, 257, 4, 16, 129
    assert B * H * 256 > 2**32
    g = rng(3)
    kv = hip.tensor(g.standard_normal((2, blocks, bs, H, D), dtype=np.float32))
    long = [0, 1, 300, B - 1]
    ctx = np.ones(B, np.int32)
    ctx[long] = [2064, 2050, 2063, 2051]  # past one partition of 2048 tokens
    bt = np.tile(np.arange(blocks, dtype=np.int32), (B, 1))
    q = hip.empty((B, H * D)).fill_normal(4)
    got = hip.paged_attention(q, None, None, kv, hip.tensor(bt, np.int32),
                              hip.tensor(ctx, np.int32), 0.5)
    rows = np.stack([q.read(i * H * D, H * D) for i in long])
    want = hip.paged_attention(hip.tensor(rows), None, None, kv, hip.tensor(bt[long], np.int32),
                               hip.tensor(ctx[long], np.int32), 0.5).numpy()
    for i, w in zip(long, want):
        assert np.max(np.abs(got.read(i * H * D, H * D) - w.ravel())) <= 1e-5, i
    v0 = kv.read(blocks * bs * H * D, H * D)
    assert np.array_equal(got.read(2 * H * D, H * D), v0)
