"""The work that programs on this framework give it, as cases to be timed.

Each case is one call, or the short run of calls that a program makes
together, through clove_amd's public entry points: small MLP inference and
training, fused elementwise chains, row softmax and layer norm, the vocabulary
loss with its gradient, matmul and its backward, the paged decode, the
attention prefill and a whole transformer block.  Sizes are those of the
repository's configurations and benchmark (the 784-128-10 MLP, 4096-wide
layers of 32 heads of 128, 16-token KV blocks, a 50257-word vocabulary) and
generic ones around them; ``draw`` spreads over the same ranges.

A program keeps its tensors on the device, so ``prepare`` makes the inputs
there (torch owns the memory, the framework's handles borrow it) and ``run``
returns the framework's output tensors as torch views of the same memory.
"""
import math

import numpy as np
import torch

import clove_amd as ca

DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the 784-128-10 MLP's forward on one batch of 64: the smallest call a
        # program makes, all launch latency
        dict(name="mlp_infer", kind="mlp_infer", batch=64, d_in=784, hidden=128, classes=10),
        # one training step of the same MLP: forward, loss, every gradient,
        # the AdamW update -- some twenty small launches
        dict(name="mlp_train", kind="mlp_train", batch=64, d_in=784, hidden=128, classes=10),
        # the fused chain gelu(a*b + c)*d with a broadcast c, 4096 x 4096: an
        # activation with its bias and gate, bound by memory
        dict(name="chain", kind="chain", rows=4096, cols=4096),
        # row softmax and layer norm over [8192, 4096]: the norms of a long
        # batch of 4096-wide tokens
        dict(name="rows", kind="rows", rows=8192, cols=4096),
        # cross entropy over a vocabulary and its gradient, the end of a
        # language model's forward pass and the start of its backward; the
        # vocabulary's width is odd
        dict(name="vocab_loss", kind="vocab_loss", rows=1024, cols=50257),
        # a decode step's projection: 32 tokens against a 4096 x 4096 weight
        dict(name="matmul_decode", kind="matmul", m=32, k=4096, n=4096),
        # the large square product
        dict(name="matmul_large", kind="matmul", m=4096, k=4096, n=4096),
        # both gradients of a layer at sizes that no tile divides, with the
        # bias's gradient
        dict(name="matmul_grads", kind="matmul_grads", m=2050, k=1028, n=3000),
        # one decode step of a full batch: 32 sequences of 512 to 4096 tokens
        dict(name="decode_batch", kind="decode", seqs=32, heads=32, head_dim=128, block=16,
             ctx_lo=512, ctx_hi=4096, new=False),
        # the same for two long conversations with the new token's row in
        # hand: little to spread over the chip, so latency counts
        dict(name="decode_few", kind="decode", seqs=2, heads=32, head_dim=128, block=16,
             ctx_lo=6000, ctx_hi=8192, new=True),
        # the prompt's attention, 4096 tokens of 32 heads of 128, causal + RoPE
        dict(name="prefill", kind="prefill", batch=1, s=4096, past=0, heads=32, head_dim=128,
             causal=True, rope=True),
        # a whole pre-norm transformer block over a ragged batch of tokens,
        # 12 heads of 64: three projections, attention, the MLP half as one
        # compiled graph
        dict(name="block", kind="block", batch=2, s=777, heads=12, head_dim=64, ffn=3072),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp_infer", "mlp_train", "chain", "rows", "vocab_loss", "matmul",
                       "matmul", "matmul_grads", "decode", "decode", "prefill", "prefill",
                       "block"])
    if kind in ("mlp_infer", "mlp_train"):
        return dict(kind=kind, batch=_log(rng, 1, 512), d_in=_log(rng, 16, 1024),
                    hidden=_log(rng, 16, 1024), classes=_log(rng, 2, 100))
    if kind == "chain":
        return dict(kind=kind, rows=_log(rng, 1, 4096), cols=_log(rng, 64, 4096))
    if kind == "rows":
        return dict(kind=kind, rows=_log(rng, 1, 8192), cols=_log(rng, 64, 4096))
    if kind == "vocab_loss":
        return dict(kind=kind, rows=_log(rng, 8, 1024), cols=_log(rng, 1000, 50257))
    if kind == "matmul":
        n = _log(rng, 64, 4096)
        return dict(kind=kind, m=_log(rng, 1, 4096), k=_log(rng, 64, 4096),
                    n=n if rng.random() < 0.5 else 64 * max(1, n // 64))
    if kind == "matmul_grads":
        def whole(x):
            return x if rng.random() < 0.5 else 32 * max(1, x // 32)
        return dict(kind=kind, m=whole(_log(rng, 64, 4096)), k=whole(_log(rng, 64, 3000)),
                    n=whole(_log(rng, 64, 3000)))
    if kind == "decode":
        lo = _log(rng, 16, 4096)
        return dict(kind=kind, seqs=_log(rng, 1, 32), heads=rng.choice([8, 12, 16, 32]),
                    head_dim=rng.choice([64, 64, 80, 96, 128, 128]),
                    block=rng.choice([8, 16, 16, 32]), ctx_lo=lo, ctx_hi=_log(rng, lo, 4096),
                    new=rng.random() < 0.5)
    if kind == "prefill":
        s = _log(rng, 16, 2048)
        # a later chunk of a prompt attends to the chunks before it
        past = 0 if rng.random() < 0.6 else _log(rng, 64, 4096 - s)
        return dict(kind=kind, batch=rng.choice([1, 1, 2]), s=s, past=past,
                    heads=rng.choice([8, 12, 16, 32]), head_dim=rng.choice([64, 64, 80, 96, 128]),
                    causal=rng.random() < 0.8, rope=rng.random() < 0.7)
    heads = rng.choice([4, 8, 12, 16])
    return dict(kind="block", batch=rng.choice([1, 2, 3]), s=_log(rng, 16, 1024), heads=heads,
                head_dim=64, ffn=heads * 64 * 4)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, shape, std=1.0):
    t = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    return t.mul_(std) if std != 1.0 else t


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float32).mul_(hi - lo).add_(lo)


def _classes(g, rows, classes):
    """Class indices, f32 as every tensor of the reference is."""
    return torch.randint(0, classes, (rows,), generator=g, device=DEV).float()


def _mlp_data(c, g):
    d, h, o = c["d_in"], c["hidden"], c["classes"]
    s1, s2 = math.sqrt(6.0 / d), math.sqrt(6.0 / h)
    return dict(x=_uniform(g, (c["batch"], d), 0.0, 1.0), w1=_uniform(g, (d, h), -s1, s1),
                b1=_uniform(g, (1, h), -0.1, 0.1), w2=_uniform(g, (h, o), -s2, s2),
                b2=_uniform(g, (1, o), -0.1, 0.1))


def _data(c, seed):
    """The case's inputs, torch f32 (or int32) tensors on the device."""
    g = _gen(seed)
    kind = c["kind"]
    if kind == "mlp_infer":
        return _mlp_data(c, g)
    if kind == "mlp_train":
        d = _mlp_data(c, g)
        d["t"] = _classes(g, c["batch"], c["classes"])
        d["one"] = torch.ones((1, 1), device=DEV)
        for p in ("w1", "b1", "w2", "b2"):  # moments of a run under way
            d["m_" + p] = _normal(g, d[p].shape, 1e-3)
            d["v_" + p] = _uniform(g, d[p].shape, 1e-5, 1e-4)
        return d
    if kind == "chain":
        shape = (c["rows"], c["cols"])
        return dict(a=_normal(g, shape), b=_normal(g, shape), c=_normal(g, (c["cols"],)),
                    d=_normal(g, shape))
    if kind == "rows":
        return dict(x=_normal(g, (c["rows"], c["cols"]), 2.0),
                    gamma=_uniform(g, (c["cols"],), 0.5, 1.5),
                    beta=_uniform(g, (c["cols"],), -0.1, 0.1))
    if kind == "vocab_loss":
        return dict(x=_normal(g, (c["rows"], c["cols"]), 2.0),
                    t=_classes(g, c["rows"], c["cols"]),
                    one=torch.full((1, 1), 1.0, device=DEV))
    if kind == "matmul":
        std = 1.0 / math.sqrt(c["k"])
        return dict(a=_normal(g, (c["m"], c["k"]), std), b=_normal(g, (c["k"], c["n"]), std))
    if kind == "matmul_grads":
        std = 1.0 / math.sqrt(c["k"])
        return dict(a=_normal(g, (c["m"], c["k"])), b=_normal(g, (c["k"], c["n"]), std),
                    g=_normal(g, (c["m"], c["n"]), 0.01))
    if kind == "decode":
        B, H, D, bs = c["seqs"], c["heads"], c["head_dim"], c["block"]
        ctx = torch.randint(c["ctx_lo"], c["ctx_hi"] + 1, (B,), generator=g, device=DEV)
        need = ((ctx + bs - 1) // bs).cpu().tolist()
        max_blocks = -(-c["ctx_hi"] // bs)
        # a pool about half of which these sequences hold, its blocks handed
        # out in no order
        pool = 2 * B * max_blocks
        perm = torch.randperm(pool, generator=g, device=DEV).to(torch.int32).cpu()
        bt = torch.full((B, max_blocks), -1, dtype=torch.int32)
        at = 0
        for i, n in enumerate(need):
            bt[i, :n] = perm[at:at + n]
            at += n
        d = dict(q=_normal(g, (B, H * D)), kv=_normal(g, (2, pool, bs, H, D)),
                 bt=bt.to(DEV), ctx=ctx.to(torch.int32))
        if c["new"]:
            d["k"] = _normal(g, (B, H * D))
            d["v"] = _normal(g, (B, H * D))
        return d
    if kind == "prefill":
        X = c["heads"] * c["head_dim"]
        B, S = c["batch"], c["s"]
        Sk = S + c["past"]
        return dict(q=_normal(g, (B, S, X)), k=_normal(g, (B, Sk, X)), v=_normal(g, (B, Sk, X)))
    if kind == "block":
        X, F = c["heads"] * c["head_dim"], c["ffn"]
        std, fstd = 1.0 / math.sqrt(X), 1.0 / math.sqrt(F)
        d = dict(x=_normal(g, (c["batch"], c["s"], X)))
        for n in ("g1", "g2"):
            d[n] = _uniform(g, (X,), 0.5, 1.5)
        for n in ("e1", "e2"):
            d[n] = _uniform(g, (X,), -0.1, 0.1)
        for n in ("wq", "wk", "wv", "wo"):
            d[n] = _normal(g, (X, X), std)
        d["w1"], d["c1"] = _normal(g, (X, F), std), _normal(g, (1, F), 0.1)
        d["w2"], d["c2"] = _normal(g, (F, X), fstd), _normal(g, (1, X), 0.1)
        return d
    raise ValueError(kind)


def prepare(case, seed):
    ca.init(0)
    data = _data(case, seed)
    torch.cuda.synchronize()  # the framework's stream does not wait for torch's
    h = {n: ca.wrap(t.data_ptr(), tuple(t.shape),
                    np.int32 if t.dtype == torch.int32 else np.float32)
         for n, t in data.items()}
    st = dict(case=case, data=data, h=h, run=globals()["_run_" + case["kind"]])
    if case["kind"] == "mlp_infer":
        gr = ca.Graph()
        ids = [gr.input(data[n].shape) for n in ("x", "w1", "b1", "w2", "b2")]
        y = gr.op("relu", gr.op("add", gr.op("matmul", ids[0], ids[1]), ids[2]))
        y = gr.op("softmax", gr.op("add", gr.op("matmul", y, ids[3]), ids[4]))
        st["model"] = gr.compile([y])
        st["ins"] = [h[n] for n in ("x", "w1", "b1", "w2", "b2")]
    elif case["kind"] == "chain":
        st["chain"] = ca.FusedChain([("mul", -1, -2), ("add", 0, -3), ("gelu", 1), ("mul", 2, -4)],
                                    [h[n] for n in "abcd"])
    elif case["kind"] == "block":
        rows, X = case["batch"] * case["s"], case["heads"] * case["head_dim"]
        gr = ca.Graph()
        x = gr.input((rows, X))
        g2, e2, w1, c1, w2, c2 = (gr.input(data[n].shape) for n in ("g2", "e2", "w1", "c1", "w2",
                                                                    "c2"))
        y = gr.op("layer_norm", x, g2, e2)
        y = gr.op("gelu", gr.op("add", gr.op("matmul", y, w1), c1))
        y = gr.op("add", gr.op("matmul", y, w2), c2)
        st["mlp"] = gr.compile([gr.op("add", x, y)])
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

class _Memory:
    """One output tensor's memory, for torch to view; it keeps the tensor."""

    def __init__(self, t, shape):
        self.t = t
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", version=2,
                                             data=(t.device_ptr, False))


def _view(t, shape):
    return torch.as_tensor(_Memory(t, tuple(shape)), device=DEV)


def run(state):
    return state["run"](state["case"], state["h"], state)


def _run_mlp_infer(c, h, st):
    return _view(st["model"].execute(st["ins"])[0], (c["batch"], c["classes"]))


def _run_mlp_train(c, h, st):
    a1 = ca.add(ca.matmul(h["x"], h["w1"]), h["b1"])
    r1 = ca.relu(a1)
    logits = ca.add(ca.matmul(r1, h["w2"]), h["b2"])
    loss = ca.cross_entropy(logits, h["t"])
    gl = ca.cross_entropy_backward(logits, h["t"], h["one"])
    gb2 = ca.broadcast_grad(gl, c["classes"])
    gr, gw2 = ca.matmul_backward(r1, h["w2"], gl)
    ga = ca.relu_backward(a1, gr)
    gb1 = ca.broadcast_grad(ga, c["hidden"])
    _, gw1 = ca.matmul_backward(h["x"], h["w1"], ga, want_a=False)
    names = ("w1", "b1", "w2", "b2")
    ca.adamw_step([h[n] for n in names], [gw1, gb1, gw2, gb2], [h["m_" + n] for n in names],
                  [h["v_" + n] for n in names], 100, lr=1e-5, loss_scale=1.0)
    d = st["data"]
    out = {n: d[n] for n in names}
    out.update(loss=_view(loss, (1, 1)), logits=_view(logits, (c["batch"], c["classes"])),
               gw1=_view(gw1, d["w1"].shape), gb1=_view(gb1, (c["hidden"],)),
               gw2=_view(gw2, d["w2"].shape), gb2=_view(gb2, (c["classes"],)))
    return out


def _run_chain(c, h, st):
    return _view(st["chain"]()[0], (c["rows"], c["cols"]))


def _run_rows(c, h, st):
    shape = (c["rows"], c["cols"])
    return (_view(ca.softmax(h["x"]), shape),
            _view(ca.layer_norm(h["x"], h["gamma"], h["beta"]), shape))


def _run_vocab_loss(c, h, st):
    return (_view(ca.cross_entropy(h["x"], h["t"]), (1, 1)),
            _view(ca.cross_entropy_backward(h["x"], h["t"], h["one"]), (c["rows"], c["cols"])))


def _run_matmul(c, h, st):
    return _view(ca.matmul(h["a"], h["b"]), (c["m"], c["n"]))


def _run_matmul_grads(c, h, st):
    ga, gb = ca.matmul_backward(h["a"], h["b"], h["g"])
    return (_view(ga, (c["m"], c["k"])), _view(gb, (c["k"], c["n"])),
            _view(ca.broadcast_grad(h["g"], c["n"]), (c["n"],)))


def _run_decode(c, h, st):
    o = ca.paged_attention(h["q"], h.get("k"), h.get("v"), h["kv"], h["bt"], h["ctx"])
    return _view(o, (c["seqs"], c["heads"] * c["head_dim"]))


def _run_prefill(c, h, st):
    flags = (ca.ATTN_CAUSAL if c["causal"] else 0) | (ca.ATTN_ROPE if c["rope"] else 0)
    o = ca.flash_attention(h["q"], h["k"], h["v"], c["heads"], q_pos=c["past"], k_pos=0,
                           flags=flags)
    return _view(o, (c["batch"], c["s"], c["heads"] * c["head_dim"]))


def _run_block(c, h, st):
    n = ca.layer_norm(h["x"], h["g1"], h["e1"])
    q, k, v = (ca.matmul(n, h[w]) for w in ("wq", "wk", "wv"))
    a = ca.flash_attention(q, k, v, c["heads"])
    x1 = ca.add(h["x"], ca.matmul(a, h["wo"]))
    rows, X = c["batch"] * c["s"], c["heads"] * c["head_dim"]
    flat = ca.wrap(x1.device_ptr, (rows, X))
    y = st["mlp"].execute([flat, h["g2"], h["e2"], h["w1"], h["c1"], h["w2"], h["c2"]])[0]
    return _view(y, (c["batch"], c["s"], X))


# ---------------------------------------------------------------------------
# the work of one pass, and what its result may differ by
# ---------------------------------------------------------------------------

def _visible(c):
    """(query, key) pairs of one head that the mask leaves."""
    s, past = c["s"], c["past"]
    return s * past + s * (s + 1) // 2 if c["causal"] else s * (s + past)


def work(case):
    c, kind = case, case["kind"]
    f4 = 4
    if kind in ("mlp_infer", "mlp_train"):
        B, d, h, o = c["batch"], c["d_in"], c["hidden"], c["classes"]
        params, mac = d * h + h + h * o + o, B * (d * h + h * o)
        if kind == "mlp_infer":
            return {"bytes": f4 * (B * d + params + B * o), "flops": 2 * mac}
        # weights and moments read and written, the inputs and targets read,
        # the gradients, logits and loss written
        return {"bytes": f4 * (B * d + B + 7 * params + B * o + 1),
                "flops": 2 * (2 * mac + B * h * o)}
    if kind == "chain":
        n = c["rows"] * c["cols"]
        return {"bytes": f4 * (4 * n + c["cols"]), "flops": 20 * n}
    if kind == "rows":
        n = c["rows"] * c["cols"]
        return {"bytes": f4 * (3 * n + 2 * c["cols"]), "flops": 12 * n}
    if kind == "vocab_loss":
        n = c["rows"] * c["cols"]
        return {"bytes": f4 * (2 * n + c["rows"]), "flops": 8 * n}
    if kind == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": f4 * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "matmul_grads":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": f4 * (2 * m * k + 2 * k * n + m * n + n), "flops": 4 * m * k * n}
    if kind == "decode":
        mean = (c["ctx_lo"] + c["ctx_hi"]) / 2
        row = c["heads"] * c["head_dim"]
        return {"bytes": f4 * c["seqs"] * row * (2 * mean + 2),
                "flops": 4 * c["seqs"] * row * mean}
    if kind == "prefill":
        row = c["heads"] * c["head_dim"]
        return {"bytes": f4 * c["batch"] * row * (4 * c["s"] + 2 * c["past"]),
                "flops": 4 * c["batch"] * row * _visible(c)}
    X, F, T = c["heads"] * c["head_dim"], c["ffn"], c["batch"] * c["s"]
    return {"bytes": f4 * (2 * T * X + 4 * X * X + 2 * X * F + 5 * X + F),
            "flops": 2 * T * (4 * X * X + 2 * X * F)
            + 4 * X * c["batch"] * c["s"] * (c["s"] + 1) // 2}


def tolerance(case):
    kind = case["kind"]
    if kind in ("chain", "rows", "vocab_loss"):
        return {"rel": 2e-6}     # hardware exp2 and f32 sums of one row
    if kind in ("matmul", "matmul_grads"):
        return {"rel": 8e-6}     # f32 sums of up to 4096 terms in another order
    if kind in ("mlp_infer", "mlp_train"):
        return {"rel": 8e-6}     # two layers of such sums
    if kind == "decode":
        return {"rel": 4e-6}
    return {"rel": 1e-5}         # prefill and block: products, softmax, products


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _norm(x, g, b):
    mean = x.mean(-1, keepdim=True)
    var = ((x - mean) ** 2).mean(-1, keepdim=True)
    return (x - mean) / torch.sqrt(var + 1e-5) * g + b


def _rope(x, heads, pos0):
    """Pairs (i, i + 1) of each head turned by pos / 10000^(i/D); that angle
    is formed in f32, as its definition here says."""
    B, S, X = x.shape
    D = X // heads
    i = np.arange(0, D, 2, dtype=np.float32) / np.float32(D)
    div = torch.from_numpy(np.power(10000.0, i.astype(np.float64)).astype(np.float32)).to(DEV)
    pos = torch.arange(pos0, pos0 + S, device=DEV, dtype=torch.float32)
    theta = (pos[:, None] / div[None, :]).double()
    c, s = torch.cos(theta)[None, :, None, :], torch.sin(theta)[None, :, None, :]
    x = x.view(B, S, heads, D // 2, 2)
    return torch.stack((x[..., 0] * c - x[..., 1] * s, x[..., 0] * s + x[..., 1] * c),
                       -1).reshape(B, S, X)


def _attention(q, k, v, heads, past, causal, rope):
    if rope:
        q, k = _rope(q, heads, past), _rope(k, heads, 0)
    B, S, X = q.shape
    Sk, D = k.shape[1], X // heads
    out = torch.empty_like(q)
    mask = None
    if causal:
        mask = (torch.arange(Sk, device=DEV)[None, :]
                > torch.arange(S, device=DEV)[:, None] + past)
    for b in range(B):
        for h in range(heads):
            cols = slice(h * D, (h + 1) * D)
            s = q[b, :, cols] @ k[b, :, cols].T / math.sqrt(D)
            if mask is not None:
                s.masked_fill_(mask, -math.inf)
            out[b, :, cols] = torch.softmax(s, -1) @ v[b, :, cols]
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    raw = _data(case, seed)
    if kind == "decode":
        return _exact_decode(c, raw)
    d = {n: t.double() for n, t in raw.items()}
    if kind == "mlp_infer":
        r = torch.relu(d["x"] @ d["w1"] + d["b1"])
        return torch.softmax(r @ d["w2"] + d["b2"], -1)
    if kind == "mlp_train":
        return _exact_mlp_train(c, d)
    if kind == "chain":
        return _gelu(d["a"] * d["b"] + d["c"]) * d["d"]
    if kind == "rows":
        return torch.softmax(d["x"], -1), _norm(d["x"], d["gamma"], d["beta"])
    if kind == "vocab_loss":
        t, n = raw["t"].long(), c["rows"]
        lp = torch.log_softmax(d["x"], -1)
        loss = -lp.gather(1, t[:, None]).sum() / n
        g = lp.exp_()
        g[torch.arange(n, device=DEV), t] -= 1.0
        return loss.view(1, 1), g / n
    if kind == "matmul":
        return d["a"] @ d["b"]
    if kind == "matmul_grads":
        return d["g"] @ d["b"].T, d["a"].T @ d["g"], d["g"].sum(0)
    if kind == "prefill":
        return _attention(d["q"], d["k"], d["v"], c["heads"], c["past"], c["causal"], c["rope"])
    n = _norm(d["x"], d["g1"], d["e1"])
    a = _attention(n @ d["wq"], n @ d["wk"], n @ d["wv"], c["heads"], 0, True, True)
    x1 = d["x"] + a @ d["wo"]
    y = _gelu(_norm(x1, d["g2"], d["e2"]) @ d["w1"] + d["c1"])
    return x1 + y @ d["w2"] + d["c2"]


def _exact_mlp_train(c, d):
    t, n = d["t"].long(), c["batch"]
    a1 = d["x"] @ d["w1"] + d["b1"]
    r1 = torch.relu(a1)
    logits = r1 @ d["w2"] + d["b2"]
    lp = torch.log_softmax(logits, -1)
    loss = -lp.gather(1, t[:, None]).sum() / n
    gl = lp.exp()
    gl[torch.arange(n, device=DEV), t] -= 1.0
    gl = gl / n
    ga = (gl @ d["w2"].T) * (a1 > 0)
    grads = dict(w1=d["x"].T @ ga, b1=ga.sum(0, keepdim=True), w2=r1.T @ gl,
                 b2=gl.sum(0, keepdim=True))
    lr, b1, b2, eps, decay, step = 1e-5, 0.9, 0.999, 1e-8, 0.01, 100
    out = dict(loss=loss.view(1, 1), logits=logits)
    for p, g in grads.items():
        gc = g.clamp(-1.0, 1.0)
        m = b1 * d["m_" + p] + (1 - b1) * gc
        v = b2 * d["v_" + p] + (1 - b2) * gc * gc
        w = d[p] * (1 - lr * decay)
        out[p] = w - lr * (m / (1 - b1 ** step)) / (torch.sqrt(v / (1 - b2 ** step)) + eps)
        out["g" + p] = g if p[0] == "w" else g.view(-1)
    return out


def _exact_decode(c, d):
    B, H, D, bs = c["seqs"], c["heads"], c["head_dim"], c["block"]
    out = torch.empty((B, H * D), device=DEV, dtype=torch.float64)
    for b, n in enumerate(d["ctx"].cpu().tolist()):
        blocks = d["bt"][b, :-(-n // bs)].long()
        k = d["kv"][0, blocks].reshape(-1, H, D)[:n].double().transpose(0, 1).contiguous()
        v = d["kv"][1, blocks].reshape(-1, H, D)[:n].double().transpose(0, 1).contiguous()
        if c["new"]:  # the last token comes from the rows in hand
            k[:, n - 1] = d["k"][b].view(H, D).double()
            v[:, n - 1] = d["v"][b].view(H, D).double()
        q = d["q"][b].view(H, 1, D).double()
        p = torch.softmax((k * q).sum(-1) / math.sqrt(D), -1)
        out[b] = (p[:, :, None] * v).sum(1).reshape(-1)
    return out
