"""The work that programs have this package do, as cases that can be timed: each kind of call
through its public entry point, from calls that launch latency decides to ones that fill the
chip, with odd sizes, padded strides and the options that are used in earnest.

`listed()` gives the cases, `draw(rng)` one more of the same ranges. A case is a dict of plain
values; `prepare(case, seed)` makes what a program has in hand before the call (tensors on the
GPU, weights, a model), `run(state)` is the call, `work(case)` the bytes and floating-point
operations it cannot do without, `tolerance(case)` how far another correct float32
implementation may be off, and `exact(case, seed)` the same outputs computed in float64 by plain
torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from piton_amd import cdiv, digits, next_power_of_2, tinygpt
from piton_amd.kernels import attn_fwd_kernel, dense_layer_kernel, dense_tiles, matmul_kernel, softmax_kernel
from piton_amd.kernels.attention import contiguous_strides
from piton_amd.runtime import mi355x

DEV = "cuda"


def listed() -> list:
    return [
        # the benchmark's matmul sizes: one that is over in a few microseconds, the ragged one
        # with padded rows, and the headline
        dict(name="matmul_512", kind="matmul", M=512, N=512, K=512, pad_a=0, pad_b=0, pad_c=0, b_t=False),
        dict(name="matmul_ragged", kind="matmul", M=1000, N=1800, K=700, pad_a=3, pad_b=5, pad_c=7, b_t=False),
        dict(name="matmul_4096", kind="matmul", M=4096, N=4096, K=4096, pad_a=0, pad_b=0, pad_c=0, b_t=False),
        # a product between them whose tiles neither cover its sides nor divide by the chip, B
        # stored transposed as weights often are
        dict(name="matmul_2500_bt", kind="matmul", M=2500, N=3000, K=2000, pad_a=0, pad_b=0, pad_c=0, b_t=True),
        # row softmax: the benchmark's odd row length, and rows of a large output vocabulary
        dict(name="softmax_1823", kind="softmax", rows=4096, cols=1823),
        dict(name="softmax_50000", kind="softmax", rows=512, cols=50000),
        # attention over a prompt: the benchmark's causal shape; unmasked with the widest heads
        # and a length that ends inside a block (draws also store K as [D, N])
        dict(name="attn_causal_1024", kind="attention", heads=32, n=1024, d=64, causal=True, k_layout="nd"),
        dict(name="attn_full_d128", kind="attention", heads=16, n=2000, d=128, causal=False, k_layout="nd"),
        # one new token per sequence against a long K/V cache (a decode step's attention)
        dict(name="attn_decode_4096", kind="decode", batch=8, heads=8, keys=4096, d=64),
        # one dense layer with bias and ReLU over a batch, wider than the digits network's
        dict(name="dense_2000", kind="dense", M=2000, N=1000, K=784, relu=True),
        # the digits network on one image: nothing but latency
        dict(name="digits_1", kind="digits", batch=1),
        # the decoder end to end: 64 prompts of 32 tokens, 16 more tokens
        dict(name="tinygpt_64x16", kind="tinygpt", batch=64, prompt=32, steps=16),
    ]


# -- draws --------------------------------------------------------------------------------------

def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi):
    """A size between lo and hi, evenly over its logarithm; half of them multiples of 64."""
    v = _log_int(rng, lo, hi)
    return max(lo, v // 64 * 64) if rng.random() < 0.5 and v >= 64 else v


def _draw_matmul(rng):
    M, N, K = (_side(rng, 64, 4096) for _ in range(3))
    pads = [rng.choice((0, 0, 4, rng.randint(1, 9))) for _ in range(3)]
    return dict(kind="matmul", M=M, N=N, K=K, pad_a=pads[0], pad_b=pads[1], pad_c=pads[2], b_t=rng.random() < 0.3)


def _draw_softmax(rng):
    cols = _side(rng, 64, 65536)
    return dict(kind="softmax", rows=_log_int(rng, 1, max(2, min(8192, 2 ** 25 // cols))), cols=cols)


def _draw_attention(rng):
    d, causal = rng.choice((32, 64, 64, 128)), rng.random() < 0.6
    n = _side(rng, 32, 4096)
    heads = _log_int(rng, 1, max(2, min(64, int(6e10 / (4.0 * n * n * d)))))
    return dict(kind="attention", heads=heads, n=n, d=d, causal=causal, k_layout=rng.choice(("nd", "nd", "dn")))


def _draw_decode(rng):
    batch, d = _log_int(rng, 1, 64), rng.choice((64, 64, 128))
    heads = rng.choice((4, 8, 16))
    top = max(64, min(8192, 2 ** 25 // (batch * heads * d)))
    return dict(kind="decode", batch=batch, heads=heads, keys=_log_int(rng, 32, top), d=d)


def _draw_dense(rng):
    return dict(kind="dense", M=_log_int(rng, 1, 8192), N=_side(rng, 10, 2048), K=_side(rng, 32, 2048),
                relu=rng.random() < 0.7)


def _draw_digits(rng):
    return dict(kind="digits", batch=_log_int(rng, 1, 1797))


def _draw_tinygpt(rng):
    return dict(kind="tinygpt", batch=_log_int(rng, 1, 64), prompt=rng.randint(4, 64), steps=rng.randint(2, 16))


def draw(rng) -> dict:
    kinds = ((_draw_matmul, 4), (_draw_softmax, 2), (_draw_attention, 3), (_draw_decode, 1), (_draw_dense, 2),
             (_draw_digits, 1), (_draw_tinygpt, 1))
    return rng.choices([k for k, _ in kinds], [w for _, w in kinds])[0](rng)


# -- inputs -------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _uniform(g, *shape, lo=-1.0, hi=1.0):
    return torch.rand(shape, device=DEV, generator=g) * (hi - lo) + lo


def _matmul_inputs(c, seed):
    """A [M, lda] and B [K, ldb] (or [N, ldb] when stored transposed), U[-1, 1]."""
    g = _gen(seed)
    lda, ldb, ldc = c["K"] + c["pad_a"], (c["K"] if c["b_t"] else c["N"]) + c["pad_b"], c["N"] + c["pad_c"]
    return _uniform(g, c["M"], lda), _uniform(g, c["N"] if c["b_t"] else c["K"], ldb), lda, ldb, ldc


def _softmax_inputs(c, seed):
    return torch.randn((c["rows"], c["cols"]), device=DEV, generator=_gen(seed)) * 4


def _attention_inputs(c, seed):
    """q, k, v [H, N, D], N(0, 1); k as [H, D, N] in layout "dn"."""
    g = _gen(seed)
    q, k, v = (torch.randn((c["heads"], c["n"], c["d"]), device=DEV, generator=g) for _ in range(3))
    return q, (k.transpose(1, 2).contiguous() if c["k_layout"] == "dn" else k), v


def _decode_inputs(c, seed):
    """The decoder's cache layout: rows t * batch + b of q | k | v, each heads * d wide."""
    return torch.randn((c["keys"] * c["batch"], 3 * c["heads"] * c["d"]), device=DEV, generator=_gen(seed))


def _dense_inputs(c, seed):
    g = _gen(seed)
    x = _uniform(g, c["M"], c["K"], lo=0.0)
    w = torch.randn((c["K"], c["N"]), device=DEV, generator=g) * math.sqrt(2.0 / c["K"])
    return x, w, _uniform(g, c["N"], lo=-0.1, hi=0.1)


def _digits_inputs(c, seed):
    """The digits network's He-normal layers, and images of whole pixel values 0..16 scaled to 0..1."""
    images = np.random.default_rng(seed).integers(0, 17, (c["batch"], 64))
    return digits.he_normal_mlp(seed), digits.normalize(images)


def _tinygpt_inputs(c, seed):
    cfg = tinygpt.Config()
    return cfg, tinygpt.init_weights(cfg, seed), tinygpt.seeded_prompts(c["batch"], c["prompt"], cfg.vocab, seed + 1)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "matmul":
        a, b, lda, ldb, ldc = _matmul_inputs(c, seed)
        out = torch.empty((c["M"], ldc), device=DEV)
        strides = (lda, 1, 1, ldb, ldc, 1) if c["b_t"] else (lda, 1, ldb, 1, ldc, 1)
        grid = (cdiv(c["M"], 64) * cdiv(c["N"], 64),)
        return dict(kind=kind, grid=grid, args=(a, b, out, c["M"], c["N"], c["K"], *strides), out=out[:, :c["N"]])
    if kind == "softmax":
        x = _softmax_inputs(c, seed)
        return dict(kind=kind, x=x, out=torch.empty_like(x), n=c["cols"], block=next_power_of_2(c["cols"]))
    if kind == "attention":
        q, k, v = _attention_inputs(c, seed)
        n, d = c["n"], c["d"]
        st, out = contiguous_strides(d, c["k_layout"], n), torch.empty_like(q)
        args = (q, k, v, out, 1.0 / math.sqrt(d), n * d, st["stride_qm"], n * d, st["stride_kn"], st["stride_kk"], n * d,
                st["stride_vn"], n * d, st["stride_om"], n)
        return dict(kind=kind, grid=(cdiv(n, 64), c["heads"]), args=args, out=out,
                    const=dict(HEAD_DIM=d, BLOCK_M=64, BLOCK_N=32, CAUSAL=c["causal"], EVEN_N=n % 32 == 0))
    if kind == "decode":
        cache = _decode_inputs(c, seed)
        B, H, n, d = c["batch"], c["heads"], c["keys"], c["d"]
        D = H * d
        out = torch.empty((B, D), device=DEV)
        args = (cache[(n - 1) * B:], cache[:, D:], cache[:, 2 * D:], out, 1.0 / math.sqrt(d), 3 * D, d, 3 * D, d,
                B * 3 * D, 3 * D, d, B * 3 * D, D, d, n, B, H, d)
        return dict(kind=kind, args=args, out=out)
    if kind == "dense":
        x, w, b = _dense_inputs(c, seed)
        bm, bn, bk = dense_tiles(c["N"])
        y = torch.empty((c["M"], c["N"]), device=DEV)
        return dict(kind=kind, grid=(cdiv(c["M"], bm) * cdiv(c["N"], bn),), args=(x, w, b, y, c["M"]), out=y,
                    const=dict(N=c["N"], K=c["K"], BLOCK_SIZE_M=bm, BLOCK_SIZE_N=bn, BLOCK_SIZE_K=bk, GROUP_SIZE_M=8,
                               ADD_BIAS=True, RELU=c["relu"]))
    if kind == "digits":
        layers, x = _digits_inputs(c, seed)
        return dict(kind=kind, model=digits.MLP(layers, c["batch"]), x=torch.from_numpy(x).to(DEV))
    if kind == "tinygpt":
        cfg, weights, prompts = _tinygpt_inputs(c, seed)
        model = tinygpt.TinyGPT(weights, cfg, batch=c["batch"])
        # a server's model has answered other prompts of this shape before
        model.generate(tinygpt.seeded_prompts(c["batch"], c["prompt"], cfg.vocab, seed + 2), c["steps"])
        return dict(kind=kind, model=model, prompts=prompts, steps=c["steps"])
    raise ValueError(f"unknown kind {kind!r}")


def run(state):
    kind = state["kind"]
    if kind == "matmul":
        matmul_kernel[state["grid"]](*state["args"], BLOCK_SIZE_M=64, BLOCK_SIZE_N=64, BLOCK_SIZE_K=16, GROUP_SIZE_M=8,
                                     device="mi355x")
    elif kind == "softmax":
        x, n = state["x"], state["n"]
        softmax_kernel[(x.shape[0],)](state["out"], x, n, n, n, BLOCK_SIZE=state["block"], device="mi355x")
    elif kind == "attention":
        attn_fwd_kernel[state["grid"]](*state["args"], **state["const"], device="mi355x")
    elif kind == "decode":
        mi355x.attn_decode(*state["args"])
    elif kind == "dense":
        dense_layer_kernel[state["grid"]](*state["args"], **state["const"], device="mi355x")
    elif kind == "digits":
        return state["model"].run(state["x"])
    else:
        tokens = state["model"].generate(state["prompts"], state["steps"])
        return state["model"].logits, tokens
    return state["out"]


# -- what a pass cannot do without, and how exact it is -------------------------------------------

def work(case) -> dict:
    c, kind = case, case["kind"]
    if kind == "matmul":
        M, N, K = c["M"], c["N"], c["K"]
        return dict(bytes=4 * (M * K + K * N + M * N), flops=2 * M * N * K)
    if kind == "softmax":
        n = c["rows"] * c["cols"]
        return dict(bytes=8 * n, flops=5 * n)
    if kind == "attention":
        H, n, d = c["heads"], c["n"], c["d"]
        pairs = n * (n + 1) // 2 if c["causal"] else n * n
        return dict(bytes=16 * H * n * d, flops=4 * H * d * pairs)
    if kind == "decode":
        n = c["batch"] * c["heads"] * c["d"]
        return dict(bytes=4 * (2 * n * c["keys"] + 2 * n), flops=4 * n * c["keys"])
    if kind == "dense":
        M, N, K = c["M"], c["N"], c["K"]
        return dict(bytes=4 * (M * K + K * N + N + M * N), flops=2 * M * N * K)
    if kind == "digits":
        macs = sum(k * n for k, n in zip(digits.SIZES[:-1], digits.SIZES[1:]))
        return dict(bytes=4 * (macs + sum(digits.SIZES[1:]) + c["batch"] * (64 + 10 + 1)), flops=2 * macs * c["batch"])
    cfg = tinygpt.Config()
    D, F, L, V, B = cfg.d_model, cfg.d_mlp, cfg.n_layers, cfg.vocab, c["batch"]
    T = c["prompt"] + c["steps"] - 1  # positions whose layers run
    weights = L * (4 * D * D + 2 * D * F)
    flops = 2 * B * T * weights + 4 * L * D * B * T * (T + 1) // 2 + 2 * B * c["steps"] * D * V
    # the weights once per forward, each position's q, k and v written, the cached keys and values
    # read by each later step
    cached = sum(2 * D * L * B * t for t in range(c["prompt"], T))
    nbytes = 4 * (c["steps"] * (weights + D * V) + 3 * D * L * B * T + cached)
    return dict(bytes=nbytes, flops=flops)


# Relative errors of float32 results, about four times the error against float64 that each kind
# shows over its range. A token is a whole value that a near tie of two logits may turn; the few
# steps of the decoder cases keep such a turn out of the compared logits.
_TOLERANCE = {"matmul": 5e-6, "softmax": 1e-6, "attention": 4e-6, "decode": 4e-6, "dense": 4e-6, "digits": 2e-6,
              "tinygpt": 4e-6}


def tolerance(case):
    t = {"rel": _TOLERANCE[case["kind"]]}
    if case["kind"] in ("digits", "tinygpt"):
        t["differ"] = 0.005
    return t


# -- float64 ------------------------------------------------------------------------------------

def _softmax64(s):
    e = torch.exp(s - s.amax(-1, keepdim=True))
    return e / e.sum(-1, keepdim=True)


def _attention64(q, k, v, causal):
    """One head: q, k, v [N, D] float64, 512 queries at a time."""
    n, d = k.shape
    kt, out = k.t().contiguous(), torch.empty_like(q)
    for i in range(0, q.shape[0], 512):
        s = (q[i:i + 512] @ kt) / math.sqrt(d)
        if causal:
            rows = torch.arange(i, i + s.shape[0], device=DEV)[:, None]
            s.masked_fill_(torch.arange(n, device=DEV)[None, :] > rows, float("-inf"))
        out[i:i + 512] = _softmax64(s) @ v
    return out


def _layernorm64(x, eps):
    m = x.mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + eps)


def _tinygpt64(cfg, weights, prompts, steps):
    w = {k: torch.from_numpy(v).to(DEV).double() for k, v in weights.items()}
    D, H, Dh = cfg.d_model, cfg.n_heads, cfg.head_dim
    ids = torch.from_numpy(prompts).to(DEV).long()
    for _ in range(steps):
        B, T = ids.shape
        x = (w["tok"][ids] + w["pos"][:T]).reshape(B * T, D)
        later = torch.arange(T, device=DEV)[None, :] > torch.arange(T, device=DEV)[:, None]
        for i in range(cfg.n_layers):
            qkv = (_layernorm64(x, cfg.eps) @ w[f"wqkv{i}"] + w[f"bqkv{i}"]).reshape(B, T, 3, H, Dh)
            q, k, v = (qkv[:, :, j].permute(0, 2, 1, 3).contiguous() for j in range(3))
            s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(Dh)
            p = _softmax64(s.masked_fill(later, float("-inf")))
            att = torch.matmul(p, v).permute(0, 2, 1, 3).reshape(B * T, D)
            x = x + att @ w[f"wo{i}"] + w[f"bo{i}"]
            x = x + torch.relu(_layernorm64(x, cfg.eps) @ w[f"w1{i}"] + w[f"b1{i}"]) @ w[f"w2{i}"] + w[f"b2{i}"]
        logits = _layernorm64(x.reshape(B, T, D)[:, -1], cfg.eps) @ w["lm"]
        ids = torch.cat([ids, logits.argmax(-1, keepdim=True)], 1)
    return logits, ids.to(torch.int32).cpu().numpy()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "matmul":
        a, b, *_ = _matmul_inputs(c, seed)
        b = b[:, :c["K"]].t() if c["b_t"] else b[:, :c["N"]]
        return a[:, :c["K"]].double() @ b.double().contiguous()
    if kind == "softmax":
        return _softmax64(_softmax_inputs(c, seed).double())
    if kind == "attention":
        q, k, v = _attention_inputs(c, seed)
        k = k.transpose(1, 2).contiguous() if c["k_layout"] == "dn" else k
        return torch.stack([_attention64(q[h].double(), k[h].double(), v[h].double(), c["causal"])
                            for h in range(c["heads"])])
    if kind == "decode":
        B, H, n, d = c["batch"], c["heads"], c["keys"], c["d"]
        qkv = _decode_inputs(c, seed).reshape(n, B, 3, H, d)
        return torch.stack([torch.cat([_attention64(qkv[n - 1, b, 0, h].double()[None], qkv[:, b, 1, h].double(),
                                                    qkv[:, b, 2, h].double(), False)[0] for h in range(H)])
                            for b in range(B)])
    if kind == "dense":
        x, w, b = (t.double() for t in _dense_inputs(c, seed))
        y = x @ w + b
        return torch.relu(y) if c["relu"] else y
    if kind == "digits":
        layers, x = _digits_inputs(c, seed)
        h = x.astype(np.float64)
        for i, (w, b) in enumerate(layers):
            h = h @ w.astype(np.float64) + b
            h = np.maximum(h, 0) if i + 1 < len(layers) else h
        return h, h.argmax(1).astype(np.int32)
    return _tinygpt64(*_tinygpt_inputs(c, seed), c["steps"])
