"""The work that programs built on this framework give it, as timed cases.

Each case is one layer, block or step as a training or inference program runs
it through the C ABI of libwm_hip (include/*.h): the forward entry point
followed by its closure where the program trains, with the calls in the order
the Tensor, Module, LossFunction and Optimizer classes make them.  Buffers are
torch tensors made beforehand, as a program's arena would hold them; the
library shares torch's HIP runtime because torch is imported first.

Kinds of case (the `kind` key) and what they stand for:

  linear     Linear::forward and backward: matmul, bias add, and the gradients
             of the input, the weight and the bias.
  xent       a classification head's CrossEntropyLoss, forward and backward.
  layernorm  LayerNorm, forward and backward.
  batchnorm  BatchNorm2d in training mode, forward and backward.
  bias       a broadcast bias over images or sequences followed by relu,
             forward and backward.
  pool       mean and max pooling over one axis, forward and backward.
  attention  MultiHeadAttention: self attention with the causal mask, forward
             and backward, or one pass of queries over a memory (inference).
  adamw      one AdamW step over a transformer's parameter list.
  epilogue   the fp16-storage block epilogue, forward and backward.
"""
import ctypes as C
import math

import torch

from whitematter_amd import _lib as W

F32 = 4
LN_EPS = 1e-5
BN_EPS, BN_MOMENTUM = 1e-5, 0.1
ADAMW = {"lr": 1e-3, "beta1": 0.9, "beta2": 0.999, "eps": 1e-8, "weight_decay": 0.01}
CLAMP = (-4.0, 4.0)


def listed():
    return [
        # A hidden layer of an MLP on 28 x 28 images, one small batch: the
        # smallest calls, where latency and the number of launches count.
        {"name": "linear-mlp", "kind": "linear", "rows": 64, "fin": 784, "fout": 128},
        # The MLP of a GPT-2-small block over 4096 tokens.
        {"name": "linear-transformer", "kind": "linear", "rows": 4096, "fin": 768, "fout": 3072},
        # The head of a ten-class image classifier.
        {"name": "xent-classes", "kind": "xent", "rows": 128, "classes": 10},
        # A language model's head over GPT-2's vocabulary (an odd row length).
        {"name": "xent-vocabulary", "kind": "xent", "rows": 2048, "classes": 50257},
        # The norm of a GPT-2-small block over 8192 tokens.
        {"name": "layernorm", "kind": "layernorm", "rows": 8192, "n": 768},
        # A late stage of a convolutional network (14 x 14 planes).
        {"name": "batchnorm", "kind": "batchnorm", "batch": 64, "channels": 256, "side": 14},
        # A convolution's channel bias and relu on [64, 64, 56, 56].
        {"name": "bias-channel", "kind": "bias", "layout": "channel", "outer": 64, "mid": 64, "inner": 56 * 56},
        # Mean and max pooling of a batch of token sequences (196 patches and
        # a class token).
        {"name": "pool-sequence", "kind": "pool", "outer": 64, "n": 197, "inner": 768},
        # Training: causal self attention of a GPT-2-small block.
        {"name": "attention-train", "kind": "attention", "train": True, "batch": 8, "sq": 512, "sk": 512,
         "embed": 768, "heads": 12},
        # Inference: one decoded position of 16 sequences over their memories.
        {"name": "attention-decode", "kind": "attention", "train": False, "batch": 16, "sq": 1, "sk": 333,
         "embed": 512, "heads": 8},
        # The optimizer step of a GPT-2-small-sized model (148 tensors).
        {"name": "adamw", "kind": "adamw", "width": 768, "layers": 12, "vocab": 50257, "context": 1024},
        # The block epilogue on fp16 activations.
        {"name": "epilogue-f16", "kind": "epilogue", "rows": 4096, "cols": 1024},
    ]


# ---- drawn cases --------------------------------------------------------------


def _logint(rng, lo, hi):
    """An integer in [lo, hi], uniform over the logarithm; half of the time
    rounded to a multiple of 16 (a power-of-two-ish width), else as it falls."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        v = max(lo, v // 16 * 16) if v >= 16 else v
    return min(max(v, lo), hi)


def draw(rng):
    kind = rng.choice(["linear", "xent", "layernorm", "batchnorm", "bias", "pool", "attention", "adamw", "epilogue"])
    if kind == "linear":
        fin, fout = _logint(rng, 32, 3072), _logint(rng, 8, 3072)
        rows = min(_logint(rng, 16, 8192), 4096 * 768 * 3072 // (fin * fout), (1 << 24) // max(fin, fout))
        return {"kind": kind, "rows": rows, "fin": fin, "fout": fout}
    if kind == "xent":
        classes = _logint(rng, 2, 50257)
        return {"kind": kind, "rows": min(_logint(rng, 32, 16384), 2048 * 50257 // classes), "classes": classes}
    if kind == "layernorm":
        n = _logint(rng, 32, 8192)
        return {"kind": kind, "rows": min(_logint(rng, 32, 32768), 8192 * 768 // n), "n": n}
    if kind == "batchnorm":
        side, channels = rng.randint(1, 56), _logint(rng, 3, 1024)
        most = 64 * 256 * 14 * 14 // (channels * side * side)
        return {"kind": kind, "batch": max(2, min(_logint(rng, 2, 128), most)),
                "channels": max(1, min(channels, 64 * 256 * 14 * 14 // (2 * side * side))), "side": side}
    if kind == "bias":
        layout = rng.choice(["channel", "row", "token"])
        most = 64 * 64 * 56 * 56
        if layout == "channel":
            inner = rng.randint(1, 56) ** 2
        else:
            inner = _logint(rng, 8, 4096)
        mid = _logint(rng, 2, 1024)
        return {"kind": kind, "layout": layout, "outer": max(1, min(_logint(rng, 2, 128), most // (mid * inner))),
                "mid": max(1, min(mid, most // inner)), "inner": inner}
    if kind == "pool":
        outer, n = _logint(rng, 1, 256), _logint(rng, 2, 4096)
        inner = 1 if rng.random() < 0.25 else _logint(rng, 2, 2048)
        most = 64 * 197 * 768
        n = max(1, min(n, most // outer))
        return {"kind": kind, "outer": outer, "n": n, "inner": max(1, min(inner, most // (outer * n)))}
    if kind == "attention":
        train = rng.random() < 0.5
        heads, width = rng.choice([2, 4, 6, 8, 12]), rng.choice([32, 48, 64])
        embed = heads * width
        sk = _logint(rng, 16, 1024)
        sq = sk if train else rng.choice([1, rng.randint(2, 64)])
        batch = _logint(rng, 1, 32)
        room = 8 * 512 * 768 * 12 if train else 16 * 333 * 512 * 8
        batch = max(1, min(batch, room // (sk * embed * heads)))
        if train:
            batch = max(1, min(batch, 8 * 12 * 512 * 512 // (heads * sk * sk)))
        sk = min(sk, room // (embed * heads))
        return {"kind": kind, "train": train, "batch": batch, "sq": sk if train else sq, "sk": sk, "embed": embed,
                "heads": heads}
    if kind == "adamw":
        return {"kind": kind, "width": rng.randint(3, 48) * 16, "layers": rng.randint(1, 12),
                "vocab": rng.choice([256, 10000, 32000]), "context": rng.choice([128, 512, 1024])}
    cols = _logint(rng, 64, 4096) // 8 * 8
    return {"kind": kind, "rows": min(_logint(rng, 64, 16384), 4096 * 1024 // cols), "cols": cols}


# ---- state --------------------------------------------------------------------


def _p(t):
    return C.c_void_p(t.data_ptr() if t is not None else 0)


def _i64(*v):
    return (C.c_int64 * len(v))(*v)


class _Maker:
    """Inputs from one seed, and output buffers, on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(shape, generator=self.gen, device="cuda") * std + mean

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo

    def labels(self, rows, classes):
        return torch.randint(0, classes, (rows,), generator=self.gen, device="cuda").float()


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _inputs(case, seed):
    """The case's inputs, by name, made from the seed alone."""
    m, kind = _Maker(seed), case["kind"]
    if kind == "linear":
        r, i, o = case["rows"], case["fin"], case["fout"]
        return {"x": m.normal(r, i), "w": m.normal(i, o, std=i ** -0.5), "b": m.normal(o, std=0.1),
                "g": m.normal(r, o, std=1.0 / r)}
    if kind == "xent":
        r, c = case["rows"], case["classes"]
        return {"x": m.normal(r, c, std=3.0), "labels": m.labels(r, c), "g": torch.ones(1, device="cuda")}
    if kind == "layernorm":
        r, n = case["rows"], case["n"]
        return {"x": m.normal(r, n), "gamma": m.normal(n, std=0.1, mean=1.0), "beta": m.normal(n, std=0.1),
                "g": m.normal(r, n)}
    if kind == "batchnorm":
        b, c, s = case["batch"], case["channels"], case["side"] ** 2
        return {"x": m.normal(b, c, s), "gamma": m.normal(c, std=0.1, mean=1.0), "beta": m.normal(c, std=0.1),
                "g": m.normal(b, c, s), "rm": m.normal(c, std=0.1), "rv": m.uniform(0.5, 1.5, c)}
    if kind == "bias":
        a, b = _bias_shapes(case)
        return {"x": m.normal(*a), "b": m.normal(*b, std=0.5), "g": m.normal(*a)}
    if kind == "pool":
        o, n, i = case["outer"], case["n"], case["inner"]
        return {"x": m.normal(o, n, i), "g_mean": m.normal(o, i, std=1.0 / n), "g_max": m.normal(o, i)}
    if kind == "attention":
        b, sq, sk, e = case["batch"], case["sq"], case["sk"], case["embed"]
        d = {"q": m.normal(b, sq, e)}
        d["kv"] = d["q"] if case["train"] else m.normal(b, sk, e)
        for k in "qkvo":
            d["w" + k] = m.normal(e, e, std=e ** -0.5)
            d["b" + k] = m.normal(e, std=0.1)
        if case["train"]:
            d["mask"] = torch.triu(torch.full((sq, sk), -1e9, device="cuda"), diagonal=1)
            d["g"] = m.normal(b, sq, e)
        return d
    if kind == "adamw":
        total = _spans(case)[1]
        return {"p": m.normal(total, std=0.02), "g": m.normal(total, std=1e-2),
                "m": m.normal(total, std=1e-3), "v": m.uniform(1e-6, 1e-4, total)}
    r, c = case["rows"], case["cols"]
    return {"h": m.normal(r, c).half(), "res": m.normal(r, c).half(), "gain": m.uniform(0.8, 1.2, c),
            "g": m.normal(r, std=1.0 / c)}


def _bias_shapes(case):
    o, m, i = case["outer"], case["mid"], case["inner"]
    side = math.isqrt(i)
    if case["layout"] == "channel":  # [N, C, H, W] + [1, C, 1, 1]
        return (o, m, side, side), (1, m, 1, 1)
    if case["layout"] == "token":  # [N, T, E] + [N, 1, E]
        return (o, m, i), (o, 1, i)
    return (o * m, i), (i,)  # [N T, E] + [E]


def _spans(case):
    """The parameter list of a GPT-2-like model: (element counts, where each
    starts in one arena, 256-byte aligned), and the arena's size."""
    d, v, ctx = case["width"], case["vocab"], case["context"]
    sizes = [v * d, ctx * d]
    for _ in range(case["layers"]):
        sizes += [d, d, 3 * d * d, 3 * d, d * d, d, d, d, 4 * d * d, 4 * d, 4 * d * d, d]
    sizes += [d, d]
    starts, at = [], 0
    for n in sizes:
        starts.append(at)
        at += (n + 63) // 64 * 64
    return list(zip(sizes, starts)), at


def prepare(case, seed):
    W.call("wm_init", torch.cuda.current_device())
    d, kind = _inputs(case, seed), case["kind"]
    L, f = W.lib(), C.c_float
    if kind == "linear":
        r, i, o = case["rows"], case["fin"], case["fout"]
        z, y, gz, gx, gw, gb = _empty(r, o), _empty(r, o), _empty(r, o), _empty(r, i), _empty(i, o), _empty(o)
        zs, bs = _i64(r, o), _i64(o)
        calls = [
            (L.wm_matmul, (_p(d["x"]), _p(d["w"]), r, i, o, _p(z))),
            (L.wm_binary, (W.ADD, _p(y), _p(z), zs, 2, _p(d["b"]), bs, 1)),
            (L.wm_binary_bwd, (W.ADD, _p(d["g"]), _p(z), zs, 2, _p(d["b"]), bs, 1, None, _p(gz), 0, _p(gb), 0)),
            (L.wm_matmul_bwd, (_p(gz), _p(d["x"]), _p(d["w"]), r, i, o, _p(gx), 0, _p(gw), 0)),
        ]
        out, keep = {"y": y, "gx": gx, "gw": gw, "gb": gb}, [z, gz, zs, bs]
    elif kind == "xent":
        r, c = case["rows"], case["classes"]
        stats, loss, gx = _empty(r, W.CE_STATS), _empty(1), _empty(r, c)
        calls = [
            (L.wm_cross_entropy_fwd, (_p(d["x"]), _p(d["labels"]), r, c, _p(stats), _p(loss))),
            (L.wm_cross_entropy_bwd, (_p(d["x"]), _p(d["labels"]), _p(stats), _p(d["g"]), _p(gx), 0, r, c)),
        ]
        out, keep = {"loss": loss, "gx": gx}, [stats]
    elif kind == "layernorm":
        r, n = case["rows"], case["n"]
        y, mean, inv, gx, gg, gb = _empty(r, n), _empty(r), _empty(r), _empty(r, n), _empty(n), _empty(n)
        calls = [
            (L.wm_layernorm_fwd, (_p(d["x"]), _p(d["gamma"]), _p(d["beta"]), r, n, f(LN_EPS), _p(y), _p(mean),
                                  _p(inv))),
            (L.wm_layernorm_bwd, (_p(d["g"]), _p(d["x"]), _p(d["gamma"]), _p(mean), _p(inv), r, n, _p(gx), 0, _p(gg),
                                  0, _p(gb), 0)),
        ]
        out, keep = {"y": y, "gx": gx, "ggamma": gg, "gbeta": gb}, [mean, inv]
    elif kind == "batchnorm":
        b, c, s = case["batch"], case["channels"], case["side"] ** 2
        y, gx, mean, inv = _empty(b, c, s), _empty(b, c, s), _empty(c), _empty(c)
        gg, gb = _empty(c), _empty(c)
        calls = [
            (L.wm_batchnorm2d_fwd, (_p(d["x"]), _p(d["gamma"]), _p(d["beta"]), _p(d["rm"]), _p(d["rv"]), b, c, s,
                                    f(BN_EPS), f(BN_MOMENTUM), 1, _p(y), _p(mean), _p(inv))),
            (L.wm_batchnorm2d_bwd, (_p(d["g"]), _p(d["x"]), _p(d["gamma"]), _p(mean), _p(inv), b, c, s, _p(gx), 0,
                                    _p(gg), 0, _p(gb), 0)),
        ]
        out, keep = {"y": y, "gx": gx, "ggamma": gg, "gbeta": gb, "rm": d["rm"], "rv": d["rv"]}, [mean, inv]
    elif kind == "bias":
        a, b = _bias_shapes(case)
        sa, sb, n = _i64(*a), _i64(*b), math.prod(a)
        t, y, gt, gx, gb = _empty(*a), _empty(*a), _empty(*a), _empty(*a), _empty(*b)
        calls = [
            (L.wm_binary, (W.ADD, _p(t), _p(d["x"]), sa, len(a), _p(d["b"]), sb, len(b))),
            (L.wm_unary, (W.RELU, _p(y), _p(t), n, f(0), f(0))),
            (L.wm_unary_bwd, (W.RELU, _p(d["g"]), _p(t), _p(y), _p(gt), 0, n, f(0), f(0))),
            (L.wm_binary_bwd, (W.ADD, _p(gt), _p(d["x"]), sa, len(a), _p(d["b"]), sb, len(b), None, _p(gx), 0,
                               _p(gb), 0)),
        ]
        out, keep = {"y": y, "gx": gx, "gb": gb}, [t, gt, sa, sb]
    elif kind == "pool":
        o, n, i = case["outer"], case["n"], case["inner"]
        mean, top, idx, gx = _empty(o, i), _empty(o, i), _empty(o, i, dtype=torch.int64), _empty(o, n, i)
        calls = [
            (L.wm_reduce, (W.R_MEAN, _p(d["x"]), o, n, i, _p(mean), None)),
            (L.wm_reduce, (W.R_MAX, _p(d["x"]), o, n, i, _p(top), _p(idx))),
            (L.wm_reduce_bwd, (W.R_MEAN, _p(d["g_mean"]), None, o, n, i, _p(gx), 0)),
            (L.wm_reduce_bwd, (W.R_MAX, _p(d["g_max"]), _p(idx), o, n, i, _p(gx), 1)),
        ]
        out, keep = {"mean": mean, "max": top, "index": idx, "gx": gx}, []
    elif kind == "attention":
        calls, out, keep = _attention_calls(L, case, d)
    elif kind == "adamw":
        return _adamw_state(case, d)
    else:
        r, c = case["rows"], case["cols"]
        y, mean = _empty(r, c, dtype=torch.float16), _empty(r)
        gh, gres, gg = _empty(r, c), _empty(r, c), _empty(c)
        lo, hi = f(CLAMP[0]), f(CLAMP[1])
        calls = [
            (L.wm_epilogue_f16_fwd, (_p(y), _p(mean), _p(d["h"]), _p(d["res"]), _p(d["gain"]), r, c, lo, hi)),
            (L.wm_epilogue_f16_bwd, (_p(d["g"]), _p(d["h"]), _p(d["res"]), _p(d["gain"]), _p(gh), 0, _p(gres), 0,
                                     _p(gg), 0, r, c, lo, hi)),
        ]
        out, keep = {"y": y, "mean": mean, "gh": gh, "gres": gres, "ggain": gg}, []
    torch.cuda.synchronize()
    return {"calls": calls, "out": out, "keep": (d, keep)}


def _attention_calls(L, case, d):
    b, sq, sk, e, h = case["batch"], case["sq"], case["sk"], case["embed"], case["heads"]
    y, ctx, Q = _empty(b, sq, e), _empty(b, sq, e), _empty(b, sq, e)
    K, V, attn = _empty(b, sk, e), _empty(b, sk, e), _empty(b, h, sq, sk)
    mask = d.get("mask")
    ws, bs = [_p(d["w" + k]) for k in "qkvo"], [_p(d["b" + k]) for k in "qkvo"]
    q, kv = _p(d["q"]), _p(d["kv"])
    calls = [(L.wm_mha_fwd, (q, kv, kv, _p(mask), 1, *ws, *bs, b, sq, sk, e, h, _p(y), _p(attn), _p(Q), _p(K), _p(V),
                             _p(ctx)))]
    out, keep = {"y": y, "attn": attn}, [ctx, Q, K, V]
    if case["train"]:
        # The module's gradients are added to, so the step clears them first:
        # one arena holds the eight parameter gradients and the input's.
        grads = _empty(4 * e * e + 4 * e + b * sq * e)
        gw = [grads[k * e * e:] for k in range(4)]
        gb = [grads[4 * e * e + k * e:] for k in range(4)]
        gx = grads[4 * e * e + 4 * e:]
        calls += [
            (L.wm_fill, (_p(grads), C.c_float(0), grads.numel())),
            (L.wm_mha_bwd, (_p(d["g"]), q, kv, kv, *ws, _p(Q), _p(K), _p(V), _p(attn), _p(ctx), b, sq, sk, e, h,
                            *[_p(t) for t in gw], *[_p(t) for t in gb], _p(gx), _p(gx), _p(gx))),
        ]
        out.update({"gw": grads[:4 * e * e], "gb": grads[4 * e * e:4 * e * e + 4 * e], "gx": gx})
    return calls, out, keep


def _adamw_state(case, d):
    spans, _ = _spans(case)
    keep, args = [], []
    for k in "pgmv":
        ptr, arr = W.ptr_array([d[k].data_ptr() + at * F32 for _, at in spans])
        args.append(ptr)
        keep.append(arr)
    sizes, arr = W.i64_array([n for n, _ in spans])
    keep.append(arr)
    torch.cuda.synchronize()
    return {"adamw": (W.lib().wm_adamw_step_multi, len(spans), args, sizes), "t": 0,
            "out": {"p": d["p"], "m": d["m"], "v": d["v"]}, "keep": (d, keep)}


def run(state):
    if "adamw" in state:
        step, count, args, sizes = state["adamw"]
        state["t"] += 1
        t, h = state["t"], ADAMW
        W.check(step(count, *args, sizes, h["lr"], h["beta1"], h["beta2"], h["eps"], 1.0 - h["beta1"] ** t,
                     1.0 - h["beta2"] ** t, h["weight_decay"]), "adamw")
        return state["out"]
    for fn, args in state["calls"]:
        W.check(fn(*args), fn.__name__)
    return state["out"]


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "linear":
        r, i, o = case["rows"], case["fin"], case["fout"]
        # read x, w, b, g; write y, gx, gw, gb
        return {"bytes": F32 * (2 * r * i + 2 * i * o + 2 * o + 2 * r * o), "flops": 6 * r * i * o}
    if kind == "xent":
        return {"bytes": F32 * (2 * case["rows"] * case["classes"] + case["rows"]),
                "flops": 10 * case["rows"] * case["classes"]}
    if kind == "layernorm":
        n = case["rows"] * case["n"]
        return {"bytes": F32 * (4 * n + 4 * case["n"]), "flops": 20 * n}
    if kind == "batchnorm":
        n = case["batch"] * case["channels"] * case["side"] ** 2
        return {"bytes": F32 * 4 * n, "flops": 20 * n}
    if kind == "bias":
        a, b = _bias_shapes(case)
        return {"bytes": F32 * (4 * math.prod(a) + 2 * math.prod(b)), "flops": 4 * math.prod(a)}
    if kind == "pool":
        s = case["outer"] * case["inner"]
        # read x and both upstream gradients; write both values, the index, gx
        return {"bytes": F32 * (2 * s * case["n"] + 6 * s), "flops": 3 * s * case["n"]}
    if kind == "attention":
        b, sq, sk, e, h = case["batch"], case["sq"], case["sk"], case["embed"], case["heads"]
        proj, core = 2 * b * e * e * (2 * sq + 2 * sk), 4 * b * sq * sk * e
        x = b * sq * e + (0 if case["train"] else b * sk * e)
        io = x + 4 * e * e + b * sq * e + b * h * sq * sk
        if not case["train"]:
            return {"bytes": F32 * io, "flops": proj + core}
        return {"bytes": F32 * (io + 2 * b * sq * e + 4 * e * e), "flops": 3 * (proj + core)}
    if kind == "adamw":
        n = sum(s for s, _ in _spans(case)[0])
        return {"bytes": 7 * F32 * n, "flops": 15 * n}
    n = case["rows"] * case["cols"]
    return {"bytes": 2 * 3 * n + 2 * F32 * n, "flops": 20 * n}


def tolerance(case):
    """About four times the distance from the 64-bit results that these calls
    show: products and attention 0.2-1.5e-6, a bias gradient summed in row
    order over 200704 values 5.6e-6, the other sums below 3e-7, the fp16
    result 3.4e-4 (its truncation)."""
    kind = case["kind"]
    if kind == "epilogue":
        return {"rel": 1e-3}
    if kind == "bias":
        return {"rel": 2e-5}
    if kind in ("attention", "linear"):
        return {"rel": 1e-5}
    return {"rel": 4e-6}


# ---- the same in 64 bits ----------------------------------------------------------


def exact(case, seed):
    d = {k: v.double() for k, v in _inputs(case, seed).items()}
    kind = case["kind"]
    if kind == "linear":
        return {"y": d["x"] @ d["w"] + d["b"], "gx": d["g"] @ d["w"].t().contiguous(),
                "gw": d["x"].t().contiguous() @ d["g"], "gb": d["g"].sum(0)}
    if kind == "xent":
        r = case["rows"]
        lp = torch.log_softmax(d["x"], 1)
        lab = d["labels"].long()
        gx = lp.exp()
        rows = torch.arange(r, device=gx.device)
        loss = -lp[rows, lab].sum() / r
        gx[rows, lab] -= 1.0
        return {"loss": loss.reshape(1), "gx": gx / r}
    if kind == "layernorm":
        mean = d["x"].mean(1, keepdim=True)
        inv = ((d["x"] - mean).square().mean(1, keepdim=True) + LN_EPS).rsqrt()
        xn = (d["x"] - mean) * inv
        dg = d["g"] * d["gamma"]
        gx = inv * (dg - dg.mean(1, keepdim=True) - xn * (dg * xn).mean(1, keepdim=True))
        return {"y": d["gamma"] * xn + d["beta"], "gx": gx, "ggamma": (d["g"] * xn).sum(0), "gbeta": d["g"].sum(0)}
    if kind == "batchnorm":
        x, g = d["x"], d["g"]
        mean = x.mean((0, 2), keepdim=True)
        var = (x - mean).square().mean((0, 2), keepdim=True)
        inv = (var + BN_EPS).rsqrt()
        xn = (x - mean) * inv
        gam = d["gamma"][None, :, None]
        dg = g * gam
        gx = inv * (dg - dg.mean((0, 2), keepdim=True) - xn * (dg * xn).mean((0, 2), keepdim=True))
        keep = 1.0 - BN_MOMENTUM
        return {"y": gam * xn + d["beta"][None, :, None], "gx": gx, "ggamma": (g * xn).sum((0, 2)),
                "gbeta": g.sum((0, 2)), "rm": keep * d["rm"] + BN_MOMENTUM * mean.flatten(),
                "rv": keep * d["rv"] + BN_MOMENTUM * var.flatten()}
    if kind == "bias":
        _, b = _bias_shapes(case)
        t = d["x"] + d["b"]
        gx = torch.where(t > 0, d["g"], torch.zeros_like(t))
        dims = {"channel": (0, 2, 3), "token": (1,), "row": (0,)}[case["layout"]]
        return {"y": t.clamp(min=0), "gx": gx, "gb": gx.sum(dims).reshape(b)}
    if kind == "pool":
        top, idx = d["x"].max(1)
        gx = (d["g_mean"][:, None, :]).expand_as(d["x"]).clone()
        gx.scatter_add_(1, idx[:, None, :], d["g_max"][:, None, :])
        return {"mean": d["x"].mean(1), "max": top, "index": idx, "gx": gx}
    if kind == "attention":
        return _attention_exact(case, d)
    if kind == "adamw":
        h = ADAMW
        m = h["beta1"] * d["m"] + (1.0 - h["beta1"]) * d["g"]
        v = h["beta2"] * d["v"] + (1.0 - h["beta2"]) * d["g"].square()
        step = (m / (1.0 - h["beta1"])) / ((v / (1.0 - h["beta2"])).sqrt() + h["eps"]) + h["weight_decay"] * d["p"]
        p = d["p"] - h["lr"] * step
        for n, at in _spans(case)[0]:  # the padding between tensors is left as it was
            end = at + (n + 63) // 64 * 64
            for new, old in ((p, d["p"]), (m, d["m"]), (v, d["v"])):
                new[at + n:end] = old[at + n:end]
        return {"p": p, "m": m, "v": v}
    u = (d["h"] + d["res"]) * d["gain"]
    y = torch.tanh(u.clamp(*CLAMP))
    dt = d["g"][:, None] * (1.0 - y.square()) * ((u > CLAMP[0]) & (u < CLAMP[1]))
    gh = dt * d["gain"]
    return {"y": y, "mean": y.mean(1), "gh": gh, "gres": gh, "ggain": (dt * (d["h"] + d["res"])).sum(0)}


def _attention_exact(case, d):
    b, sq, sk, e, h = case["batch"], case["sq"], case["sk"], case["embed"], case["heads"]
    hd = e // h

    def split(t, s):
        return t.reshape(b, s, h, hd).transpose(1, 2).contiguous()

    def merge(t, s):
        return t.transpose(1, 2).reshape(b, s, e).contiguous()

    def tr(t):
        return t.transpose(-1, -2).contiguous()

    Q, K, V = (split(x @ tr(d["w" + k]) + d["b" + k], s)
               for x, k, s in ((d["q"], "q", sq), (d["kv"], "k", sk), (d["kv"], "v", sk)))
    scores = Q @ tr(K) * hd ** -0.5
    if "mask" in d:
        scores = scores + d["mask"]
    attn = torch.softmax(scores, -1)
    ctx = merge(attn @ V, sq)
    out = {"y": ctx @ tr(d["wo"]) + d["bo"], "attn": attn}
    if not case["train"]:
        return out
    g, x = d["g"].reshape(-1, e), d["q"].reshape(-1, e)
    dctx = split(d["g"] @ d["wo"], sq)
    da = dctx @ tr(V)
    ds = attn * (da - (da * attn).sum(-1, keepdim=True)) * hd ** -0.5
    dq, dk, dv = (merge(t, s).reshape(-1, e) for t, s in ((ds @ K, sq), (tr(ds) @ Q, sk), (tr(attn) @ dctx, sk)))
    gw = [tr(dq) @ x, tr(dk) @ x, tr(dv) @ x, tr(g) @ ctx.reshape(-1, e)]
    gx = dv @ d["wv"] + dk @ d["wk"] + dq @ d["wq"]
    out.update({"gw": torch.cat([t.reshape(-1) for t in gw]),
                "gb": torch.cat([dq.sum(0), dk.sum(0), dv.sum(0), g.sum(0)]), "gx": gx.reshape(-1)})
    return out
