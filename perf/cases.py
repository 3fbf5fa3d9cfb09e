"""The performance cases: what programs built on this framework call, over the range of sizes they call it at.

A case is one call (or one forward + backward, or one whole-model pass) through the public entry points:
`pdum_dsl_amd.kernels` for attention, decode and the row templates, the seat `compile_tile_hip(...).run_dev` for the
planned contraction and pointwise regions, `PlanExecutor` for carved whole models. `listed()` holds one case for each
path and regime, `draw(rng)` gives further cases of the same ranges: odd sizes, grouped heads, windows, strided
layouts and the other element types.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from pdum_dsl_amd import kernels as K
from pdum_dsl_amd.executor import PlanExecutor
from pdum_dsl_amd.hip_tile import compile_tile_hip
from pdum_dsl_amd.tl import autodiff, fusion, zoo
from pdum_dsl_amd.tl.partition import plan_model

TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BYTES = {"f32": 4, "bf16": 2, "f16": 2}
FILL = -1e9


# ------------------------------------------------------------------ the cases


def _attn(kind, dtype, batch, heads, kv_heads, t, s, d, mask, window=0, layout="bhtd", **kw):
    return dict(kind=kind, dtype=dtype, batch=batch, heads=heads, kv_heads=kv_heads, t=t, s=s, d=d, mask=mask,
                window=window, layout=layout, **kw)


def _gpt2(mode, dtype, t, d, heads, mlp, layers, vocab, **kw):
    return dict(kind="gpt2", mode=mode, dtype=dtype, t=t, d=d, heads=heads, mlp=mlp, layers=layers, vocab=vocab, **kw)


def listed() -> list:
    return [
        # one attention head over a short fp32 sequence: the smallest call, where its latency counts
        _attn("attention", "f32", 1, 1, 1, 256, 256, 64, "none", name="attn_f32_1x1x256x64"),
        # a training or prefill batch's causal attention at full size: matrix-core throughput
        _attn("attention", "bf16", 8, 32, 32, 4096, 4096, 128, "causal", name="attn_bf16_8x32x4096x128"),
        # a chunk of new tokens against a cache that already holds earlier ones, grouped heads, odd lengths
        _attn("attention", "f16", 2, 32, 8, 500, 3001, 128, "causal", name="prefill_f16_2x32g8x500x3001x128"),
        # attention's forward and backward in a 16-bit training step
        _attn("attention_train", "bf16", 4, 16, 16, 2048, 2048, 64, "causal", name="train_bf16_4x16x2048x64"),
        # the same in fp32, the element type of the planned programs, gpt2-small's heads at an odd length
        _attn("attention_train", "f32", 2, 12, 12, 1000, 1000, 64, "causal", name="train_f32_2x12x1000x64"),
        # one decoding step of a large serving batch over long caches: reads 2 GiB of keys and values
        _attn("decode", "bf16", 64, 32, 8, 1, 8192, 128, "none", name="decode_bf16_64x32g8x8192x128"),
        # one decoding step of a single conversation: latency
        _attn("decode", "f16", 1, 32, 8, 1, 1500, 128, "none", name="decode_f16_1x32g8x1500x128"),
        # the row-normalization template at streaming size
        dict(kind="softmax", dtype="f32", rows=8192, cols=4096, name="softmax_f32_8192x4096"),
        # the contraction-epilogue template: gpt2-small's MLP up-projection with bias and gelu over 8192 tokens
        dict(kind="linear_gelu", dtype="bf16", t=8192, d=768, f=3072, name="linear_gelu_bf16_8192x768x3072"),
        # the stencil template: a diffusion step over a large grid
        dict(kind="stencil", dtype="f32", rows=8192, cols=8192, name="stencil_f32_8192x8192"),
        # a whole gpt2-small forward as one replayed plan
        _gpt2("forward", "bf16", 1024, 768, 12, 3072, 12, 50257, name="gpt2_forward_bf16_t1024_l12"),
        # a training step's compute: forward and every weight's gradient, gpt2-small's widths, four layers
        _gpt2("train", "f32", 1024, 768, 12, 3072, 4, 50257, name="gpt2_train_f32_t1024_l4"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_attention(rng, kind):
    dtype = rng.choice(("bf16", "bf16", "f16", "f32"))
    cap = {"attention": 1.0e12, "attention_train": 1.2e12}[kind] if dtype != "f32" else 1.6e10
    while True:
        d = rng.choice((64, 128))
        kv = rng.choice((1, 2, 4, 8, 12, 16, 32))
        group = rng.choice((1, 1, 2, 4))
        mask = rng.choice(("causal", "causal", "none", "window"))
        s = _log_int(rng, 48, 6000)
        t = s if kind == "attention_train" or rng.random() < 0.6 else _log_int(rng, 17, max(18, s))
        c = _attn(kind, dtype, _log_int(rng, 1, 8), kv * group, kv, min(t, s), s, d, mask,
                  window=_log_int(rng, 32, max(33, s)) if mask == "window" else 0,
                  layout=rng.choice(("bhtd", "bthd")) if kind == "attention" else "bhtd")
        flops = 4.0 * c["batch"] * c["heads"] * c["t"] * c["s"] * d * (3.5 if kind == "attention_train" else 1.0)
        if c["heads"] <= 64 and flops <= cap:
            return c


def _draw_decode(rng):
    while True:
        kv = rng.choice((1, 2, 4, 8, 16, 32))
        group = rng.choice((1, 2, 4, 8))
        d = rng.choice((64, 128))
        b, s = _log_int(rng, 1, 64), _log_int(rng, 100, 16000)
        if kv * group <= 64 and 4.0 * b * kv * s * d <= 2.1e9:
            return _attn("decode", rng.choice(("bf16", "f16")), b, kv * group, kv, 1, s, d, "none")


def _draw_rows(rng):
    while True:
        rows, cols = _log_int(rng, 32, 32000), _log_int(rng, 48, 8192)
        if rows * cols <= 1 << 25:
            return dict(kind=rng.choice(("softmax", "layernorm")), dtype=rng.choice(("f32", "f32", "bf16", "f16")),
                        rows=rows, cols=cols)


def _draw_linear(rng):
    dtype = rng.choice(("bf16", "bf16", "f16", "f32"))
    cap = 2e11 if dtype != "f32" else 6e10
    while True:
        t, d, f = _log_int(rng, 24, 8192), _log_int(rng, 64, 6144), _log_int(rng, 64, 8192)
        if rng.random() < 0.7:  # model widths are mostly multiples of 64
            d, f = -(-d // 64) * 64, -(-f // 64) * 64
        if 2.0 * t * d * f <= cap:
            return dict(kind="linear_gelu", dtype=dtype, t=t, d=d, f=f)


def _draw_pointwise(rng):
    kind = rng.choice(("stencil", "masked_activation"))
    rows, cols = _log_int(rng, 40, 8192), _log_int(rng, 40, 8192)
    return dict(kind=kind, dtype=rng.choice(("f32", "f32", "bf16")), rows=rows, cols=cols)


def _draw_gpt2(rng):
    mode = rng.choice(("forward", "forward", "train"))
    d, heads = rng.choice(((256, 4), (512, 8), (768, 12)))
    return _gpt2(mode, "f32" if mode == "train" else rng.choice(("bf16", "bf16", "f32")), _log_int(rng, 48, 1024), d,
                 heads, 4 * d, rng.randint(1, 4 if mode == "train" else 6), rng.choice((5003, 16384, 50257)))


def draw(rng) -> dict:
    kind = rng.choice(("attention", "attention", "attention_train", "attention_train", "decode", "decode", "rows",
                       "rows", "linear", "linear", "pointwise", "gpt2"))
    return {"attention": lambda: _draw_attention(rng, "attention"),
            "attention_train": lambda: _draw_attention(rng, "attention_train"),
            "decode": lambda: _draw_decode(rng), "rows": lambda: _draw_rows(rng),
            "linear": lambda: _draw_linear(rng), "pointwise": lambda: _draw_pointwise(rng),
            "gpt2": lambda: _draw_gpt2(rng)}[kind]()


# ------------------------------------------------------------------ inputs


class _Random:
    """Tensors of one seed, in the order asked for: rounded to the case's element type."""

    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = TORCH[dtype]

    def normal(self, *shape, std=1.0, mean=0.0):
        x = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return x.mul_(std).add_(mean).to(self.dtype)

    def index(self, n, below):
        return torch.randint(0, below, (n,), generator=self.gen, device="cuda")


def _inputs(case, seed) -> dict:
    """The values a case's call reads, by name."""
    r = _Random(seed, case["dtype"])
    kind = case["kind"]
    if kind in ("attention", "attention_train", "decode"):
        b, h, kv, t, s, d = (case[k] for k in ("batch", "heads", "kv_heads", "t", "s", "d"))
        if case["layout"] == "bthd":  # a projection's output, its heads moved forward by a view
            q, k, v = (r.normal(b, n, hh, d).transpose(1, 2) for n, hh in ((t, h), (s, kv), (s, kv)))
        else:
            q, k, v = r.normal(b, h, t, d), r.normal(b, kv, s, d), r.normal(b, kv, s, d)
        out = dict(q=q, k=k, v=v)
        if kind == "attention_train":
            out["do"] = r.normal(b, h, t, d)
        return out
    if kind == "softmax":
        return dict(x=r.normal(case["rows"], case["cols"], std=2.0))
    if kind == "layernorm":
        n = case["cols"]
        return dict(x=r.normal(case["rows"], n), gamma=r.normal(n, std=0.1, mean=1.0), beta=r.normal(n, std=0.1))
    if kind == "linear_gelu":
        t, d, f = case["t"], case["d"], case["f"]
        return dict(x=r.normal(t, d), w=r.normal(d, f, std=d**-0.5), bias=r.normal(f, std=0.1))
    if kind == "stencil":
        return dict(u=r.normal(case["rows"] + 2, case["cols"] + 2))
    if kind == "masked_activation":
        return dict(x=r.normal(case["rows"], case["cols"]), s=r.normal(case["cols"]))
    out = dict(ids=r.index(case["t"], case["vocab"]))
    for name, shape in _gpt2_plan(*_gpt2_key(case))["shapes"].items():
        if name == "ids":
            continue
        if name == "dlogits":
            out[name] = r.normal(*shape, std=1e-2)
        elif "ln" in name and name.endswith("g"):  # GPT-2's own initialization scale
            out[name] = r.normal(*shape, std=0.02, mean=1.0)
        else:
            out[name] = r.normal(*shape, std=0.01 if name == "wpe" else 0.02)
    return out


def _gpt2_key(case):
    return (case["mode"],) + tuple(case[k] for k in ("t", "d", "heads", "mlp", "layers", "vocab"))


@functools.lru_cache(maxsize=4)
def _gpt2_plan(mode, t, d, heads, mlp, layers, vocab) -> dict:
    """The model's region and its plan, which a program makes once: ``shapes`` are its params by name, in order."""
    cfg = zoo.GPT2Config(t=t, d=d, nh=heads, hk=d // heads, m=mlp, layers=layers, v=vocab)
    model = zoo.gpt2(cfg, init="gpt2")
    names = [model.names[id(p)] for p in model.region.params]
    region, order, outputs = model.region, model.order, ("logits",)
    if mode == "train":
        wrt = tuple(n for n in names if n != "ids")
        joint = autodiff.grad(region, "logits", seed="dlogits", wrt=wrt,
                              names=autodiff.region_names(region, tuple(names), ("logits",)))
        nodes = [joint.nodes[n] for n in joint.outputs]
        back = {joint.grads[w]: w for w in wrt}
        outputs = tuple(back.get(n, "logits") for n in joint.outputs)
        region, names = joint.region, names + ["dlogits"]
    else:
        nodes = [region.body[-1].args[0]]
    shapes = {n: tuple(p.type.shape) for n, p in zip(names, region.params)}
    param_dims = {n: p.type.names for n, p in zip(names, region.params)}
    # each output's dims, to lay the plain computation's values out alike
    perms = [[(order if n == "logits" else param_dims[n]).index(x) for x in y.type.names]
             for n, y in zip(outputs, nodes)]
    seed_perm = [param_dims["dlogits"].index(x) for x in order] if mode == "train" else None
    return dict(region=region, plan=plan_model(region), shapes=shapes, outputs=outputs, perms=perms,
                seed_perm=seed_perm)


# ------------------------------------------------------------------ calls


def _band(case):
    """The mask as a band of key - query: the last query sees the last key."""
    off = case["s"] - case["t"]
    if case["mask"] == "none":
        return None
    return K.Band(None, off) if case["mask"] == "causal" else K.Band(off + 1 - case["window"], off)


@functools.lru_cache(maxsize=16)
def _seat(kind, dtype, rows, cols, inner=0):
    """A planned region's runner, bound once per program."""
    if kind == "linear_gelu":
        region = zoo.linear_gelu(T=rows, D=inner, F=cols).region
    elif kind == "stencil":
        region = zoo.stencil_tile(MI=rows, NI=cols).naive
    else:
        region = zoo.masked_activation(I=rows, J=cols).region
    (group,) = fusion.plan_region(region).groups
    return compile_tile_hip(group.kernel, dtype=dtype)


def prepare(case, seed) -> dict:
    state = dict(case=case, inputs=_inputs(case, seed))
    kind = case["kind"]
    if kind == "linear_gelu":
        state["runner"] = _seat(kind, case["dtype"], case["t"], case["f"], case["d"])
    elif kind in ("stencil", "masked_activation"):
        state["runner"] = _seat(kind, case["dtype"], case["rows"], case["cols"])
    elif kind == "gpt2":
        p = _gpt2_plan(*_gpt2_key(case))
        ex = PlanExecutor(p["plan"], p["region"], case["dtype"])
        ex.bind([state["inputs"][n] for n in p["shapes"]])
        ex.capture()
        state["executor"] = ex
    else:
        state["band"] = _band(case) if "mask" in case else None
    return state


def run(state):
    case, x = state["case"], state["inputs"]
    kind = case["kind"]
    if kind == "attention":
        r = K.flash_fwd(x["q"], x["k"], x["v"], band=state["band"])
        return {"o": r.o, "lse": r.lse}
    if kind == "attention_train":
        r = K.flash_fwd(x["q"], x["k"], x["v"], band=state["band"])
        dq, dk, dv = K.flash_bwd(x["q"], x["k"], x["v"], r.o, x["do"], r.lse, band=state["band"])
        return {"o": r.o, "lse": r.lse, "dq": dq, "dk": dk, "dv": dv}
    if kind == "decode":
        o, lse = K.attn_decode(x["q"], x["k"], x["v"])
        return {"o": o, "lse": lse}
    if kind == "softmax":
        return K.row_softmax(x["x"])
    if kind == "layernorm":
        return K.layernorm(x["x"], x["gamma"], x["beta"])
    if kind == "gpt2":
        return state["executor"].replay(check=False)
    return state["runner"].run_dev(list(x.values()))


# ------------------------------------------------------------------ work and tolerance


def _live_pairs(case):
    """(query, key) pairs the mask leaves, per head."""
    t, s = case["t"], case["s"]
    if case["mask"] == "none":
        return t * s
    last = np.arange(t, dtype=np.int64) + (s - t)
    seen = last + 1 if case["mask"] == "causal" else np.minimum(last + 1, case["window"])
    return int(seen.sum())


def work(case) -> dict:
    kind, w = case["kind"], BYTES[case["dtype"]]
    if kind in ("attention", "attention_train", "decode"):
        b, h, kv, t, s, d = (case[k] for k in ("batch", "heads", "kv_heads", "t", "s", "d"))
        qo, kvs = b * h * t * d * w, 2 * b * kv * s * d * w
        flops = 4.0 * d * b * h * _live_pairs(case)
        if kind == "attention_train":  # two products forward, five backward; dO in, dQ / dK / dV out
            return {"bytes": 4 * qo + 2 * kvs + 4 * b * h * t, "flops": 3.5 * flops}
        return {"bytes": 2 * qo + kvs + 4 * b * h * t, "flops": flops}
    if kind in ("softmax", "layernorm"):
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * n * w, "flops": (4 if kind == "softmax" else 7) * n}
    if kind == "linear_gelu":
        t, d, f = case["t"], case["d"], case["f"]
        return {"bytes": (t * d + d * f + f + t * f) * w, "flops": 2.0 * t * d * f}
    if kind in ("stencil", "masked_activation"):
        n = case["rows"] * case["cols"]
        if kind == "stencil":
            return {"bytes": ((case["rows"] + 2) * (case["cols"] + 2) + n) * w, "flops": 7 * n}
        return {"bytes": 2 * n * w, "flops": 6 * n}
    t, d, m, layers, v = (case[k] for k in ("t", "d", "mlp", "layers", "vocab"))
    matrices = layers * (4 * d * d + 2 * d * m)
    flops = 2.0 * t * (matrices + d * v) + layers * 4.0 * d * (t * (t + 1) // 2)
    weights = matrices + v * d + t * d
    if case["mode"] == "train":  # the backward takes two products for each one forward (five for attention's two)
        back = 4.0 * t * (matrices + d * v) + layers * 10.0 * d * (t * (t + 1) // 2)
        return {"bytes": (2 * weights + 2 * t * v) * w, "flops": flops + back}
    return {"bytes": (weights + t * v) * w, "flops": flops}


def tolerance(case) -> dict:
    """About four times the distance to the 64-bit values seen over the ranges (`exact`): one rounding of the result
    and of the probabilities at 16 bits (2.6e-3 bf16, 3.1e-4 f16), sums of up to some thousand terms in 32 (8e-7, up
    to 3e-6 through a model's gradients), and a 12-layer model's roundings in turn (9e-3 bf16)."""
    if case["kind"] == "gpt2" and case["dtype"] != "f32":
        return {"rel": 3e-2}
    return {"rel": {"f32": 1.2e-5, "bf16": 1e-2, "f16": 1.3e-3}[case["dtype"]]}


# ------------------------------------------------------------------ the same in 64 bits


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(0.7978845608028654 * (z + 0.044715 * z**3)))


def _exact_attention(case, x):
    b, h, kv, t, s, d = (case[k] for k in ("batch", "heads", "kv_heads", "t", "s", "d"))
    scale = d**-0.5
    band = _band(case)
    live = None
    if band is not None:
        rel = torch.arange(s, device="cuda")[None, :] - torch.arange(t, device="cuda")[:, None]
        live = rel <= band.hi
        if band.lo is not None:
            live &= rel >= band.lo
    train = case["kind"] == "attention_train"
    new = lambda *shape: torch.empty(shape, dtype=torch.float64, device="cuda")  # noqa: E731
    out = {"o": new(b, h, t, d), "lse": new(b, h, t)}
    if train:
        out.update(dq=new(b, h, t, d), dk=new(b, kv, s, d), dv=new(b, kv, s, d))
    for i in range(b):
        for j in range(kv):
            hs = slice(j * (h // kv), (j + 1) * (h // kv))
            k, v = x["k"][i, j].double().contiguous(), x["v"][i, j].double().contiguous()
            q = x["q"][i, hs].double().contiguous()
            sc = (q @ k.t().contiguous()) * scale
            if live is not None:
                sc = torch.where(live, sc, torch.full_like(sc, FILL))
            lse = torch.logsumexp(sc, dim=-1)
            p = torch.exp(sc - lse[..., None])
            o = p @ v
            out["o"][i, hs], out["lse"][i, hs] = o, lse
            if train:
                do = x["do"][i, hs].double()
                ds = p * (do @ v.t().contiguous() - (do * o).sum(-1, keepdim=True))
                if live is not None:
                    ds = torch.where(live, ds, torch.zeros_like(ds))
                flat = lambda z: z.reshape(-1, z.shape[-1])  # noqa: E731
                out["dq"][i, hs] = (ds @ k) * scale
                out["dk"][i, j] = (flat(ds).t().contiguous() @ flat(q)) * scale
                out["dv"][i, j] = flat(p).t().contiguous() @ flat(do)
    return out


def _exact_gpt2(case, x):
    plan = _gpt2_plan(*_gpt2_key(case))
    train = case["mode"] == "train"
    w = {n: v if n == "ids" else v.double().requires_grad_(train and n != "dlogits") for n, v in x.items()}
    t, d, nh = case["t"], case["d"], case["heads"]
    hk = d // nh
    norm = torch.nn.functional.layer_norm
    mask = torch.ones((t, t), dtype=torch.bool, device="cuda").tril()
    with torch.set_grad_enabled(train):
        h = w["wte"][w["ids"]] + w["wpe"]
        for i in range(case["layers"]):
            a, m = f"h.{i}.attn.", f"h.{i}.mlp."
            y = norm(h, (d,), w[a + "ln1g"], w[a + "ln1b"], eps=1e-5)
            q, k, v = ((y @ w[a + n].reshape(d, d)).view(t, nh, hk).transpose(0, 1).contiguous()
                       for n in ("wq", "wk", "wv"))
            sc = (q @ k.transpose(1, 2).contiguous()) * hk**-0.5
            p = torch.softmax(torch.where(mask, sc, torch.full_like(sc, FILL)), dim=-1)
            h = h + (p @ v).transpose(0, 1).reshape(t, d) @ w[a + "wo"].reshape(d, d)
            y = norm(h, (d,), w[m + "ln2g"], w[m + "ln2b"], eps=1e-5)
            h = h + _gelu(y @ w[m + "w1"] + w[m + "b1"]) @ w[m + "w2"] + w[m + "b2"]
        logits = norm(h, (d,), w["lnfg"], w["lnfb"], eps=1e-5) @ w["wte"].t().contiguous()
    if not train:
        return logits.permute(plan["perms"][0])
    wrt = [n for n in plan["outputs"] if n != "logits"]
    grads = torch.autograd.grad(logits, [w[n] for n in wrt], w["dlogits"].permute(plan["seed_perm"]))
    got = dict(zip(wrt, grads), logits=logits.detach())
    return tuple(got[n].permute(p) for n, p in zip(plan["outputs"], plan["perms"]))


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("attention", "attention_train", "decode"):
        return _exact_attention(case, x)
    if kind == "gpt2":
        return _exact_gpt2(case, x)
    x = {n: v.double() for n, v in x.items()}
    if kind == "softmax":
        return torch.softmax(x["x"], dim=-1)
    if kind == "layernorm":
        return torch.nn.functional.layer_norm(x["x"], (case["cols"],), x["gamma"], x["beta"], eps=1e-5)
    if kind == "linear_gelu":
        return _gelu(x["x"] @ x["w"] + x["bias"])
    if kind == "stencil":
        u = x["u"]
        mid = u[1:-1, 1:-1]
        return mid + 0.1 * (u[:-2, 1:-1] + u[2:, 1:-1] + u[1:-1, :-2] + u[1:-1, 2:] - 4.0 * mid)
    i = torch.arange(case["rows"], device="cuda")[:, None]
    j = torch.arange(case["cols"], device="cuda")[None, :]
    y = torch.tanh(x["x"] * x["s"]) + torch.exp(-x["x"].abs())
    return torch.where(j > i, y, torch.zeros_like(y))
