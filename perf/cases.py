"""The work that a program using this framework has it do, as measurable cases.

Four kinds of call, each through the Python binding's public entry points:

- ``layer``: one MoE layer of a decode step with every expert resident --
  ``router_topk`` and then ``indexed_moe_fused_decode``;
- ``prefill``: one MoE layer of a prompt chunk -- ``router_topk`` (the routed
  experts' columns of the table) and then ``moe_prefill``, with always-on shared
  experts and the residual where the model has them;
- ``stack``: a whole decode step through a stack of layers (``stack_decode``);
- ``cached``: decode steps through layers whose expert cache holds a part of the
  experts, the misses uploaded from pinned host memory
  (``CachedLayer.stack_forward``).

Activations are N(0, 1), weights N(0, 0.02) quantised to GGUF blocks, routers
N(0, 0.02) in f32: what the benchmark and the tests use.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "naiwa-rs_amd"))
import naiwa_moe as nm  # noqa: E402

DEV = "cuda"
DTYPES = {"q4_k": nm.Q4_K, "q8_0": nm.Q8_0}
BLOCK = {"q4_k": (256, 144), "q8_0": (32, 34)}
MODES = {"softmax_topk_renorm": nm.ROUTE_SOFTMAX_TOPK_RENORM, "topk_softmax": nm.ROUTE_TOPK_SOFTMAX,
         "softmax_topk": nm.ROUTE_SOFTMAX_TOPK}
ACTS = {"silu": nm.ACT_SILU, "gelu": nm.ACT_GELU_PYTORCH_TANH}

# Shapes that the repository's configurations and benchmark name: hidden, intermediate, experts, top-k,
# gate/up and down formats, router mode, shared experts.
SHAPES = {
    "small": dict(hidden=1024, inter=2048, experts=8, topk=2, gate="q8_0", down="q8_0", mode="topk_softmax", shared=0),
    "qwen3": dict(hidden=2048, inter=768, experts=128, topk=8, gate="q4_k", down="q4_k", mode="softmax_topk_renorm",
                  shared=0),
    "deepseek": dict(hidden=2048, inter=1408, experts=64, topk=6, gate="q4_k", down="q8_0", mode="softmax_topk",
                     shared=2),
    "mixtral": dict(hidden=4096, inter=14336, experts=8, topk=2, gate="q4_k", down="q4_k", mode="topk_softmax",
                    shared=0),
}


def _case(name, kind, shape, rows, **more):
    c = dict(name=name, kind=kind, rows=rows, layers=1, act="silu", x="bf16", residual=False, accumulate=False)
    c.update(SHAPES[shape])
    c.update(more)
    return c


def listed():
    return [
        # the smallest call: one token through a small 8-expert layer, where launches and latency count
        _case("small_layer_1row", "layer", "small", 1),
        # single-user decode: the whole 48-layer step of one token, all experts resident
        _case("qwen3_step_1row", "stack", "qwen3", 1, layers=48),
        # small-batch serving: one layer, 8 rows, about 50 of the 128 experts touched
        _case("qwen3_layer_8rows", "layer", "qwen3", 8),
        # continuous batching: one layer at 96 concurrent sequences, every expert touched by a few rows
        _case("qwen3_layer_96rows", "layer", "qwen3", 96),
        # an odd batch of a model with mixed formats, f32 activations as a host engine hands them over
        _case("deepseek_layer_5rows", "layer", "deepseek", 5, x="f32"),
        # single-user decode of a model with few large experts
        _case("mixtral_layer_1row", "layer", "mixtral", 1),
        # the same at a serving batch: every expert read once for a few rows
        _case("mixtral_layer_16rows", "layer", "mixtral", 16),
        # the same at a large serving batch
        _case("mixtral_layer_64rows", "layer", "mixtral", 64),
        # a 512-token prompt chunk of a model with fine-grained and shared experts, residual added in place
        _case("deepseek_prefill_512", "prefill", "deepseek", 512, residual=True),
        # a whole prompt of odd length in one call
        _case("qwen3_prefill_1999", "prefill", "qwen3", 1999),
        # a long prompt through few large experts
        _case("mixtral_prefill_4096", "prefill", "mixtral", 4096),
        # decode with a quarter of the experts cached: misses travel over PCIe
        _case("qwen3_cached_4layers", "cached", "qwen3", 1, layers=4, usable=32, steps=8),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["layer", "prefill", "stack", "cached"], [5, 4, 2, 1])[0]
    c = dict(kind=kind, layers=1, act="silu", x="bf16", residual=False, accumulate=False, shared=0)
    if kind == "stack":
        c.update(SHAPES["qwen3"])
        c["rows"] = rng.choice([1, 1, 2, 3, 4, 5, 6, 8, 11])
        c["layers"] = rng.randint(3, 40)
        return c
    if kind == "cached":
        c.update(SHAPES["qwen3"])
        c.update(rows=1, layers=rng.randint(1, 4), usable=rng.randint(24, 96), steps=rng.randint(2, 8))
        return c
    c["gate"] = rng.choice(["q4_k", "q4_k", "q8_0"])
    c["down"] = rng.choice(["q4_k", "q8_0"])
    c["mode"] = rng.choice(sorted(MODES))
    c["act"] = rng.choice(["silu", "silu", "gelu"])
    if rng.random() < 0.25:  # few large experts
        c.update(hidden=4096, inter=256 * rng.randint(24, 56), experts=8, topk=2)
    else:  # many small ones; odd block counts among them
        c.update(hidden=256 * rng.randint(4, 20), experts=rng.choice([8, 16, 32, 60, 64, 128]), topk=rng.randint(1, 8))
        c["inter"] = 256 * rng.randint(2, 8) if c["down"] == "q4_k" else 128 * rng.randint(4, 17)
    c["shared"] = rng.choice([0, 0, 0, 1, 2])
    if kind == "layer":
        c["rows"] = _log_uniform(rng, 1, 256)
        c["x"] = rng.choice(["bf16", "bf16", "f32"])
        c["accumulate"] = rng.random() < 0.2
        return c
    c["residual"] = rng.random() < 0.5
    # at most the largest listed case's products, and the table's 65,536 pairs
    top = 4096 * 2 * 4096 * 14336 // ((c["topk"] + c["shared"]) * c["hidden"] * c["inter"])
    c["rows"] = _log_uniform(rng, 48, max(64, min(4096, top, 65536 // (c["topk"] + c["shared"]))))
    return c


# ---- what a program has in hand -----------------------------------------------------------


def _row_bytes(fmt, k):
    bs, ts = BLOCK[fmt]
    return k // bs * ts


def _down_std(case):
    # a chain of layers stays of the scale of its input, as the benchmark's chains do
    return 0.02 if case["inter"] <= 1024 else 0.004 if case["inter"] <= 2048 else 0.0015


def _fill(bank, fmt, seed, std):
    """Every slot of a bank with quantised N(0, std) weights."""
    bs, ts = BLOCK[fmt]
    n = bank.expert_bytes // ts * bs
    if bank.stride == bank.expert_bytes:
        nm.synth(DTYPES[fmt], seed, n * bank.slots, bank.base, 0.0, std)
    else:
        for s in range(bank.slots):
            nm.synth(DTYPES[fmt], seed, n, bank.slot_ptr(s), 0.0, std, offset=s * n)


def _layer(case, seed):
    slots = case["experts"] + case["shared"]
    banks = nm.LayerBanks(slots, case["hidden"], case["inter"],
                          (DTYPES[case["gate"]], DTYPES[case["gate"]], DTYPES[case["down"]]))
    _fill(banks.gate, case["gate"], seed, 0.02)
    _fill(banks.up, case["gate"], seed + 1, 0.02)
    _fill(banks.down, case["down"], seed + 2, _down_std(case))
    router = torch.empty(case["experts"], case["hidden"], device=DEV)
    nm.synth(nm.F32, seed + 3, router.numel(), router.data_ptr(), 0.0, 0.02)
    return banks, router


def _rows(case, seed, rows):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(rows, case["hidden"], device=DEV, generator=g)
    return x if case["x"] == "f32" else x.bfloat16()


def prepare(case, seed):
    seed = 7919 * (seed + 1)
    s = {"case": case}
    T, H = case["rows"], case["hidden"]
    if case["kind"] == "cached":
        return _prepare_cached(case, seed, s)
    layers = [_layer(case, seed * 512 + 8 * l) for l in range(case["layers"])]
    s["banks"], s["routers"] = [b for b, _ in layers], [r for _, r in layers]
    s["x0"] = _rows(case, seed, T)
    s["x"] = s["x0"].clone()
    if case["kind"] == "stack":
        s["descs"] = (nm._lib.Layer * len(layers))(*[nm.layer_desc(r.data_ptr(), b) for b, r in layers])
        s["y"] = torch.zeros(case["layers"], T, H, device=DEV)
        return s
    width = case["topk"] + case["shared"]
    s["ids"] = torch.zeros(T, width, dtype=torch.int32, device=DEV)
    s["w"] = torch.ones(T, width, device=DEV)
    s["ids"][:, case["topk"]:] = torch.arange(case["experts"], case["experts"] + case["shared"], device=DEV)
    s["out"] = torch.zeros(T, H, device=DEV)
    s["out0"] = 0.1 * _rows(dict(case, x="f32"), seed + 1, T) if case["accumulate"] else None
    return s


def _prepare_cached(case, seed, s):
    L, H, E, K, I, usable = (case[k] for k in ("layers", "hidden", "experts", "topk", "inter", "usable"))
    dt = (DTYPES[case["gate"]], DTYPES[case["gate"]], DTYPES[case["down"]])
    s["compute"], s["copy"] = 0, nm.Stream()
    s["ring"] = nm.policy.StagingRing()
    s["stacks"], s["banks"], s["routers"], s["bias"], s["layers"] = [], [], [], [], []
    for l in range(L):
        full, router = _layer(dict(case, shared=0), seed * 512 + 8 * l)
        stacks = nm.HostExpertStacks(E, H, I, dt, interleaved=True)
        for p, bank in enumerate((full.gate, full.up, full.down)):
            nm._lib.check(nm.lib().naiwa_memcpy_2d(stacks.ptrs[p], stacks.stride, bank.base, bank.stride,
                                                   bank.expert_bytes, E, 0), "memcpy_2d")
        nm.synchronize()
        # expert popularity Zipf(1.1) over a random ranking, and the most popular ones cached at the start
        ranks = np.random.default_rng(seed + l).permutation(E) + 1
        p = ranks.astype(np.float64) ** -1.1
        bias = torch.from_numpy(np.log(p / p.sum()).astype(np.float32)).to(DEV)
        banks = nm.LayerBanks(usable + s["ring"].length, H, I, dt, contiguous=True)
        layer = nm.policy.CachedLayer(router.data_ptr(), banks, stacks, E, K, usable, s["ring"], s["copy"].handle,
                                      mode=MODES[case["mode"]], router_bias=bias.data_ptr())
        layer.seed([int(e) for e in np.argsort(ranks)])
        for key, v in (("stacks", stacks), ("banks", banks), ("routers", router), ("bias", bias), ("layers", layer)):
            s[key].append(v)
    s["tokens"] = _rows(case, seed, 64)
    s["out"] = torch.zeros(case["steps"], case["rows"], H, dtype=torch.bfloat16, device=DEV)
    s["y"] = torch.zeros(case["rows"], H, device=DEV)
    s["at"] = 0
    return s


# ---- one pass -----------------------------------------------------------------------------


def run(s):
    case = s["case"]
    T, H, E, K = case["rows"], case["hidden"], case["experts"], case["topk"]
    mode, act = MODES[case["mode"]], ACTS[case["act"]]
    if case["kind"] == "stack":
        s["x"].copy_(s["x0"])
        # the fused kernel serves up to 4 rows, the layered chain more: the benchmark's choice
        nm.stack_decode(s["descs"], s["x"].data_ptr(), T, H, E, K, mode=mode, act=act, fused=T <= 4,
                        y_out=s["y"].data_ptr())
        return {"x": s["x"], "y": s["y"]}
    if case["kind"] == "cached":
        for i in range(case["steps"]):
            x = s["out"][i]
            x.copy_(s["tokens"][s["at"] % 64])
            s["at"] += 1
            nm.policy.CachedLayer.stack_forward(s["layers"], x.data_ptr(), T, s["y"].data_ptr(),
                                                stream=s["compute"])
        return {"x": s["out"], "y": s["y"]}
    x, xdt = s["x"], nm.F32 if case["x"] == "f32" else nm.BF16
    ids, w, out = s["ids"].data_ptr(), s["w"].data_ptr(), s["out"].data_ptr()
    if case["kind"] == "layer":
        # always-on experts take the columns behind the routed ones, at weight 1
        width = K + case["shared"]
        nm.router_topk(x.data_ptr(), xdt, s["routers"][0].data_ptr(), T, H, E, K, ids, w, mode=mode,
                       ld=width if case["shared"] else 0)
        if case["accumulate"]:
            s["out"].copy_(s["out0"])
        nm.indexed_moe_fused_decode(s["banks"][0], x.data_ptr(), xdt, ids, w, T, width, out, act=act,
                                    accumulate=case["accumulate"])
        return {"ids": s["ids"], "w": s["w"], "out": s["out"]}
    width = K + case["shared"]
    if case["residual"]:
        x.copy_(s["x0"])
    nm.router_topk(x.data_ptr(), xdt, s["routers"][0].data_ptr(), T, H, E, K, ids, w, mode=mode, ld=width)
    nm.moe_prefill(s["banks"][0], x.data_ptr(), ids, w, T, width, out, act=act, residual=case["residual"])
    got = {"ids": s["ids"], "w": s["w"], "out": s["out"]}
    if case["residual"]:
        got["x"] = x
    return got


# ---- what a pass cannot do without ----------------------------------------------------------


def work(case):
    T, H, I, E, K, L = (case[k] for k in ("rows", "hidden", "inter", "experts", "topk", "layers"))
    width = K + case["shared"]
    expert = 2 * I * _row_bytes(case["gate"], H) + H * _row_bytes(case["down"], I)
    touched = E * (1.0 - (1.0 - K / E) ** T) + case["shared"]  # distinct experts of T uniform draws
    xb = 4 if case["x"] == "f32" else 2
    layer = {"bytes": touched * expert + E * H * 4 + T * H * (xb + 4) + T * width * 8,
             "flops": 6.0 * T * width * H * I + 2.0 * T * H * E}
    times = L * case.get("steps", 1)
    return {k: v * times for k, v in layer.items()}


# ---- tolerance and the 64-bit results ---------------------------------------------------------


def tolerance(case):
    # 16-bit activations, intermediate values and (on the matrix cores) weights: single layers measure up to
    # 3.4e-3 from the 64-bit result; ids are exact
    if case["kind"] in ("layer", "prefill"):
        return {"rel": 0.013, "max": 0.3}
    # a chain stores bf16 activations after each layer, and a change of rounding can flip an expert near the
    # cut of the top-k
    return {"rel": 0.03, "max": 0.9}


def _dequant(fmt, raw, n, k):
    """[n, k] f64 weights of GGUF blocks."""
    bs, ts = BLOCK[fmt]
    b = raw.view(n, k // bs, ts)
    if fmt == "q8_0":
        d = b[..., :2].contiguous().view(torch.float16).double()
        return (b[..., 2:].contiguous().view(torch.int8).double() * d).view(n, k)
    d = b[..., 0:2].contiguous().view(torch.float16).double()
    dmin = b[..., 2:4].contiguous().view(torch.float16).double()
    s = b[..., 4:16].int()
    lo, mid, hi = s[..., 0:4], s[..., 4:8], s[..., 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1).double()
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], -1).double()
    q = b[..., 16:].int().view(n, k // bs, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 3).view(n, k // bs, 8, 32).double()
    return ((d * sc)[..., None] * q - (dmin * mn)[..., None]).view(n, k)


def _expert(raw, fmt, n, k):
    """raw: (device or host pointer) of one expert's projection."""
    t = torch.empty(n * _row_bytes(fmt, k), dtype=torch.uint8, device=DEV)
    nm._lib.check(nm.lib().naiwa_memcpy_2d(t.data_ptr(), t.numel(), raw, t.numel(), t.numel(), 1, 0), "copy")
    nm.synchronize()
    return _dequant(fmt, t, n, k)


def _route(case, x, router, bias):
    logits = x @ router.double().T
    if bias is not None:
        logits = logits + bias.double()
    top, ids = torch.sort(logits, dim=-1, descending=True, stable=True)
    top, ids = top[:, :case["topk"]], ids[:, :case["topk"]]
    if case["mode"] == "softmax_topk":
        return ids, torch.gather(torch.softmax(logits, -1), 1, ids)
    return ids, torch.softmax(top, -1)  # renormalised or taken over the top-k: the same numbers


def _experts(case, x, ids, w, pointers):
    act = torch.nn.functional.silu if case["act"] == "silu" else lambda v: torch.nn.functional.gelu(
        v, approximate="tanh")
    out = torch.zeros_like(x)
    H, I = case["hidden"], case["inter"]
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        g, u, d = pointers(e)
        xe = x[t]
        h = act(xe @ _expert(g, case["gate"], I, H).T) * (xe @ _expert(u, case["gate"], I, H).T)
        out.index_add_(0, t, (h @ _expert(d, case["down"], H, I).T) * w[t, j][:, None])
    return out


def exact(case, seed):
    if case["kind"] in ("stack", "cached") and case["layers"] > 4:
        return None  # one flipped expert changes all that follows: no single right answer to compare with
    s = prepare(case, seed)
    if case["kind"] in ("layer", "prefill"):
        b = s["banks"][0]
        x = s["x0"].double()
        ids, w = _route(case, x, s["routers"][0], None)
        ids = torch.cat([ids, s["ids"][:, case["topk"]:].long()], 1)
        w = torch.cat([w, torch.ones_like(w[:, :1]).expand(-1, case["shared"])], 1)
        out = _experts(case, x, ids, w, lambda e: (b.gate.slot_ptr(e), b.up.slot_ptr(e), b.down.slot_ptr(e)))
        if s.get("out0") is not None:
            out = out + s["out0"].double()
        got = {"ids": None, "w": w, "out": out}
        if case["residual"]:
            got["x"] = x + out
        return got
    if case["kind"] == "stack":
        banks = s["banks"]
        where = [lambda e, b=b: (b.gate.slot_ptr(e), b.up.slot_ptr(e), b.down.slot_ptr(e)) for b in banks]
        return _chain(case, s["x0"].double(), s["routers"], [None] * len(banks), where)
    where = [st.expert_ptrs for st in s["stacks"]]
    steps = [_chain(case, s["tokens"][i:i + 1].double(), s["routers"], s["bias"], where) for i in range(case["steps"])]
    return {"x": torch.stack([r["x"] for r in steps]), "y": steps[-1]["y"][-1]}


def _chain(case, x, routers, biases, where):
    ys = []
    for router, bias, pointers in zip(routers, biases, where):
        ids, w = _route(case, x, router, bias)
        ys.append(_experts(case, x, ids, w, pointers))
        x = (x + ys[-1]).bfloat16().double()  # the activations are stored as bf16 after each layer
    return {"x": x, "y": torch.stack(ys)}
