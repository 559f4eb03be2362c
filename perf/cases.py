"""Performance cases of the quantized-matmul path: the calls a host of this library makes, over the range of sizes it makes
them at, each through the public Python binding (which is a thin layer over the C ABI).

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a host has in hand before the call: resident weights, activations, a captured graph
    run(state)           one pass of the call(s); returns its outputs
    work(case)           bytes and operations that a pass cannot do without
    tolerance(case)      how far another correct implementation may be away

Kinds of case:
    rows        `gemv_dev` over `layers` resident weights: activations on the device, m rows each (1: a decode step's
                projections; 2..32: the rows of a speculative-verify step or of a short chunk)
    trait_gemv  one host-pointer `gemv` / `gemv_f32`, what a CPU forward calls per weight through the accelerator trait
    trait_batch one host-pointer `gemv_batch`: the q/k/v or gate/up group of a decode step
    trait_moe   one host-pointer `moe_ffn`: the routed experts of one token
    decode      one token through the FFN half of a decoder stack as ONE captured graph, routed on the device
    lm_head     host-pointer `lm_head_argmax_rows` over a vocabulary-sized weight (greedy pick of a decode or verify step)
    gemm        one prefill projection with the activations on the device
    ffn         the dense FFN of a prefill chunk: norm + gate, norm + up, SwiGLU + down
    moe_layer   the routed experts of a prefill chunk, grouped by expert (host buffers or device buffers)
    trait_gemm  one host-pointer `prefill_q8_gemm`: activations in from and results out to host memory

Weights are random blocks in the GGUF formats (ty: 2 = Q4_0, 8 = Q8_0, 14 = Q6_K), activations N(0, 1), expert popularity
Zipf(1.1), as in the benchmark.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

Q4_0, Q8_0, Q6_K = 2, 8, 14
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q6_K: (256, 210)}   # elements, bytes
EPS = 1e-6


def _load(name, *path):
    if name not in sys.modules:
        file = os.path.join(os.getcwd(), "strix.rs_amd", *path)
        is_pkg = path == ("__init__.py",)
        spec = importlib.util.spec_from_file_location(name, file, submodule_search_locations=[os.path.dirname(file)] if is_pkg else None)
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ---- the cases

def listed():
    return [
        # the smallest call of a decode step: one token's router logits (64 experts) or a small projection, alone
        {"name": "router_logits", "kind": "rows", "ty": Q8_0, "m": 1, "n": 64, "k": 2048, "layers": 1},
        # one weight of a CPU forward through the trait, in the arithmetic the trait binding uses by default
        {"name": "trait_gemv", "kind": "trait_gemv", "ty": Q4_0, "n": 9728, "k": 2560, "f32": True},
        # q, k and v of a decode step with grouped key/value heads, one host call
        {"name": "trait_qkv", "kind": "trait_batch", "ty": Q8_0, "n": 2560, "n2": 640, "k": 2560, "items": 3, "f32": True},
        # one token's routed experts through the trait
        {"name": "trait_moe_token", "kind": "trait_moe", "ty": Q8_0, "ne": 64, "hidden": 2048, "eff": 768, "top": 8},
        # the latency of a decode token: 20 dependent launches over 274 MB of weights, replayed from one graph
        {"name": "decode_token", "kind": "decode", "ty": Q4_0, "ety": Q8_0, "layers": 4, "hidden": 2048, "ffn": 8192, "ne": 64,
         "eff": 768, "top": 8},
        # a speculative-verify step of 6 rows through the down projections of ten layers
        {"name": "verify_rows", "kind": "rows", "ty": Q8_0, "m": 6, "n": 2560, "k": 9728, "layers": 10},
        # greedy pick for three verified positions over a large vocabulary
        {"name": "lm_head_pick", "kind": "lm_head", "ty": Q6_K, "m": 3, "n": 262144, "k": 3840},
        # a ragged prompt tail against a long-K projection
        {"name": "gemm_q4_ragged", "kind": "gemm", "ty": Q4_0, "m": 333, "n": 2560, "k": 9728},
        # a prompt chunk against a Q6_K up projection
        {"name": "gemm_q6", "kind": "gemm", "ty": Q6_K, "m": 1000, "n": 15360, "k": 3840},
        # the dense FFN of a full 2048-token prefill chunk: the largest work
        {"name": "ffn_prefill", "kind": "ffn", "ty": Q8_0, "m": 2048, "hidden": 3840, "ffn": 15360},
        # the routed experts of a 512-token prefill chunk, activations resident
        {"name": "moe_prefill", "kind": "moe_layer", "ty": Q8_0, "m": 512, "ne": 64, "hidden": 2048, "eff": 768, "top": 8, "host": False},
        # a prefill projection called through the trait with host buffers
        {"name": "trait_prefill", "kind": "trait_gemm", "ty": Q8_0, "m": 1024, "n": 9728, "k": 2560},
    ]


KINDS = ("rows", "trait_gemv", "trait_batch", "trait_moe", "decode", "lm_head", "gemm", "ffn", "moe_layer", "trait_gemm")


def _log(rng, lo, hi, step=1):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    """A case of the same ranges: dimensions spread over their logarithm, ragged row counts among them."""
    kind = rng.choice(KINDS)
    ty = rng.choice((Q4_0, Q8_0, Q6_K))
    be = BLOCK[ty][0]
    for _ in range(1000):
        if kind == "rows":
            c = {"ty": ty, "m": _log(rng, 1, 32), "n": _log(rng, 64, 16384), "k": _log(rng, 512, 16384, be), "layers": rng.randint(1, 12)}
            if c["n"] * c["k"] * c["layers"] <= 250e6:
                break
        elif kind == "trait_gemv":
            c = {"ty": ty, "n": _log(rng, 64, 16384), "k": _log(rng, 512, 16384, be), "f32": rng.random() < 0.7}
            if c["n"] * c["k"] <= 60e6:
                break
        elif kind == "trait_batch":
            c = {"ty": ty, "n": _log(rng, 256, 8192), "n2": _log(rng, 128, 2048), "k": _log(rng, 512, 8192, be), "items": rng.randint(2, 8),
                 "f32": rng.random() < 0.7}
            if c["n"] * c["k"] <= 30e6:
                break
        elif kind in ("trait_moe", "decode", "moe_layer"):
            ty = rng.choice((Q8_0, Q6_K))
            step = 256 if ty == Q6_K else 32
            c = {"ty": ty, "ne": rng.randint(8, 64), "hidden": _log(rng, 512, 4096, 256), "eff": _log(rng, 256, 1536, step), "top": rng.randint(1, 8)}
            if kind == "decode":
                c.update(ty=rng.choice((Q4_0, Q8_0, Q6_K)), ety=ty, layers=rng.randint(1, 4), ffn=_log(rng, 1024, 12288, 256))
                if c["hidden"] * c["ffn"] > 20e6:
                    continue
            if kind == "moe_layer":
                c.update(m=_log(rng, 8, 640), host=rng.random() < 0.5)
            if c["ne"] * c["hidden"] * c["eff"] <= 101e6:
                break
        elif kind == "lm_head":
            c = {"ty": ty, "m": rng.randint(1, 8), "n": _log(rng, 30000, 262144), "k": _log(rng, 512, 3840, be)}
            if c["n"] * c["k"] <= 600e6:
                break
        elif kind == "gemm":
            c = {"ty": ty, "m": _log(rng, 17, 2048), "n": _log(rng, 512, 15360, 16), "k": _log(rng, 512, 15360, be)}
            if c["n"] * c["k"] <= 60e6 and c["m"] * c["n"] * c["k"] <= 130e9:
                break
        elif kind == "ffn":
            c = {"ty": ty, "m": _log(rng, 33, 2048), "hidden": _log(rng, 1024, 4096, 256), "ffn": _log(rng, 2048, 15360, 256)}
            if c["m"] * c["hidden"] * c["ffn"] <= 80e9:
                break
        else:
            c = {"ty": ty, "m": _log(rng, 33, 1024), "n": _log(rng, 512, 15360, 16), "k": _log(rng, 512, 15360, be)}
            if c["n"] * c["k"] <= 60e6 and c["m"] * (c["n"] + c["k"]) <= 12e6:
                break
    c["kind"] = kind
    return c


# ---- what a host has in hand before the call

_ACC = []
_FREE_LAYERS = []
_NEXT = [0, 0]   # weight keys, expert layer numbers


def _acc():
    """The process's one accelerator context (a host keeps one per device)."""
    if not _ACC:
        _ACC.append(_load("strix_rs_amd", "__init__.py").Mi355WeightAccel(0))
    return _ACC[0]


class State:
    """One case's resident weights and buffers; gives them back when it goes away."""

    def __init__(self, case):
        self.case, self.keys, self.layers, self.graph = case, [], [], None

    def weight(self, ty, n, k, gen):
        key = f"perf.w{_NEXT[0]}"
        _NEXT[0] += 1
        acc = _acc()
        assert {Q4_0: acc.upload_q4_0, Q8_0: acc.upload_q8_0, Q6_K: acc.upload_q6_k}[ty](key, _blocks(ty, n, k, gen), k, n)
        self.keys.append(key)
        return key

    def experts(self, ty, tensors, hidden, eff, ne):
        if _FREE_LAYERS:
            layer = _FREE_LAYERS.pop()
        else:
            layer, _NEXT[1] = _NEXT[1], _NEXT[1] + 1
        acc = _acc()
        assert (acc.upload_moe_q6 if ty == Q6_K else acc.upload_moe_q8)(layer, *tensors, hidden, eff, ne)
        self.layers.append(layer)
        return layer

    def __del__(self):
        try:
            if self.graph is not None:
                _acc().graph_destroy(self.graph)
            for key in self.keys:
                _acc().evict(key)
            _FREE_LAYERS.extend(self.layers)   # the next upload under this number takes the memory back
        except Exception:   # the interpreter is going away
            pass


def _blocks(ty, n, k, gen):
    """n rows of k elements as raw GGUF blocks in host memory: uniform quants, f16 block scales (made on the GPU, which is quick)."""
    be, bb = BLOCK[ty]
    nb = n * (k // be)
    lo, hi = (1e-4, 2e-3) if ty == Q6_K else (1e-3, 2e-2)
    d = (torch.rand(nb, device="cuda", generator=gen) * (hi - lo) + lo).half().view(torch.uint8).view(nb, 2)
    if ty == Q8_0:
        q = torch.randint(-127, 128, (nb, 32), dtype=torch.int8, device="cuda", generator=gen).view(torch.uint8)
        raw = torch.cat([d, q], 1)
    elif ty == Q4_0:
        raw = torch.cat([d, torch.randint(0, 256, (nb, 16), dtype=torch.uint8, device="cuda", generator=gen)], 1)
    else:
        q = torch.randint(0, 256, (nb, 192), dtype=torch.uint8, device="cuda", generator=gen)
        sc = torch.randint(-64, 64, (nb, 16), dtype=torch.int8, device="cuda", generator=gen).view(torch.uint8)
        raw = torch.cat([q, sc, d], 1)
    assert raw.shape[1] == bb
    return raw.reshape(-1).cpu().numpy()


def _acts(gen, *shape):
    return torch.randn(*shape, device="cuda", generator=gen)


def _routing(c, seed):
    synth = _load("strix_rs_amd_synth", "synth.py")
    return synth.zipf_routing(c.get("m", 1), c["ne"], c["top"], seed)


def _expert_tensors(ty, c, gen):
    ne, hidden, eff = c["ne"], c["hidden"], c["eff"]
    return _blocks(ty, ne * eff, hidden, gen), _blocks(ty, ne * eff, hidden, gen), _blocks(ty, ne * hidden, eff, gen)


def prepare(case, seed):
    c = case
    s = State(c)
    gen = torch.Generator("cuda").manual_seed(seed)
    kind = c["kind"]
    if kind == "rows":
        s.w = [s.weight(c["ty"], c["n"], c["k"], gen) for _ in range(c["layers"])]
        s.x = _acts(gen, c["m"], c["k"])
        s.y = [torch.empty(c["m"], c["n"], device="cuda") for _ in s.w]
    elif kind == "trait_gemv":
        s.w = s.weight(c["ty"], c["n"], c["k"], gen)
        s.x = _acts(gen, c["k"]).cpu().numpy()
    elif kind == "trait_batch":
        s.dims = [c["n"]] + [c["n2"]] * (c["items"] - 1)
        x = _acts(gen, c["k"]).cpu().numpy()
        s.calls = [(s.weight(c["ty"], n, c["k"], gen), x) for n in s.dims]
    elif kind == "trait_moe":
        s.layer = s.experts(c["ty"], _expert_tensors(c["ty"], c, gen), c["hidden"], c["eff"], c["ne"])
        ids, w = _routing(c, seed)
        s.ids, s.wexp = ids[0].copy(), w[0].copy()
        s.x = _acts(gen, c["hidden"]).cpu().numpy()
    elif kind == "decode":
        _prepare_decode(s, c, gen)
    elif kind == "lm_head":
        s.w = s.weight(c["ty"], c["n"], c["k"], gen)
        s.x = _acts(gen, c["m"], c["k"]).cpu().numpy()
    elif kind == "gemm":
        s.w = s.weight(c["ty"], c["n"], c["k"], gen)
        s.x = _acts(gen, c["m"], c["k"])
        s.y = torch.empty(c["m"], c["n"], device="cuda")
    elif kind == "ffn":
        s.w = [s.weight(c["ty"], c["ffn"], c["hidden"], gen), s.weight(c["ty"], c["ffn"], c["hidden"], gen), s.weight(c["ty"], c["hidden"], c["ffn"], gen)]
        s.x = _acts(gen, c["m"], c["hidden"])
        s.norm = 1 + 0.1 * _acts(gen, c["hidden"])
        s.g, s.u = (torch.empty(c["m"], c["ffn"], device="cuda") for _ in range(2))
        s.y = torch.empty(c["m"], c["hidden"], device="cuda")
    elif kind == "moe_layer":
        s.layer = s.experts(c["ty"], _expert_tensors(c["ty"], c, gen), c["hidden"], c["eff"], c["ne"])
        ids, w = _routing(c, seed)
        s.plan, s.slot_tok, s.wslot = _load("strix_rs_amd_synth", "synth.py").group_by_expert(ids, w, c["ne"])
        s.x = _acts(gen, c["m"], c["hidden"])
        if c["host"]:
            s.x = s.x.cpu().numpy()
        else:
            s.y = torch.empty(c["m"], c["hidden"], device="cuda")
    else:
        s.w = s.weight(c["ty"], c["n"], c["k"], gen)
        s.x = _acts(gen, c["m"], c["k"]).cpu().numpy()
    torch.cuda.synchronize()   # the library runs on a stream of its own
    return s


def _prepare_decode(s, c, gen):
    acc, hidden, ffn, ne = _acc(), c["hidden"], c["ffn"], c["ne"]
    tensors = _expert_tensors(c["ety"], c, gen)   # every layer has its own resident copy of them
    dense, experts = [], []
    for _ in range(c["layers"]):
        dense.append((s.weight(c["ty"], ffn, hidden, gen), s.weight(c["ty"], ffn, hidden, gen), s.weight(c["ty"], hidden, ffn, gen),
                      s.weight(Q8_0, ne, hidden, gen)))
        experts.append(s.experts(c["ety"], tensors, hidden, c["eff"], ne))
    s.norm = 1 + 0.1 * _acts(gen, hidden)
    s.x = _acts(gen, hidden)
    held = {}

    class Chain(_load("strix_rs_amd_chain", "chain.py").FfnMoeChain):
        def _alloc(self, nbytes):   # the caller's own tensors as the chain's buffers
            t = torch.zeros(nbytes // 4, device="cuda")
            held[t.data_ptr()] = t
            return t.data_ptr()

    chain = Chain(acc, c["layers"], hidden, ffn, ne, min(c["top"], ne), lambda l: dense[l], lambda l: experts[l], s.norm.data_ptr(), eps=EPS)
    torch.cuda.synchronize()
    out = chain.enqueue(s.x.data_ptr())   # every shape is seen once before the capture
    acc.sync()
    acc.graph_begin()
    chain.enqueue(s.x.data_ptr())
    s.graph = acc.graph_end()
    s.held = held
    s.out = {"y": held[out], "logits": held[chain.stage[0]["logits"]], "w": held[chain.stage[0]["w"]]}


# ---- one pass

def run(s):
    c, acc = s.case, _acc()
    kind = c["kind"]
    if kind == "rows":
        x, m = s.x.data_ptr(), c["m"]
        for w, y in zip(s.w, s.y):
            acc.gemv_dev(w, x, m, y.data_ptr())
        return s.y
    if kind == "trait_gemv":
        return (acc.gemv_f32 if c["f32"] else acc.gemv)(s.w, s.x, c["n"])
    if kind == "trait_batch":
        return acc.gemv_batch(s.calls, s.dims, f32=c["f32"])
    if kind == "trait_moe":
        return acc.moe_ffn(s.layer, s.ids, s.wexp, s.x)
    if kind == "decode":
        acc.graph_launch(s.graph)
        return s.out
    if kind == "lm_head":
        return acc.lm_head_argmax_rows(s.w, s.x, c["m"])
    if kind == "gemm":
        acc.gemm_dev(s.w, s.x.data_ptr(), c["m"], s.y.data_ptr())
        return s.y
    if kind == "ffn":
        x, g, u, y, norm, m = s.x.data_ptr(), s.g.data_ptr(), s.u.data_ptr(), s.y.data_ptr(), s.norm.data_ptr(), c["m"]
        acc.gemm_fused_dev(s.w[0], 1, x, norm, m, g, EPS)    # rmsnorm in front of gate and up
        acc.gemm_fused_dev(s.w[1], 1, x, norm, m, u, EPS)
        acc.gemm_fused_dev(s.w[2], 2, g, u, m, y)            # silu(gate) * up in front of down
        return {"gate": s.g, "up": s.u, "y": s.y}
    if kind == "moe_layer":
        if c["host"]:
            return acc.moe_layer_q8_dev(s.layer, s.x, c["m"], s.plan, s.slot_tok, s.wslot)
        acc.moe_layer_resident(s.layer, s.x.data_ptr(), c["m"], s.plan, s.slot_tok, s.wslot, s.y.data_ptr())
        return s.y
    return acc.prefill_q8_gemm(s.w, s.x, c["m"], c["n"])


# ---- what a pass cannot do without, and how far results may differ

def _wbytes(ty, n, k):
    be, bb = BLOCK[ty]
    return n * (k // be) * bb


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("rows", "trait_gemv", "lm_head", "gemm", "trait_gemm"):
        m, n, k, layers = c.get("m", 1), c["n"], c["k"], c.get("layers", 1)
        out = m * 4 if kind == "lm_head" else m * n * 4
        return {"bytes": layers * (_wbytes(c["ty"], n, k) + out) + m * k * 4, "flops": 2 * m * n * k * layers}
    if kind == "trait_batch":
        rows = c["n"] + c["n2"] * (c["items"] - 1)
        return {"bytes": _wbytes(c["ty"], rows, c["k"]) + (c["k"] + rows) * 4, "flops": 2 * rows * c["k"]}
    if kind == "ffn":
        m, h, f = c["m"], c["hidden"], c["ffn"]
        return {"bytes": 2 * _wbytes(c["ty"], f, h) + _wbytes(c["ty"], h, f) + m * (2 * h + 2 * f) * 4, "flops": 6 * m * h * f}
    h, e, top = c["hidden"], c["eff"], min(c["top"], c["ne"])
    if kind == "decode":
        per = 2 * _wbytes(c["ty"], c["ffn"], h) + _wbytes(c["ty"], h, c["ffn"]) + _wbytes(Q8_0, c["ne"], h) + top * (
            2 * _wbytes(c["ety"], e, h) + _wbytes(c["ety"], h, e))
        return {"bytes": c["layers"] * per + 3 * h * 4, "flops": c["layers"] * 2 * (3 * h * c["ffn"] + c["ne"] * h + top * 3 * h * e)}
    m = c.get("m", 1)
    active = min(c["ne"], m * top)   # the experts that m tokens can reach (with Zipf popularity a short chunk reaches fewer)
    return {"bytes": active * (2 * _wbytes(c["ty"], e, h) + _wbytes(c["ty"], h, e)) + 2 * m * h * 4, "flops": 6 * m * top * h * e}


def tolerance(case):
    kind = case["kind"]
    if kind == "lm_head":
        return "exact"            # indices
    if kind == "decode":
        return {"rel": 1e-2}      # every stage's result is quantised to int8 again, two or three times per layer
    if kind in ("ffn", "trait_moe", "moe_layer"):
        return {"rel": 1e-3}      # an intermediate result is quantised to int8: a last-bit difference moves a quant now and then
    return {"rel": 1e-5}          # exact integer block dots, summed in fp32
