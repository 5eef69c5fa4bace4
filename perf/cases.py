"""The calls whose speed this package is judged by: what a decoding or prompt-reading program spends its time in.

A case is a dict of plain values; ``kind`` names the path:

  moe          one routed-expert layer: router logits, top-k, both expert projections, weighted combine.  Decode form
               (a token or a few, a verify window) and prompt form (``prefill``); with a shared expert through
               ``moe.run``, without one through ``moe.router`` and ``moe.decode`` or ``moe.moe`` and ``moe.combine``
  qkv          an attention block's head at decode: residual add + RMSNorm + group sums, then q, k and v in one launch
  matmul       a 4-bit projection in decode form, for one to a few dozen rows (batched decode, verify windows)
  prompt       a 4-bit projection in prompt form, from short prompts to whole chunks
  exl3_mlp     an EXL3 gate/up/down MLP at decode
  exl3_prompt  an EXL3 projection on a prompt
  exl3_moe     EXL3 routed experts at decode

Sizes are those of ``bench.py``, ``bench_configs.py`` and the tests; inputs are drawn on the GPU from the seed.
"""

from __future__ import annotations

import math

import torch

from tensorfold_amd import experts, glue, moe, qmm, synthetic
from tensorfold_amd.exl3 import experts as exl3_experts
from tensorfold_amd.exl3 import linear as exl3
from tensorfold_amd.exl3 import prefill as exl3_prefill

DEV = "cuda:0"
EPS = 1e-6


def _moe(name: str, shape: synthetic.MoEShape, rows: int, prefill: bool) -> dict:
    # a decode step's picks are spread over the experts; over a prompt some are far more popular than others
    return dict(name=name, kind="moe", rows=rows, hidden=shape.hidden, experts=shape.experts, width=shape.width,
                top_k=shape.top_k, gs=shape.gs, swiglu=shape.swiglu, shared=shape.shared, prefill=prefill,
                zipf=1.1 if prefill else 0.0)


def listed() -> list[dict]:
    return [
        # one sequence being decoded: a token goes through a layer of 128 experts
        _moe("moe_decode_1", synthetic.C1, 1, False),
        # eight sequences decoded together: the benchmark's headline batch
        _moe("moe_decode_8", synthetic.C1, 8, False),
        # a verify window of 32 drafted tokens through a layer of 512 experts and a shared one
        _moe("moe_window_32", synthetic.C2, 32, False),
        # a prompt of ordinary, ragged length (relu^2 layers take the bf16 prompt arithmetic)
        _moe("moe_prompt_777", synthetic.C1, 777, True),
        # a full prompt chunk
        _moe("moe_prompt_4096", synthetic.C2, 4096, True),
        # the smallest call of a decode step: the normed residual stream into q, k and v
        dict(name="qkv_1", kind="qkv", rows=1, k=4096, n=4096, kv=1024, gs=64),
        # the widest projection of a dense layer for a window of tokens, an odd number of them
        dict(name="matmul_21", kind="matmul", rows=21, n=17408, k=5120, gs=64),
        # a short chat turn
        dict(name="prompt_100", kind="prompt", rows=100, n=4096, k=4096, gs=64),
        # a full prompt chunk through the widest projection
        dict(name="prompt_4096", kind="prompt", rows=4096, n=17408, k=5120, gs=64),
        # one sequence being decoded by a 3-bit EXL3 model
        dict(name="exl3_mlp_1", kind="exl3_mlp", rows=1, d=5120, width=17408, bits=3.0, codebook="3inst"),
        # a prompt of ordinary, ragged length through the same model's gate projection
        dict(name="exl3_prompt_1000", kind="exl3_prompt", rows=1000, k=5120, n=17408, bits=3.0, codebook="3inst"),
        # eight sequences through 4-bit EXL3 routed experts
        dict(name="exl3_moe_8", kind="exl3_moe", rows=8, d=4096, width=2048, experts=288, top_k=8, bits=4.0,
             codebook="mcg"),
    ]


def _log(rng, low: int, high: int, step: int = 1) -> int:
    """A multiple of ``step`` in [low, high], uniform over its logarithm."""

    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high // step, max(-(-low // step), round(v / step))) * step


def _drawn(rng) -> dict:
    kind, prefill = rng.choice([(c["kind"], c.get("prefill", False)) for c in listed()])
    gs = rng.choice((32, 64))
    if kind == "moe":
        swiglu, n_experts = rng.random() < 0.5, _log(rng, 16, 512)
        top_k = rng.randint(1, 10)
        # a decode call holds at most 1,024 pairs of a row and an expert; a prompt at most a chunk of 4,096 tokens
        rows = _log(rng, 64, 4096) if prefill else _log(rng, 1, 64)
        return dict(kind="moe", rows=rows, hidden=_log(rng, 512, 2688, 64), experts=n_experts,
                    width=_log(rng, 256, 768 if swiglu else 1856, 64), top_k=top_k, gs=gs, swiglu=swiglu,
                    shared=rng.random() < 0.5, prefill=prefill, zipf=1.1 if prefill else 0.0)
    if kind == "qkv":
        return dict(kind="qkv", rows=_log(rng, 1, 8), k=_log(rng, 1024, 8192, 128), n=_log(rng, 1024, 8192, 64),
                    kv=_log(rng, 128, 1024, 64), gs=gs)
    if kind == "matmul":
        return dict(kind="matmul", rows=_log(rng, 1, 64), n=_log(rng, 512, 17408), k=_log(rng, 512, 5120, gs), gs=gs)
    if kind == "prompt":
        return dict(kind="prompt", rows=_log(rng, 17, 4096), n=_log(rng, 512, 17408), k=_log(rng, 512, 5120, gs), gs=gs)
    bits, codebook = rng.choice((2.0, 2.5, 3.0, 3.5, 4.0, 5.0, 6.0)), rng.choice(("3inst", "mcg", "mul1"))
    if bits != int(bits):
        codebook = "mul1"                       # half-bit widths come with this codebook only
    if kind == "exl3_mlp":
        return dict(kind="exl3_mlp", rows=_log(rng, 1, 16), d=_log(rng, 1024, 5120, 128),
                    width=_log(rng, 2048, 17408, 128), bits=bits, codebook=codebook)
    if kind == "exl3_prompt":
        return dict(kind="exl3_prompt", rows=_log(rng, 129, 4096), k=_log(rng, 1024, 5120, 128),
                    n=_log(rng, 1024, 17408, 128), bits=bits, codebook=codebook)
    return dict(kind="exl3_moe", rows=_log(rng, 1, 16), d=_log(rng, 1024, 4096, 128), width=_log(rng, 512, 2048, 128),
                experts=_log(rng, 16, 288), top_k=rng.randint(1, 8), bits=bits, codebook=codebook)


def draw(rng) -> dict:
    """One more case: the kinds as often as they are listed, sizes over the ranges that the listed ones span, none
    larger than the largest of them (an EXL3 prompt pays for its decode besides its products)."""

    while True:
        case = _drawn(rng)
        most = {"moe": 292e9, "exl3_prompt": 550e9}.get(case["kind"], 731e9)
        if work(case)["flops"] <= most and not (case["kind"] == "moe" and not case["prefill"]
                                                and case["rows"] * (case["top_k"] + 1) > 1024):
            return case


# ---- what a program holds before the call ------------------------------------------------------------------------------


def _affine(gen, n: int, k: int, gs: int, lead: tuple[int, ...] = ()) -> tuple[torch.Tensor, ...]:
    words = torch.randint(-(2 ** 31), 2 ** 31, (*lead, n, k // 8), generator=gen, device=DEV,
                          dtype=torch.int64).to(torch.int32)
    scales = (torch.rand((*lead, n, k // gs), generator=gen, device=DEV) * 0.018 + 0.002).bfloat16()
    return words, scales, (scales.float() * -8).bfloat16()


def _rows(gen, rows: int, k: int, dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    return torch.randn((rows, k), generator=gen, device=DEV).to(dtype)


def _popularity(n_experts: int, zipf: float) -> torch.Tensor:
    """What expert e's logit has on top of its noise: with Gumbel-sized noise, picks follow (e + 1) ** -zipf."""

    return -zipf * torch.log(torch.arange(n_experts, dtype=torch.float32) + 1)


NOISE = 1.28           # standard deviation of a logit's noise: that of a Gumbel variable


def _prepare_moe(case: dict, gen) -> dict:
    d, width, gs, ne, rows = case["hidden"], case["width"], case["gs"], case["experts"], case["rows"]
    shared = int(case["shared"])
    up = [_affine(gen, width, d, gs, (ne + shared,)) for _ in range(2 if case["swiglu"] else 1)]
    ex = experts.make(up, _affine(gen, d, width, gs, (ne + shared,)), gs)
    del up
    # the residual stream has a direction that all its rows share; the router reads an expert's popularity off it
    common = torch.sign(torch.randn((d,), generator=gen, device=DEV)) * 0.25
    x = (torch.randn((rows, d), generator=gen, device=DEV) + common).bfloat16()
    router = torch.randn((ne + shared, d), generator=gen, device=DEV) * (NOISE / math.sqrt(d))
    router[:ne] += _popularity(ne, case["zipf"]).to(DEV)[:, None] * (common / common.square().sum())
    state = dict(case=case, x=x, layer=moe.Routed(router.bfloat16().contiguous(), ex, case["top_k"]))
    if not shared:
        cfg = type("Config", (), dict(num_experts_per_tok=case["top_k"], num_experts=ne, moe_intermediate_size=width,
                                      hidden_size=d))
        y_dtype = torch.float16 if case["prefill"] and ex.arith == experts.ARITH_F16 else torch.float32
        state["buffers"] = moe.MoEBuffers(rows, cfg, DEV, prefill=case["prefill"], shared=False, y_dtype=y_dtype)
    return state


def _exl3_layer(gen, k: int, n: int, bits: float, codebook: str) -> exl3.Exl3Linear:
    trellis = torch.randint(-2 ** 15, 2 ** 15, (k // 16, n // 16, int(16 * bits)), generator=gen, device=DEV,
                            dtype=torch.int32).to(torch.int16)
    # scales that leave an output as large as the input, with the signs of a checkpoint's
    scale = lambda size, mean: ((torch.rand(size, generator=gen, device=DEV) + 0.5) * mean
                                * torch.sign(torch.randn(size, generator=gen, device=DEV))).half()
    return exl3.Exl3Linear.from_tensors(trellis, scale(k, 1.0), scale(n, 1.0 / math.sqrt(k)), codebook, device=DEV)


def prepare(case: dict, seed: int) -> dict:
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    kind, rows = case["kind"], case["rows"]
    if kind == "moe":
        return _prepare_moe(case, gen)
    if kind == "qkv":
        k, gs = case["k"], case["gs"]
        weights = [qmm.pack(*_affine(gen, n, k, gs), gs) for n in (case["n"], case["kv"], case["kv"])]
        return dict(case=case, x=_rows(gen, rows, k), residual=_rows(gen, rows, k), weights=weights,
                    norm=(torch.rand((k,), generator=gen, device=DEV) + 0.5).bfloat16())
    if kind in ("matmul", "prompt"):
        return dict(case=case, x=_rows(gen, rows, case["k"]),
                    weight=qmm.pack(*_affine(gen, case["n"], case["k"], case["gs"]), case["gs"]))
    bits, codebook = case["bits"], case["codebook"]
    if kind == "exl3_mlp":
        d, width = case["d"], case["width"]
        mlp = exl3.Exl3MLP.of(_exl3_layer(gen, d, width, bits, codebook), _exl3_layer(gen, d, width, bits, codebook),
                              _exl3_layer(gen, width, d, bits, codebook))
        return dict(case=case, x=_rows(gen, rows, d, torch.float16), mlp=mlp)
    if kind == "exl3_prompt":
        return dict(case=case, x=_rows(gen, rows, case["k"], torch.float16),
                    layer=_exl3_layer(gen, case["k"], case["n"], bits, codebook), workspace=exl3_prefill.Workspace(),
                    out=torch.empty((rows, case["n"]), dtype=torch.float16, device=DEV))
    d, width, ne, top_k = case["d"], case["width"], case["experts"], case["top_k"]
    trellis = lambda k, n: torch.randint(-2 ** 15, 2 ** 15, (ne, k // 16, n // 16, int(16 * bits)), generator=gen,
                                         device=DEV, dtype=torch.int32).to(torch.int16)
    scale = lambda n, m: (torch.randn((ne, n), generator=gen, device=DEV) * m).half()
    ex = exl3_experts.prepare_stacked(trellis(d, width), trellis(d, width), trellis(width, d), scale(d, 1.0),
                                      scale(d, 1.0), scale(width, 1.0 / math.sqrt(d)), scale(width, 1.0 / math.sqrt(d)),
                                      scale(width, 1.0), scale(d, 1.0 / math.sqrt(width)), codebook)
    pick = torch.rand((rows, ne), generator=gen, device=DEV).topk(top_k, dim=1).indices.int().contiguous()
    wts = torch.softmax(torch.randn((rows, top_k), generator=gen, device=DEV), 1).bfloat16().float().contiguous()
    return dict(case=case, x=_rows(gen, rows, d), pick=pick, wts=wts, experts=ex,
                scratch=exl3_experts.Scratch(ex, rows, top_k), out=torch.empty((rows, d), device=DEV))


# ---- one pass ------------------------------------------------------------------------------------------------------------


def run(state: dict):
    case = state["case"]
    kind, rows = case["kind"], case["rows"]
    if kind == "moe":
        x, layer = state["x"], state["layer"]
        if case["shared"]:
            return moe.run(x, layer, prefill=case["prefill"])
        buf = state["buffers"]
        if case["prefill"]:
            moe.moe(x, layer.router, layer.experts, buf, case["top_k"], case["experts"])
            return moe.combine(buf.y, buf.wts)
        logits = moe.router(x, layer.router, buf.logits)
        return moe.decode(x, logits, layer.experts, buf, case["top_k"], case["experts"])
    if kind == "qkv":
        h, y, sums = glue.add_rmsnorm(state["x"], state["residual"], state["norm"], EPS, case["gs"])
        return [h, y, *qmm.matmul_group(y, state["weights"], sums)]
    if kind == "matmul":
        return qmm.matmul(state["x"], state["weight"])
    if kind == "prompt":
        return qmm.prefill_matmul(state["x"], state["weight"])
    if kind == "exl3_mlp":
        return state["mlp"](state["x"])
    if kind == "exl3_prompt":
        return exl3_prefill.matmul(state["layer"], state["x"], state["out"], state["workspace"])
    return exl3_experts.routed(state["x"], state["pick"], state["wts"], state["experts"], state["scratch"],
                               state["out"], rows)


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------


def _distinct(rows: int, n_experts: int, top_k: int, zipf: float) -> int:
    """Experts that some row picks, from one draw of logits with the case's distribution."""

    gen = torch.Generator().manual_seed(1)
    logits = torch.randn((rows, n_experts), generator=gen) * NOISE + _popularity(n_experts, zipf)
    return int(logits.topk(top_k, dim=1).indices.unique().numel())


def work(case: dict) -> dict:
    kind, rows = case["kind"], case["rows"]
    affine = lambda n, k: n * k // 2 + 4 * n * (k // case["gs"])           # 4-bit codes, a bf16 scale and bias a group
    if kind == "moe":
        d, width, ne, shared = case["hidden"], case["width"], case["experts"], int(case["shared"])
        matrices = 2 if case["swiglu"] else 1
        used = _distinct(rows, ne, case["top_k"], case["zipf"]) + shared
        per_expert = matrices * affine(width, d) + affine(d, width)
        pairs = rows * (case["top_k"] + shared)
        return {"bytes": used * per_expert + 2 * (ne + shared) * d + 2 * 2 * rows * d,
                "flops": 2 * pairs * (matrices + 1) * d * width + 2 * rows * (ne + shared) * d}
    if kind == "qkv":
        k, n = case["k"], case["n"] + 2 * case["kv"]
        return {"bytes": affine(n, k) + 2 * k + 2 * rows * (4 * k + n), "flops": 2 * rows * k * n}
    if kind in ("matmul", "prompt"):
        n, k = case["n"], case["k"]
        return {"bytes": affine(n, k) + 2 * rows * (n + k), "flops": 2 * rows * n * k}
    trellis = lambda k, n: int(k * n * case["bits"] / 8) + 2 * (k + n)
    if kind == "exl3_mlp":
        d, width = case["d"], case["width"]
        return {"bytes": 3 * trellis(d, width) + 2 * 2 * rows * d, "flops": 6 * rows * d * width}
    if kind == "exl3_prompt":
        k, n = case["k"], case["n"]
        return {"bytes": trellis(k, n) + 2 * rows * (k + n), "flops": 2 * rows * k * n}
    d, width, top_k = case["d"], case["width"], case["top_k"]
    return {"bytes": _distinct(rows, case["experts"], top_k, 0.0) * 3 * trellis(d, width) + rows * (2 + 4) * d
            + 8 * rows * top_k, "flops": 6 * rows * top_k * d * width}


# About four times a path's relative error against the same layer in 64 bits without any rounding (moe 2.0e-3 to 4.1e-3,
# qkv 3.1e-3, matmul and prompt 1.7e-3: mostly what rounding a result to bf16 costs; EXL3, fp16 results: 7.5e-4 the MLP,
# 2.9e-4 the prompt, 5.6e-4 the experts).
_REL = {"moe": 1e-2, "qkv": 1e-2, "matmul": 7e-3, "prompt": 7e-3, "exl3_mlp": 3e-3, "exl3_prompt": 1.2e-3, "exl3_moe": 2.2e-3}


def tolerance(case: dict) -> dict:
    return {"rel": _REL[case["kind"]]}
