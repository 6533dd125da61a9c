"""The work that is timed: MoE layers, their experts, the router and the token
dispatch, through the package's public entry points.

Every case is a plain dict; ``kind`` names the path:

* ``layer``: ``MoE`` (or, with ``train``, its training step): what a model's
  block calls. The output, and in training every gradient and the token counts.
* ``experts``: ``GroupedExperts`` on rows already sorted by expert, in bf16
  (``recipe`` "bf16"), with the fp8 / MXFP8 converters applied ("fp8", "mxfp8"),
  in fp32 through the per-expert path ("fp32"), or ``GptOssGroupedExperts``
  ("gptoss", biased and clamped).
* ``router``: ``TokenChoiceTopKRouter`` with its gate, forward and backward.
* ``dispatch``: ``TokenReorderer`` with the permute and combine ops around
  experts that are left out, forward and backward.

Sizes are those of the layers that this repository's benchmark and tests name
(dims 256/512, 2304/1024, 7168/2048, 2880/2880) and generic ones between them.
Row counts per expert are ragged, with empty experts where rows are few.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch
import torch.nn.functional as F

DEV = "cuda"
BF16_BYTES = 2


def listed() -> list[dict]:
    return [
        # A debug model's layer on a short sequence: fp32 parameters, experts on the
        # bf16 grouped kernels. Launches and host work are most of it.
        dict(name="layer_tiny_train", kind="layer", train=True, tokens=512, dim=256, hidden=512, experts=8, top_k=2,
             shared=0, score="softmax", norm=False, groups=0, limited=0, before=True, fp32=True),
        # One generation step of a batch of 64 sequences through a 256-expert layer:
        # a couple of rows per expert, all weights read once.
        dict(name="layer_decode", kind="layer", train=False, tokens=64, dim=2304, hidden=1024, experts=256, top_k=8,
             shared=1024, score="sigmoid", norm=True, groups=0, limited=0, before=True, fp32=False),
        # The benchmark's layer: pre-training of a 256-expert model, 4 x 4096 tokens.
        dict(name="layer_train", kind="layer", train=True, tokens=16384, dim=2304, hidden=1024, experts=256, top_k=8,
             shared=1024, score="sigmoid", norm=True, groups=0, limited=0, before=True, fp32=False),
        # Prefill of one prompt of 1000 tokens (top 8), its routing skewed.
        dict(name="experts_prefill", kind="experts", recipe="bf16", train=False, rows=8000, dim=2304, hidden=1024,
             experts=256, skew=1.0),
        # Fine-tuning on short sequences: 2048 tokens, top 8, 64 rows per expert.
        dict(name="experts_train_short", kind="experts", recipe="bf16", train=True, rows=16384, dim=2304,
             hidden=1024, experts=256, skew=0.5),
        # One rank's 32 experts of a wide layer (7168 / 2048), an odd number of rows.
        dict(name="experts_train_wide", kind="experts", recipe="bf16", train=True, rows=8199, dim=7168, hidden=2048,
             experts=32, skew=0.3),
        # gpt-oss-20b's experts: biased, clamped, 2880 is no multiple of a tile.
        dict(name="experts_train_gptoss", kind="experts", recipe="gptoss", train=True, rows=16384, dim=2880,
             hidden=2880, experts=32, skew=0.3),
        # The tiny fp32 layer's experts on the per-expert path, all in fp32.
        dict(name="experts_train_fp32", kind="experts", recipe="fp32", train=True, rows=8192, dim=256, hidden=512,
             experts=8, skew=0.3),
        # fp8 and MXFP8 experts in training: 64 experts, about 512 rows each.
        dict(name="experts_train_fp8", kind="experts", recipe="fp8", train=True, rows=32768, dim=2304, hidden=1024,
             experts=64, skew=0.3),
        dict(name="experts_train_mxfp8", kind="experts", recipe="mxfp8", train=True, rows=32768, dim=2304,
             hidden=1024, experts=64, skew=0.3),
        # The group-limited router of the wide layer, gate included.
        dict(name="router_train", kind="router", tokens=8192, dim=7168, experts=256, top_k=8, score="sigmoid",
             norm=True, groups=8, limited=4),
        # Sorting, spreading and summing the rows of the benchmark's layer.
        dict(name="dispatch_train", kind="dispatch", tokens=16384, dim=2304, experts=256, top_k=8, before=True),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (dim, hidden, experts) of the ranges: the repository's layers and sizes between them
_SHAPES = [(2304, 1024, 256), (2304, 1024, 64), (1024, 704, 64), (2048, 1408, 64), (1600, 832, 48), (4096, 1536, 32)]


def draw(rng) -> dict:
    kind = rng.choice(["layer", "layer", "experts", "experts", "experts", "experts", "experts", "experts", "router",
                       "dispatch"])
    if kind == "layer":
        train = rng.random() < 0.5
        if rng.random() < 0.35:
            return dict(kind=kind, train=train, tokens=_log_int(rng, 64, 4096), dim=256, hidden=512, experts=8,
                        top_k=2, shared=0, score="softmax", norm=False, groups=0, limited=0, before=True, fp32=True)
        dim, hidden, experts = rng.choice(_SHAPES)
        tokens = _log_int(rng, 256, 8192) if train else _log_int(rng, 8, 4096)
        return dict(kind=kind, train=train, tokens=tokens, dim=dim, hidden=hidden, experts=experts,
                    top_k=rng.choice([4, 6, 8]), shared=rng.choice([0, hidden]), score="sigmoid", norm=True, groups=0,
                    limited=0, before=rng.random() < 0.7, fp32=False)
    if kind == "experts":
        recipe = rng.choice(["bf16", "bf16", "bf16", "gptoss", "fp32", "fp8", "mxfp8"])
        train = rng.random() < 0.65
        if recipe == "fp32":
            dim, hidden, experts = rng.choice([(256, 512, 8), (512, 1024, 8), (320, 704, 16)])
            rows = _log_int(rng, 256, 16384)
        elif recipe == "gptoss":
            dim, hidden, experts = rng.choice([(2880, 2880, 32), (1472, 1472, 32)])
            rows = _log_int(rng, 64, 16384)
        elif recipe in ("fp8", "mxfp8"):
            dim, hidden, experts = rng.choice([(2304, 1024, 64), (1280, 768, 48), (4096, 1536, 16)])
            rows = _log_int(rng, 1024, 32768)
        else:
            dim, hidden, experts = rng.choice(_SHAPES + [(7168, 2048, 32)])
            rows = _log_int(rng, 64, 16384 if dim == 7168 else 65536)
        return dict(kind=kind, recipe=recipe, train=train, rows=rows, dim=dim, hidden=hidden, experts=experts,
                    skew=rng.choice([0.0, 0.3, 0.7, 1.0]))
    if kind == "router":
        return dict(kind=kind, tokens=_log_int(rng, 64, 16384), dim=rng.choice([1024, 2304, 4096]),
                    experts=rng.choice([64, 128, 256]), top_k=rng.choice([4, 6, 8]),
                    score=rng.choice(["softmax", "sigmoid"]), norm=rng.random() < 0.7,
                    **rng.choice([dict(groups=0, limited=0), dict(groups=8, limited=4)]))
    return dict(kind=kind, tokens=_log_int(rng, 64, 16384), dim=rng.choice([1024, 1600, 2304, 2880]),
                experts=rng.choice([32, 64, 256]), top_k=rng.choice([4, 6, 8]), before=rng.random() < 0.7)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(gen, *shape, std=1.0, dtype=torch.bfloat16) -> torch.Tensor:
    t = torch.randn(*shape, generator=gen, device=DEV, dtype=dtype)
    return t.mul_(std) if std != 1.0 else t


def _counts(case: dict, seed: int) -> torch.Tensor:
    """Rows per expert: a multinomial draw over exp(skew * normal) loads."""
    gen = torch.Generator().manual_seed(seed + 17)
    e = case["experts"]
    load = torch.exp(case["skew"] * torch.randn(e, generator=gen, dtype=torch.float64))
    pick = torch.multinomial(load / load.sum(), case["rows"], replacement=True, generator=gen)
    return torch.bincount(pick, minlength=e)


def _fill(module, gen, dtype, std=0.02) -> None:
    for p in module.parameters():
        p.data = torch.empty(p.shape, device=DEV, dtype=dtype).normal_(0.0, std, generator=gen)


def _make_experts(case: dict, gen) -> torch.nn.Module:
    from torchtitan_amd import GroupedExperts
    from torchtitan_amd.gpt_oss import GptOssGroupedExperts
    from torchtitan_amd.quantization import Float8GroupedMMConverter, MXFP8Converter

    d, h, e, recipe = case["dim"], case["hidden"], case["experts"], case["recipe"]
    cls = GptOssGroupedExperts if recipe == "gptoss" else GroupedExperts
    with torch.device("meta"):
        experts = cls.Config(dim=d, hidden_dim=h, num_experts=e, use_grouped_mm=recipe != "fp32").build()
    experts = experts.to_empty(device=DEV)
    model = torch.nn.ModuleDict({"experts": experts})
    _fill(model, gen, torch.float32 if recipe == "fp32" else torch.bfloat16)
    dims = SimpleNamespace(pp_enabled=False, cp_enabled=False, ep_enabled=False)
    if recipe == "fp8":
        Float8GroupedMMConverter.Config(fqns=["experts"]).build(
            parallel_dims=dims, model_compile_enabled=False).convert(model)
    elif recipe == "mxfp8":
        MXFP8Converter.Config(recipe_name="mxfp8_rceil", fqns=["experts"]).build(
            parallel_dims=dims, model_compile_enabled=False).convert(model)
    return experts


def _make_layer(case: dict, gen) -> torch.nn.Module:
    from torchtitan_amd import FeedForward, GroupedExperts, Linear, MoE

    d, h, e, hs = case["dim"], case["hidden"], case["experts"], case["shared"]
    cfg = MoE.Config(
        num_experts=e,
        experts=GroupedExperts.Config(dim=d, hidden_dim=h, num_experts=e),
        router=_router_config(case),
        score_before_experts=case["before"],
        shared_experts=FeedForward.Config(
            w1=Linear.Config(in_features=d, out_features=hs), w2=Linear.Config(in_features=hs, out_features=d),
            w3=Linear.Config(in_features=d, out_features=hs)) if hs else None,
    )
    with torch.device("meta"):
        moe = cfg.build()
    moe = moe.to_empty(device=DEV)
    _fill(moe, gen, torch.float32 if case["fp32"] else torch.bfloat16)
    moe.expert_bias.copy_(_bias(gen, e))
    moe.tokens_per_expert.zero_()
    return moe


def _router_config(case: dict):
    from torchtitan_amd import Linear, TokenChoiceTopKRouter

    return TokenChoiceTopKRouter.Config(
        num_experts=case["experts"], gate=Linear.Config(in_features=case["dim"], out_features=case["experts"]),
        top_k=case["top_k"], score_func=case["score"], route_norm=case["norm"], route_scale=_scale(case),
        num_expert_groups=case["groups"] or None, num_limited_groups=case["limited"] or None)


def _scale(case: dict) -> float:
    return 2.5 if case["norm"] else 1.0


def _bias(gen, e: int) -> torch.Tensor:
    return (torch.rand(e, generator=gen, device=DEV) * 2 - 1) * 0.01


def prepare(case: dict, seed: int) -> dict:
    gen = _gen(seed)
    kind = case["kind"]
    st: dict = {"kind": kind, "train": case.get("train", True)}
    if kind == "experts":
        dt = torch.float32 if case["recipe"] == "fp32" else torch.bfloat16
        st["module"] = _make_experts(case, gen)
        st["counts"] = _counts(case, seed).to(DEV)
        st["x"] = _normal(gen, case["rows"], case["dim"], dtype=dt)
        st["dy"] = _normal(gen, case["rows"], case["dim"], dtype=dt) if st["train"] else None
    elif kind == "layer":
        dt = torch.float32 if case["fp32"] else torch.bfloat16
        st["module"] = _make_layer(case, gen)
        st["x"] = _normal(gen, 1, case["tokens"], case["dim"], dtype=dt)
        st["dy"] = _normal(gen, 1, case["tokens"], case["dim"], dtype=dt) if st["train"] else None
    elif kind == "router":
        with torch.device("meta"):
            router = _router_config(case).build()
        router = router.to_empty(device=DEV)
        _fill(router, gen, torch.bfloat16)
        st["module"] = router
        st["bias"] = _bias(gen, case["experts"])
        st["x"] = _normal(gen, case["tokens"], case["dim"])
        st["dy"] = _normal(gen, case["tokens"], case["top_k"], dtype=torch.float32)
    else:
        from torchtitan_amd.moe import TokenReorderer

        n, e, k = case["tokens"], case["experts"], case["top_k"]
        st["module"] = TokenReorderer(num_experts=e, top_k=k)
        st["before"] = case["before"]
        st["ids"] = torch.rand(n, e, generator=gen, device=DEV).topk(k, dim=1).indices
        st["scores"] = torch.rand(n, k, generator=gen, device=DEV).requires_grad_(True)
        st["x"] = _normal(gen, n, case["dim"])
        st["shared"] = _normal(gen, n, case["dim"]).requires_grad_(True)
        st["dy"] = _normal(gen, n, case["dim"])
    if st["train"]:
        st["x"].requires_grad_(True)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st: dict):
    kind, module, x = st["kind"], st["module"], st["x"]
    if kind == "experts":
        if not st["train"]:
            with torch.no_grad():
                return module(x, st["counts"])
        y = module(x, st["counts"])
        return [y.detach(), *torch.autograd.grad(y, [x, *module.parameters()], st["dy"])]
    if kind == "layer":
        if not st["train"]:
            with torch.no_grad():
                return [module(x), module.tokens_per_expert]
        y = module(x)
        grads = torch.autograd.grad(y, [x, *module.parameters()], st["dy"])
        return [y.detach(), module.tokens_per_expert, *grads]
    if kind == "router":
        top, idx, counts = module(x, st["bias"])
        grads = torch.autograd.grad(top, [x, *module.parameters()], st["dy"])
        return [top.detach(), idx, counts, *grads]
    from torchtitan_amd import ops

    layout = module(st["scores"], st["ids"])
    scores, token_idx, counts = layout
    before = st["before"]
    routed = ops.permute(x, layout.slot_pos, layout.tok_pos, scores if before else None)
    out = ops.combine(st["shared"], routed, layout.slot_pos, layout.tok_pos, None if before else scores)
    grads = torch.autograd.grad(out, [x, st["shared"], st["scores"]], st["dy"])
    return [out.detach(), routed.detach(), token_idx, counts, *grads]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _expert_work(rows: int, d: int, h: int, e: int, train: bool, bytes_per: int) -> tuple[float, float]:
    used = e * (1.0 - (1.0 - 1.0 / e) ** rows)  # experts that get a row
    weights = 3.0 * d * h * bytes_per
    nbytes = used * weights + 2.0 * rows * d * bytes_per
    flops = 6.0 * rows * d * h
    if train:
        nbytes += e * weights + 2.0 * rows * d * bytes_per
        flops *= 3
    return nbytes, flops


def work(case: dict) -> dict:
    kind, d, e = case["kind"], case["dim"], case["experts"]
    if kind == "experts":
        b, f = _expert_work(case["rows"], d, case["hidden"], e, case["train"], 4 if case["recipe"] == "fp32" else 2)
        return {"bytes": b, "flops": f}
    n, k = case["tokens"], case["top_k"]
    if kind == "layer":
        el = 4 if case["fp32"] else 2
        train = case["train"]
        used = e * (1.0 - (1.0 - k / e) ** n)
        dense = d * e + 3 * d * case["shared"]  # gate and shared expert weights
        b = el * (3.0 * d * case["hidden"] * used + dense + 2.0 * n * d)
        f = 6.0 * n * k * d * case["hidden"] + 2.0 * n * dense
        if train:
            b += el * (3.0 * d * case["hidden"] * e + dense + 2.0 * n * d)
            f *= 3
        return {"bytes": b, "flops": f}
    if kind == "router":
        return {"bytes": BF16_BYTES * (2.0 * n * d + 2.0 * e * d) + 16.0 * n * k, "flops": 6.0 * n * d * e}
    # x, the shared rows, dy in; out, two row gradients; ids, scores and their gradient;
    # the routed rows (and their gradient), which the experts between would read and write
    return {"bytes": BF16_BYTES * (6.0 * n * d + 4.0 * n * k * d) + 24.0 * n * k, "flops": 6.0 * n * k * d}


def tolerance(case: dict) -> dict:
    kind = case["kind"]
    if kind == "experts" and case["recipe"] == "fp32":  # 7e-7 off 64 bits as measured, in any order of the sums
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "dispatch":  # 0.0033 off 64 bits (eight bf16 adds); indices are whole
        return {"rel": 1e-2, "max": 0.1}
    # bf16 results 0.004 to 0.006 off 64 bits; two roundings of one value differ by that
    # times 1.4; ties of the top k may fall either way
    return {"rel": 1e-2, "max": 0.5, "differ": 1e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _leaf(t: torch.Tensor) -> torch.Tensor:
    return t.detach().double().requires_grad_(True)


def _act_gptoss(h1: torch.Tensor) -> torch.Tensor:
    glu, lin = h1[:, ::2].clamp(max=7.0), h1[:, 1::2].clamp(min=-7.0, max=7.0)
    return glu * torch.sigmoid(1.702 * glu) * (lin + 1)


def _expert64(params: list[torch.Tensor], x: torch.Tensor) -> torch.Tensor:
    if len(params) == 4:
        w1, b1, w2, b2 = params
        return _act_gptoss(x @ w1.t() + b1) @ w2.t() + b2
    w1, w2, w3 = params
    return (F.silu(x @ w1.t()) * (x @ w3.t())) @ w2.t()


def _experts64(params, x, dy, counts):
    """(y, [dx, dparams...]) expert by expert; params are [E, ...] tensors."""
    y, dx = [], []
    grads = [torch.zeros(p.shape, device=DEV, dtype=torch.float64) for p in params] if dy is not None else []
    r = 0
    for e, c in enumerate(counts.tolist()):
        if c == 0:
            continue
        pe, xe = [_leaf(p[e]) for p in params], _leaf(x[r:r + c])
        ye = _expert64(pe, xe)
        y.append(ye.detach())
        if dy is not None:
            got = torch.autograd.grad(ye, [xe, *pe], dy[r:r + c].double())
            dx.append(got[0])
            for g, v in zip(grads, got[1:]):
                g[e] = v
        r += c
    return torch.cat(y), ([torch.cat(dx), *grads] if dy is not None else [])


def _route64(case, x, gate, bias):
    """Scores in 64 bits for the experts that fp32 logits select: (top, idx)."""
    logits32 = F.linear(x.detach().float(), gate.detach().float())
    logits = x @ gate.t()
    act = (lambda v: v.softmax(-1)) if case["score"] == "softmax" else torch.sigmoid
    choice = act(logits32) + bias
    if case["groups"]:
        n = choice.shape[0]
        grp = choice.view(n, case["groups"], -1)
        best = grp.topk(2, dim=-1).values.sum(-1).topk(case["limited"], dim=-1).indices
        keep = torch.zeros(n, case["groups"], dtype=torch.bool, device=DEV).scatter_(1, best, True)
        choice = grp.masked_fill(~keep.unsqueeze(-1), float("-inf")).view(n, -1)
    idx = torch.topk(choice, case["top_k"], dim=-1, sorted=False).indices
    top = act(logits).gather(1, idx)
    if case["norm"]:
        top = top / (top.sum(-1, keepdim=True) + 1e-20)
    return top * _scale(case), idx


def exact(case: dict, seed: int):
    st = prepare(case, seed)
    kind, module = case["kind"], st["module"]
    if kind == "experts":
        y, grads = _experts64([p.detach() for p in module.parameters()], st["x"].detach(), st["dy"], st["counts"])
        return [y, *grads] if st["train"] else y
    if kind == "dispatch":
        x, sh, sc = _leaf(st["x"]), _leaf(st["shared"]), _leaf(st["scores"])
        # a token's rows are summed with their scores wherever those are applied
        out = sh + x * sc.sum(1, keepdim=True)
        order = torch.argsort(st["ids"].reshape(-1), stable=True)
        counts = torch.bincount(st["ids"].reshape(-1), minlength=case["experts"])
        tok = order // case["top_k"]
        routed = x.detach()[tok]
        if case["before"]:
            routed = routed * sc.detach().reshape(-1)[order].unsqueeze(1)
        return [out.detach(), routed, tok, counts, *torch.autograd.grad(out, [x, sh, sc], st["dy"].double())]
    if kind == "router":
        x, gate = _leaf(st["x"]), _leaf(module.gate.weight)
        top, idx = _route64(case, x, gate, st["bias"])
        counts = torch.bincount(idx.reshape(-1), minlength=case["experts"])
        return [top.detach(), idx, counts, *torch.autograd.grad(top, [x, gate], st["dy"].double())]

    named = dict(module.named_parameters())
    x = _leaf(st["x"].view(-1, case["dim"]))
    leaf = {n: _leaf(p) for n, p in named.items() if not n.startswith("experts.")}
    top, idx = _route64(case, x, leaf["router.gate.weight"], module.expert_bias)
    counts = torch.bincount(idx.reshape(-1), minlength=case["experts"])
    order = torch.argsort(idx.reshape(-1), stable=True)
    tok, score = order // case["top_k"], top.reshape(-1)[order].unsqueeze(1)
    routed = x[tok] * score if case["before"] else x[tok]
    dy = st["dy"].view(-1, case["dim"]).double() if st["train"] else None
    weights = [named[f"experts.{n}"].detach() for n in ("w1", "w2", "w3")]
    # the experts stand apart from the rest of the graph: their output rows' gradient
    # is dy (times the score, where that comes after them)
    rows_dy = None if dy is None else (dy[tok] if case["before"] else dy[tok] * score.detach())
    y, eg = _experts64(weights, routed.detach(), rows_dy, counts)
    out = torch.zeros_like(x).index_add(0, tok, y if case["before"] else y * score)
    if case["shared"]:
        s1, s2, s3 = (leaf[f"shared_experts.w{i}.weight"] for i in (1, 2, 3))
        out = out + (F.silu(x @ s1.t()) * (x @ s3.t())) @ s2.t()
    shape = st["x"].shape
    if dy is None:
        return [out.detach().view(shape), counts.double()]
    wrt = [x, *leaf.values()]
    total = (out * dy).sum() + (routed * eg[0]).sum()
    got = dict(zip(["x", *leaf], torch.autograd.grad(total, wrt)))
    got.update(zip(["experts.w1", "experts.w2", "experts.w3"], eg[1:]))
    return [out.detach().view(shape), counts.double(), got["x"].view(shape), *(got[n] for n in named)]
