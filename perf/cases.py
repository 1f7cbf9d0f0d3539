"""The calls this library is measured on: MoE layers of the three model families (synthetic weights of the shapes in
moe_gen_amd/synthetic.py) from single-token decode to the largest prefill batch, a dense MLP of the same models, and
layers whose expert weights are streamed from host memory.

A case is a dict of plain values:
  path      "block"  -- the layer's forward, block(hidden_states)
            "norm"   -- norm, layer and residual add in one call, norm_moe_residual(block, hidden_states, weight)
            "mlp"    -- DeepseekV3MLP on its own: the dense MLP of DeepSeek-V3's first layers (fp8 weights)
            "staged" -- three layers in turn, every expert delivered from pinned host memory by a Stager
  workload  a name of synthetic.WORKLOADS: shapes, routing rules and weight type
  n         tokens in the call
"""
from __future__ import annotations

import math

import torch
from torch import nn

from moe_gen_amd import DeepseekV3Config, DeepseekV3MLP, StagedExpert, Stager, norm_moe_residual, synthetic
from moe_gen_amd.block import attach_fp8_weight

STAGED_LAYERS = 3
STAGED_POOL = 20          # routed-expert slots of the engine's prefill phase

# largest token count of each workload (the batch it is benchmarked with)
MAX_TOKENS = {"deepseek_v2_lite": 4096, "mixtral_8x7b": 16384, "mixtral_8x22b": 8192,
              "deepseek_v2_236b": 32768, "deepseek_v3_w8a16": 65536}
MAX_TOKENS_MLP = 8192
MAX_TOKENS_STAGED = 2048


def listed():
    def case(name, path, workload, n):
        return {"name": name, "path": path, "workload": workload, "n": n}
    return [
        # one user's token through a small model: nothing but launches, host work and six experts' weights
        case("v2_lite_1", "block", "deepseek_v2_lite", 1),
        # a few users on the largest model: a few dozen of 256 experts, one row each
        case("v3_5", "block", "deepseek_v3_w8a16", 5),
        # a decode batch of the middle model, with the norm and residual of the decoder layer around it
        case("v2_236b_64_norm", "norm", "deepseek_v2_236b", 64),
        # the engine's decode batches: every expert's weights are streamed once for a handful of rows
        case("v3_256", "block", "deepseek_v3_w8a16", 256),
        case("mixtral_8x22b_256", "block", "mixtral_8x22b", 256),
        # the engine's default prefill: a few prompts of a small model
        case("v2_lite_4096", "block", "deepseek_v2_lite", 4096),
        # a ragged prefill chunk of the largest model: about 90 rows an expert, no multiple of any tile
        case("v3_2997_norm", "norm", "deepseek_v3_w8a16", 2997),
        # large prefill batches: matrix-core work; Mixtral a few large experts, the other two many small ones
        case("mixtral_8x7b_16384", "block", "mixtral_8x7b", 16384),
        case("v2_236b_32768", "block", "deepseek_v2_236b", 32768),
        case("v3_65536", "block", "deepseek_v3_w8a16", 65536),
        # the dense layers at the bottom of DeepSeek-V3
        case("v3_dense_mlp_1000", "mlp", "deepseek_v3_w8a16", 1000),
        # weights that do not fit the card: host link bound
        case("v2_lite_staged_2048", "staged", "deepseek_v2_lite", 2048),
    ]


def draw(rng):
    path = rng.choice(["block"] * 5 + ["norm"] * 3 + ["mlp"] * 2 + ["staged"])
    if path == "mlp":
        workload, top = "deepseek_v3_w8a16", MAX_TOKENS_MLP
    elif path == "staged":
        workload, top = "deepseek_v2_lite", MAX_TOKENS_STAGED
    else:
        workload = rng.choice(sorted(MAX_TOKENS))
        top = MAX_TOKENS[workload]
    n = min(top, max(1, round(math.exp(rng.uniform(0.0, math.log(top))))))
    return {"path": path, "workload": workload, "n": n}


def _workload(case, seed):
    # one sequence of n tokens, or n sequences of one: the layers flatten it either way
    return synthetic.WORKLOADS[case["workload"]].scaled(n=case["n"], seq=case["n"], seed=seed)


def _norm_weight(h, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed + 31)
    return (1.0 + 0.1 * torch.randn(h, generator=g, device="cuda")).to(torch.bfloat16)


def _dense_mlp(h, seed):
    cfg = DeepseekV3Config(hidden_size=h)
    with torch.device("meta"):
        mlp = DeepseekV3MLP(cfg)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed + 17)
    for lin in mlp.projections():
        w = torch.randn(lin.weight.shape, generator=g, device="cuda") * 0.02
        attach_fp8_weight(lin, *synthetic.quantize_fp8_block128(w))
    return mlp.eval()


def _staged_layers(w, seed):
    """Three layers whose experts, routed and shared, live in pinned host memory behind one Stager."""
    layers, stager = [], None
    for j in range(STAGED_LAYERS):
        blk = synthetic.build_block(w.scaled(seed=seed + 101 * j), device="cuda")
        layer = 1 + j
        modules = [(e, ex) for e, ex in enumerate(blk.experts)] + [(-1, blk.shared_experts)]
        if stager is None:
            def shapes(mlp):
                return {f"{p}.weight": (tuple(getattr(mlp, p).weight.shape), torch.bfloat16) for p in mlp.names}
            stager = Stager({"routed_expert": shapes(blk.experts[0]), "shared_expert": shapes(blk.shared_experts)},
                            {"routed_expert": STAGED_POOL, "shared_expert": 2}, model_type="deepseek_v2",
                            num_hidden_layers=1 + STAGED_LAYERS, num_local_experts=w.E)
        staged = []
        for e, mlp in modules:
            host = {f"{p}.weight": torch.empty(getattr(mlp, p).weight.shape, dtype=torch.bfloat16, pin_memory=True)
                    .copy_(getattr(mlp, p).weight.data) for p in mlp.names}
            key, kind = (f"routed_expert_{layer}_{e}", "routed_expert") if e >= 0 else (f"shared_expert_{layer}",
                                                                                         "shared_expert")
            stager.add_module(key, kind, host)
            for p in mlp.names:                       # the engine's placeholder: the parameter holds nothing
                getattr(mlp, p).weight = nn.Parameter(torch.empty(0, dtype=torch.bfloat16), requires_grad=False)
            staged.append(StagedExpert(mlp, layer, e, stager))
        blk.shared_experts = staged.pop()
        blk.experts = nn.ModuleList(staged)
        layers.append(blk)
    stager.pump()
    return layers, stager


def prepare(case, seed):
    w = _workload(case, seed)
    state = {"path": case["path"], "x": synthetic.hidden_states(w, "cuda")}
    if case["path"] == "mlp":
        state["mlp"] = _dense_mlp(w.h, seed)
    elif case["path"] == "staged":
        state["layers"], state["stager"] = _staged_layers(w, seed)
    else:
        state["block"] = synthetic.build_block(w, device="cuda")
        if case["path"] == "norm":
            state["norm_weight"] = _norm_weight(w.h, seed)
    return state


def run(state):
    if state["path"] == "mlp":
        return state["mlp"](state["x"])
    if state["path"] == "staged":
        return [layer(state["x"]) for layer in state["layers"]]
    if state["path"] == "norm":
        return norm_moe_residual(state["block"], state["x"], state["norm_weight"])
    return state["block"](state["x"])


def _experts_with_tokens(w, n):
    """Experts of the layer that n tokens reach: logits drawn as the synthetic gate gives them (a normal per token and
    expert, plus the expert's Zipf bias), then the workload's top-k rule.  Past 4096 tokens no more are reached."""
    g = torch.Generator()
    g.manual_seed(0)
    logits = torch.randn((min(n, 4096), w.E), generator=g) * (0.02 * math.sqrt(w.h))
    if w.zipf is not None:
        logits -= w.zipf * torch.log(1.0 + torch.randperm(w.E, generator=g))
    if w.n_group > 1:
        per_group = logits.view(len(logits), w.n_group, -1)
        best = per_group.topk(2 if w.family == "v3" else 1, dim=2).values.sum(2).topk(w.topk_group, dim=1).indices
        kept = torch.zeros(len(logits), w.n_group, dtype=torch.bool).scatter_(1, best, True)
        logits = per_group.masked_fill(~kept.unsqueeze(2), -math.inf).view(len(logits), w.E)
    return int(logits.topk(w.k, dim=1).indices.unique().numel())


def work(case):
    """Weights of the experts that receive a token read once, hidden states read once and written once (Mixtral: and
    its bf16 logits); products of the router and of the experts' three matrices."""
    w = synthetic.WORKLOADS[case["workload"]]
    n = case["n"]
    rows = 4.0 * n * w.h
    if case["path"] == "mlp":
        inter = DeepseekV3Config().intermediate_size
        return {"bytes": 3.0 * w.h * inter + rows, "flops": 6.0 * n * w.h * inter}
    touched = w.E if case["path"] == "staged" else _experts_with_tokens(w, n)      # (staged: the engine delivers all)
    matrices = 3.0 * w.h * w.I * (touched + w.S) * (1.0 if w.fp8 else 2.0)
    logits = 2.0 * n * w.E if w.family == "mixtral" else 0.0
    layers = STAGED_LAYERS if case["path"] == "staged" else 1
    return {"bytes": layers * (matrices + 2.0 * w.E * w.h + rows + logits),
            "flops": layers * (6.0 * n * (w.k + w.S) * w.h * w.I + 2.0 * n * w.E * w.h)}


def tolerance(case):
    """Activations, expert results and outputs are rounded to bf16, fp8 weights also as they are dequantised.  The paths
    differ from a float64 evaluation that rounds at the same places by a relative 0.6e-3 to 3.2e-3 (sums in another
    order move values by a rounding step), from one that rounds nowhere by 4.3e-3 to 5.2e-3."""
    return {"rel": 1e-2}
