"""Whole-layer parity: the three blocks behind the reference's forward(hidden_states) surface
against the CPU oracle (indices / permutation bit-exact, output within the stated bf16 bound)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from util import bits, oracle_spec, oracle_weights, rel_max, rel_rms

pytestmark = pytest.mark.gpu

TOL = 2e-2   # max|y - y_ref| / max|y_ref|, y_ref = fp32 evaluation on bf16-rounded inputs/weights


def small(name):
    from moe_gen_amd.synthetic import WORKLOADS
    w = WORKLOADS[name]
    return {
        "deepseek_v2_lite": w.scaled(n=384, h=512, I=256, seq=128),
        "mixtral_8x7b": w.scaled(n=320, h=512, I=1024, seq=64),
        "mixtral_8x22b": w.scaled(n=200, h=768, I=512, seq=1),
        "mixtral_8x22b_decode": w.scaled(n=96, h=768, I=512, seq=1),
        "deepseek_v2_236b": w.scaled(n=512, h=512, I=256, seq=128),
        "deepseek_v3_w8a16": w.scaled(n=512, h=512, I=256, seq=128),
    }[name]


COMBINE = {"v3": O.COMBINE_F32, "v2": O.COMBINE_BF16_PROD, "mixtral": O.COMBINE_BF16_SEQ}


@pytest.mark.parametrize("name", ["deepseek_v2_lite", "mixtral_8x7b", "mixtral_8x22b", "mixtral_8x22b_decode",
                                  "deepseek_v2_236b", "deepseek_v3_w8a16"])
@pytest.mark.parametrize("fused_gather", [True, False])
def test_block_vs_oracle(name, fused_gather):
    from moe_gen_amd import synthetic
    w = small(name)
    print(f"layer case {name} fused_gather={fused_gather}", flush=True)
    blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
    blk.fused_gather = fused_gather
    x = synthetic.hidden_states(w, "cpu")
    res = blk(x.cuda())
    out = res[0] if isinstance(res, tuple) else res
    torch.cuda.synchronize()
    assert out.shape == x.shape and out.dtype == torch.bfloat16
    lw = oracle_weights(blk, w.family)
    spec = oracle_spec(w)
    xb = bits(x).reshape(w.n, w.h)
    ref32, aux = O.layer(xb, lw, spec, COMBINE[w.family], rounding="f32")
    refr, _ = O.layer(xb, lw, spec, COMBINE[w.family], rounding="ref")
    assert np.array_equal(blk.last_topk_idx.cpu().numpy(), aux["idx"])
    assert np.array_equal(blk.last_topk_weight.cpu().numpy().view(np.uint32), aux["w"].view(np.uint32))
    assert np.array_equal(blk.last_counts.cpu().numpy(), aux["counts"])
    y = O.bf16_to_f32(bits(out)).reshape(w.n, w.h)
    e32, er = rel_max(y, ref32), rel_max(y, O.bf16_to_f32(refr))
    print(f"  max-rel vs fp32 {e32:.3e} (rms {rel_rms(y, ref32):.3e}); vs reference-rounding {er:.3e}", flush=True)
    assert e32 <= TOL and er <= TOL
    if w.family == "mixtral":
        assert np.array_equal(O.bf16_to_f32(bits(res[1])), aux["logits"])


def test_gate_module_surface():
    """MoEGate.forward keeps the reference's return convention."""
    from moe_gen_amd import DeepseekV2Config, DeepseekV3Config, deepseek_v2, deepseek_v3
    x = torch.randn(2, 5, 256, device="cuda").to(torch.bfloat16)
    g3 = deepseek_v3.MoEGate(DeepseekV3Config(hidden_size=256, n_routed_experts=32, n_group=4, topk_group=2,
                                              num_experts_per_tok=4)).cuda().eval()
    g3.weight.data = g3.weight.data.to(torch.bfloat16)
    idx, w = g3(x)
    assert idx.dtype == torch.int64 and idx.shape == (10, 4) and w.dtype == torch.float32
    g2 = deepseek_v2.MoEGate(DeepseekV2Config(hidden_size=256, n_routed_experts=16, num_experts_per_tok=3,
                                              topk_method="greedy")).cuda().eval()
    g2.weight.data = g2.weight.data.to(torch.bfloat16)
    idx, w, aux = g2(x)
    assert aux is None and idx.shape == (10, 3)
    g2.scoring_func = "sigmoid"
    with pytest.raises(NotImplementedError):
        g2(x)


def test_dense_equivalence():
    """k = E and identical experts: every token visits every expert, so the layer equals the
    dense MLP scaled by the sum of the routing weights (= 1 after softmax over all experts)."""
    from moe_gen_amd import DeepseekV2Config, DeepseekV2MoE
    cfg = DeepseekV2Config(hidden_size=256, moe_intermediate_size=128, n_routed_experts=4, num_experts_per_tok=4,
                           topk_method="greedy")
    blk = DeepseekV2MoE(cfg).cuda().to(torch.bfloat16).eval()
    for ex in blk.experts[1:]:
        for a, b in zip(ex.projections(), blk.experts[0].projections()):
            a.weight.data = b.weight.data.clone()
    x = torch.randn(1, 200, 256, device="cuda").to(torch.bfloat16)
    y = blk(x).float()
    ref = blk.experts[0](x).float()
    assert rel_max(y.cpu().numpy(), ref.cpu().numpy()) <= TOL


@pytest.mark.parametrize("name", ["deepseek_v3_w8a16", "deepseek_v2_lite", "mixtral_8x7b"])
def test_block_edge_shapes(name):
    """Empty batch, a single token, a non-contiguous view, a batch of identical tokens (every row
    takes the same experts: k experts get everything, the rest nothing)."""
    from moe_gen_amd import synthetic
    w = synthetic.WORKLOADS[name].scaled(n=64, h=512, I=256, seq=64)
    blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
    first = lambda r: r[0] if isinstance(r, tuple) else r
    x = synthetic.hidden_states(w, "cpu").cuda()                      # [1, 64, 512]
    full = first(blk(x)).clone()
    # empty
    out = first(blk(x[:, :0]))
    assert out.shape == (1, 0, w.h)
    # one token: same bits as that token inside the batch (rows are independent)
    one = first(blk(x[:, 5:6].contiguous()))
    assert torch.equal(one, full[:, 5:6])
    # non-contiguous input
    xt = torch.empty(w.h, 64, dtype=torch.bfloat16, device="cuda").t().unsqueeze(0)   # strides (1, 64)
    xt.copy_(x)
    assert not xt.is_contiguous() and torch.equal(first(blk(xt)), full)
    # identical tokens
    same = x[:, :1].expand(1, 64, w.h).contiguous()
    out = first(blk(same))
    torch.cuda.synchronize()
    assert int((blk.last_counts > 0).sum()) == w.k and int(blk.last_counts.max()) == 64
    assert torch.equal(out, full[:, :1].expand_as(out))


@pytest.mark.parametrize("name", ["mixtral_8x22b_decode", "deepseek_v2_lite", "deepseek_v3_w8a16"])
def test_block_forward_can_be_captured_in_a_graph(name):
    """The block's forward with resident weights launches kernels and nothing else (no host read, no memset, no
    allocation outside torch's), so a decode loop may capture it in a HIP graph.  Replayed three times with eager
    forwards and synchronisations in between, then on a new input: every replay bit-for-bit the eager result."""
    from moe_gen_amd import synthetic
    w = small(name)
    print(f"graph capture {name}", flush=True)
    blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
    first = lambda o: o[0] if isinstance(o, tuple) else o
    x = synthetic.hidden_states(w, "cuda")
    y_ref = first(blk(x)).clone()
    torch.cuda.synchronize()
    x_static = x.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            blk(x_static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y_static = first(blk(x_static))
    torch.cuda.synchronize()
    for it in range(3):
        y_static.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y_static, y_ref), f"replay {it} differs from the eager forward"
        assert torch.equal(first(blk(x)), y_ref)         # the program's own eager work between the replays
        torch.cuda.synchronize()
    x2 = x.flip(0).contiguous()
    y2 = first(blk(x2)).clone()
    x_static.copy_(x2)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y_static, y2), "replay on a new input differs from the eager forward"


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
def test_single_shared_expert_joins_the_routed_call_at_small_batches(fp8):
    """A DeepSeek-V3-shaped block (one shared expert of the routed experts' shape) under a small batch runs the shared
    expert as one more group of the routed experts' grouped call.  The stage timer then shows no launches of its own,
    and with bf16 weights the output equals, bit for bit, what the two separate calls give (every bf16 path adds in
    one order); with fp8 weights the two agree within the layer bound, since a call that the one-workgroup-per-tile
    kernel serves alone adds in another order than the persistent kernel.  (test_block_vs_oracle holds the joined
    path to the oracle: its DeepSeek-V3 cases are small batches.)"""
    from moe_gen_amd import synthetic
    from moe_gen_amd.block import StageTimer
    w = synthetic.WORKLOADS["deepseek_v3_w8a16"].scaled(n=384, h=512, I=256, seq=64, fp8=fp8)
    blk = synthetic.build_block(w, device="cuda:0", gen_device="cpu")
    x = synthetic.hidden_states(w, "cpu").to("cuda:0")
    blk.stage_timer = StageTimer()
    joined = blk(x)
    torch.cuda.synchronize()
    keys = set(blk.stage_timer.totals_ms())
    blk.stage_timer = StageTimer()
    blk.join_shared = False
    apart = blk(x)
    torch.cuda.synchronize()
    keys_apart = set(blk.stage_timer.totals_ms())
    blk.stage_timer = None
    assert "shared_gate_up" not in keys and "routed_gate_up" in keys
    assert "shared_gate_up" in keys_apart
    a, b = joined.float(), apart.float()
    if fp8:
        assert (a - b).abs().max().item() <= 2e-2 * b.abs().max().item()
    else:
        assert torch.equal(joined, apart)


@pytest.mark.parametrize("name,E", [("deepseek_v3_w8a16", 256), ("deepseek_v2_236b", 160), ("deepseek_v2_lite", 64), ("deepseek_v2_lite", 24),
                                    ("mixtral_8x7b", 8)])
def test_layer_call_equals_the_separate_calls(name, E):
    """The whole-layer call of the library (selection and dispatch in one launch up to 16 ... 64 tokens) against the stage-by-stage
    path that an attached timer takes, at both sides of 64 tokens and of 16, where the experts change kernels, with and
    without the norm around the layer: output, routing, counts and Mixtral's logits bit for bit."""
    from moe_gen_amd import norm_moe_residual, synthetic
    from moe_gen_amd.block import StageTimer
    w = synthetic.WORKLOADS[name].scaled(n=200, h=512, I=256, seq=200, E=E)
    blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
    xs = synthetic.hidden_states(w, "cpu").cuda()
    nw = (1 + 0.1 * torch.randn(512, generator=torch.Generator().manual_seed(1))).to(torch.bfloat16).cuda()
    for n in (1, 15, 16, 17, 63, 64, 65, 200):
        x = xs[:, :n].contiguous()
        for norm in (False, True):
            print(f"layer call {name} E={E} n={n} norm={norm}", flush=True)
            run = lambda: norm_moe_residual(blk, x, nw) if norm else blk(x)
            got = []
            for timer in (None, StageTimer()):
                blk.stage_timer = timer
                res = run()
                res = res if isinstance(res, tuple) else (res,)
                got.append([*res, blk.last_topk_idx, blk.last_topk_weight, blk.last_counts])
            torch.cuda.synchronize()
            assert len(got[0]) == len(got[1])
            for a, b in zip(*got):
                assert a.dtype == b.dtype and torch.equal(a, b), (n, norm)


@pytest.mark.parametrize("E,I,S,fits", [(64, 128, 30, True), (64, 128, 31, False), (64, 256, 32, False), (33, 128, 30, True), (256, 128, 24, True),
                                        (256, 128, 25, False), (65, 128, 29, True), (65, 128, 30, False), (40, 128, 1, True)])
@pytest.mark.parametrize("fp8", [False, True])
def test_shared_expert_next_to_the_router(E, I, S, fits, fp8):
    """The shared expert's gate and up projection runs in the router's launch while that has at most one workgroup per CU (256): 16 columns
    each, behind 8 per 32 experts; and from a hidden size of 2048 on, 6144 with fp8 weights.  On both sides of these lines the bits are those
    of the stage-by-stage path, also from a graph."""
    import ctypes
    from moe_gen_amd import _native as N, synthetic
    from moe_gen_amd.block import StageTimer
    inter, line = S * I, 6144 if fp8 else 2048
    first = ctypes.CDLL(N.LIB_PATH)["_ZN3moe18layer_shared_firstERK13moe_mlp_groupS2_i"]
    first.restype = ctypes.c_bool

    def group(n_experts, width, rows):                       # (the rule reads no memory)
        g = N.MlpGroup()
        for f in ("x", "w_gate", "w_up", "w_down", "s_gate", "s_up", "s_down", "offsets", "act", "y"):
            setattr(g, f, 256)
        g.x_rows, g.n_rows, g.n_experts, g.inter, g.fp8, g.max_rows = 2, rows, n_experts, width, int(fp8), 2
        return g
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        for h, pays in ((line, True), (line - 128, False), (2 * line, True)):
            assert first(ctypes.byref(group(E, I, 4)), ctypes.byref(group(1, inter, 2)), h) == (fits and pays), h
    w = synthetic.WORKLOADS["deepseek_v2_lite"].scaled(n=17, h=line, I=I, S=S, seq=17, E=E, k=2, n_group=1, topk_group=1, fp8=fp8)
    blk = synthetic.build_block(w, device="cuda")
    xs = synthetic.hidden_states(w, "cpu").cuda()
    for n in (1, 2, 16, 17):
        print(f"shared expert next to the router E={E} shared={inter} fp8={fp8} n={n}", flush=True)
        x = xs[:, :n].contiguous()
        blk.stage_timer = StageTimer()
        want = blk(x).clone()
        blk.stage_timer = None
        assert torch.equal(blk(x), want)
        if n != 2:
            continue
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = blk(x)
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)
            assert torch.equal(blk(x), want)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("name,E,k,h", [("deepseek_v2_lite", 64, 6, 1024), ("deepseek_v2_lite", 17, 3, 576), ("deepseek_v3_w8a16", 256, 8, 384),
                                        ("mixtral_8x7b", 8, 2, 512), ("mixtral_8x7b", 8, 8, 256), ("deepseek_v2_lite", 33, 16, 256),
                                        ("mixtral_8x22b", 32, 16, 192)])
def test_few_tokens_in_fewer_launches(name, E, k, h, fp8):
    """Calls whose router also sorts, whose down projection has 16 columns a wave and also combines (a counter per column
    tile, set anew by every call), and their neighbours in tokens and columns, h no multiple of 128 and E no power of two
    among them: bit for bit the stage-by-stage path; again on the same buffers, and replayed from a graph."""
    from moe_gen_amd import norm_moe_residual, synthetic
    from moe_gen_amd.block import StageTimer
    group = dict(n_group=1, topk_group=1) if name == "deepseek_v2_lite" else dict(n_group=4, topk_group=2) if name == "deepseek_v3_w8a16" else {}
    w = synthetic.WORKLOADS[name].scaled(n=17, h=h, I=256, seq=17, E=E, k=k, fp8=fp8, **group)
    if fp8 and h % 128:
        pytest.skip("fp8 weights come in blocks of 128")
    blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
    xs = synthetic.hidden_states(w, "cpu").cuda()
    nw = (1 + 0.1 * torch.randn(h, generator=torch.Generator().manual_seed(1))).to(torch.bfloat16).cuda()
    for n in (1, 2, 4, 5, 8, 9, 16, 17):
        x = xs[:, :n].contiguous()
        for norm in (False, True):
            print(f"few tokens {name} E={E} k={k} h={h} fp8={fp8} n={n} norm={norm}", flush=True)
            def run():
                res = norm_moe_residual(blk, x, nw) if norm else blk(x)
                res = res if isinstance(res, tuple) else (res,)
                return [*res, blk.last_topk_idx, blk.last_topk_weight, blk.last_counts]
            blk.stage_timer = StageTimer()
            want = [t.clone() for t in run()]
            blk.stage_timer = None
            for _ in range(3):
                for a, b in zip(run(), want):
                    assert a.dtype == b.dtype and torch.equal(a, b), (n, norm)
            if n != 1:
                continue
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                got = run()
            for _ in range(3):
                graph.replay()
                torch.cuda.synchronize()
                for a, b in zip(got, want):
                    assert torch.equal(a, b), norm


@pytest.mark.parametrize("fp8", [False, True])
def test_dense_mlp_sees_replaced_weights_and_a_copied_block_its_own(fp8):
    """A dense MLP whose up projection (fp8: or its block scales) is replaced between two calls computes with the new one,
    and a deep copy of a block that has run gives the block's results after the block's weights are gone."""
    import copy
    from moe_gen_amd import synthetic
    w = synthetic.WORKLOADS["deepseek_v3_w8a16" if fp8 else "deepseek_v2_lite"].scaled(n=24, h=512, I=256, seq=24)
    blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
    x = synthetic.hidden_states(w, "cpu").cuda()
    mlp = blk.shared_experts
    first = mlp(x)
    lin = mlp.up_proj
    name = "weight_scale_inv" if fp8 else "weight"
    setattr(lin, name, torch.nn.Parameter(getattr(lin, name).data * 2, requires_grad=False))
    second = mlp(x)
    assert torch.equal(second, 2 * first)                  # (a power of two: every product, sum and rounding scales)
    out = blk(x)
    twin = copy.deepcopy(blk)
    for ex in blk.experts:
        for lin in (ex.gate_proj, ex.up_proj, ex.down_proj):
            lin.weight.data.view(torch.uint8).zero_()
    assert torch.equal(twin(x), out)


@pytest.mark.parametrize("E", [1, 8])
def test_layer_call_reads_only_the_weights_of_its_groups(E):
    """The other fields of a layer call's groups may hold anything.  The sizes are ones at which an fp8 MLP with a
    workspace of its own cuts its down projection into slices of k (one expert, 4096 inner columns, few rows): a buffer
    offered in those fields stays as it was, and the output is that of a call without one."""
    from moe_gen_amd import synthetic
    w = synthetic.WORKLOADS["deepseek_v2_lite"].scaled(n=16, h=512, I=4096, S=1, seq=16, E=E, k=1, fp8=True)
    blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
    blk.join_shared = False
    x = synthetic.hidden_states(w, "cpu").cuda()
    print(f"layer call with a foreign workspace E={E}", flush=True)
    want = blk(x)
    sentinel = torch.full((64 * 2 ** 20,), 7, dtype=torch.uint8, device="cuda")
    for tables in (blk._moe_cache["routed"]["ptrs"], blk._moe_cache["shared"]["ptrs"]):
        tables.weights.workspace, tables.weights.workspace_bytes = sentinel.data_ptr(), sentinel.numel()
    assert torch.equal(blk(x), want)
    assert (sentinel == 7).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("path", ["layer", "stages"])
def test_layer_sees_every_replaced_weight_and_scale(fp8, path):
    """A block that has run, and then gets a middle expert's up projection, the shared expert's up projection (fp8: and one
    expert's block scales) anew, computes what a block that never ran before computes with them."""
    from moe_gen_amd import synthetic
    from moe_gen_amd.block import StageTimer
    w = synthetic.WORKLOADS["deepseek_v3_w8a16" if fp8 else "deepseek_v2_lite"].scaled(n=96, h=512, I=256, seq=96)
    x = synthetic.hidden_states(w, "cpu").cuda()
    print(f"replaced weights fp8={fp8} {path}", flush=True)

    def block():
        b = synthetic.build_block(w, device="cuda", gen_device="cpu")
        b.stage_timer = StageTimer() if path == "stages" else None
        return b

    def replace(b, what):
        ex = b.shared_experts if what == "shared" else b.experts[len(b.experts) // 2]
        lin, name = (ex.down_proj, "weight_scale_inv") if what == "scale" else (ex.up_proj, "weight")
        old = getattr(lin, name).data
        new = old * 2 if what == "scale" else old.flip(0).contiguous() if not fp8 else old.view(torch.uint8).flip(0).contiguous().view(old.dtype)
        if what == "data":
            getattr(lin, name).data = new
        else:
            setattr(lin, name, torch.nn.Parameter(new, requires_grad=False))

    ran, last = block(), None
    last = ran(x).clone()
    done = []
    for what in ["weight", "shared", "data"] + (["scale"] if fp8 else []):
        replace(ran, what)
        done.append(what)
        got, fresh = ran(x), block()
        for d in done:
            replace(fresh, d)
        assert torch.equal(got, fresh(x)), what
        assert not torch.equal(got, last), what
        last = got.clone()


def test_first_call_of_a_block_on_another_stream_finds_its_tables():
    """A block whose first call runs on one stream and whose next call follows at once on another: the tables that the
    first call made are there for both."""
    from moe_gen_amd import synthetic
    w = synthetic.WORKLOADS["deepseek_v3_w8a16"].scaled(n=48, h=512, I=256, seq=48)
    x = synthetic.hidden_states(w, "cpu").cuda()
    print("first call on a stream of its own", flush=True)
    want = synthetic.build_block(w, device="cuda", gen_device="cpu")(x).clone()
    busy = torch.randn(4096, 4096, device="cuda")
    for _ in range(3):
        blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
        streams = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        outs = []
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                if i == 0:                          # (the first stream is busy when its call comes, the second is not)
                    for _ in range(20):
                        busy = busy @ busy * 1e-3
                outs.append(blk(x))
        torch.cuda.synchronize()
        assert torch.equal(outs[0], want) and torch.equal(outs[1], want)


@pytest.mark.parametrize("name,n,E", [("deepseek_v2_lite", 1500, 64), ("deepseek_v2_lite", 700, 16), ("deepseek_v2_236b", 2000, 40),
                                      ("mixtral_8x7b", 600, 8), ("mixtral_8x22b", 1300, 8), ("deepseek_v3_w8a16", 1500, 64),
                                      ("deepseek_v3_w8a16", 600, 16)])
def test_claimed_tiles_give_the_bits_of_launched_ones(name, n, E):
    """Calls of both kinds of tiles: the layer call's workgroups claim the tiles that are not persistent ones from counters that the
    dispatch clears, the stage-by-stage path of an attached timer launches one for each.  Skewed counts, so that experts of every
    kind, pairs and last rounds in halves occur; again on other tokens, and in replays of a graph between eager calls."""
    from moe_gen_amd import synthetic
    from moe_gen_amd.block import StageTimer
    first = lambda r: r[0] if isinstance(r, tuple) else r
    w = synthetic.WORKLOADS[name].scaled(n=n, h=768, I=640, seq=n, E=E)
    print(f"claimed tiles {name} n={n} E={E}", flush=True)
    blk = synthetic.build_block(w, device="cuda", gen_device="cpu")
    x = synthetic.hidden_states(w, "cpu").cuda()
    more = [x, x.flip(-1).contiguous(), (0.5 * x).contiguous()]
    blk.stage_timer = StageTimer()
    want = [first(blk(v)).clone() for v in more]
    blk.stage_timer = None
    for rep in range(2):
        for v, y in zip(more, want):
            assert torch.equal(first(blk(v)), y), rep
    static = x.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        blk(static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = first(blk(static))
    for v, y in zip(more + more, want + want):
        static.copy_(v)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, y)
        assert torch.equal(first(blk(v)), y)
