"""GPU parity of the grouped SwiGLU GEMMs (bf16 and W8A16) and of the fp8 block dequantisation."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from util import bits, rel_max, rel_rms

pytestmark = pytest.mark.gpu

TOL = 2e-2     # max|y - y_ref| / max|y_ref| against the fp32 evaluation (bf16 inputs/weights)


def make_experts(E, h, I, fp8, seed):
    from moe_gen_amd.synthetic import quantize_fp8_block128
    g = torch.Generator().manual_seed(seed)
    mats = []
    for _ in range(E):
        one = []
        for shape in ((I, h), (I, h), (h, I)):
            m = torch.randn(shape, generator=g) * 0.05
            one.append(quantize_fp8_block128(m) if fp8 else m.to(torch.bfloat16))
        mats.append(one)
    return mats


def bits_t(t):
    return t.cpu().view(torch.int16)


def f32_of(m):
    if isinstance(m, tuple):
        return O.bf16_to_f32(O.dequant_block(bits(m[0]), m[1].numpy()))
    return O.bf16_to_f32(bits(m))


def run_case(E, h, I, counts, fp8, seed, use_row_map=False):
    from moe_gen_amd import ops
    counts = np.asarray(counts, np.int32)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n_rows = int(offsets[-1])
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(max(n_rows, 1), h, generator=g).to(torch.bfloat16)[:n_rows]
    mats = make_experts(E, h, I, fp8, seed + 1)
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    dm = [[dev(m) for m in one] for one in mats]
    if fp8:
        ptrs = ops.expert_pointers([o[0][0] for o in dm], [o[1][0] for o in dm], [o[2][0] for o in dm],
                                   [o[0][1] for o in dm], [o[1][1] for o in dm], [o[2][1] for o in dm])
    else:
        ptrs = ops.expert_pointers([o[0] for o in dm], [o[1] for o in dm], [o[2] for o in dm])
    off_d = torch.from_numpy(offsets).cuda()
    if use_row_map:
        rm = torch.randperm(n_rows, generator=g).to(torch.int32)
        xin = torch.empty_like(x)
        xin[rm.long()] = x                       # row r of the sorted matrix lives at xin[rm[r]]
        y = ops.grouped_swiglu(xin.cuda(), rm.cuda(), ptrs, off_d, n_rows)
    else:
        y = ops.grouped_swiglu(x.cuda(), None, ptrs, off_d, n_rows)
    torch.cuda.synchronize()
    yf = O.bf16_to_f32(bits(y))
    xf = O.bf16_to_f32(bits(x))
    ref32 = np.zeros((n_rows, h), np.float32)
    refr = np.zeros((n_rows, h), np.float32)
    for e in range(E):
        a, b = offsets[e], offsets[e + 1]
        if b > a:
            wg, wu, wd = (f32_of(m) for m in mats[e])
            ref32[a:b] = O.mlp_f32(xf[a:b], wg, wu, wd)
            refr[a:b] = O.mlp_ref_rounding(xf[a:b], wg, wu, wd)
    return yf, ref32, refr


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("E,h,I,counts", [
    (1, 128, 128, [64]),
    (1, 256, 128, [300]),
    (4, 256, 384, [0, 1, 255, 257]),
    (8, 512, 256, [5, 0, 130, 64, 0, 0, 700, 31]),
    (3, 1024, 640, [1000, 3, 500]),
    (8, 256, 256, [3, 0, 40, 17, 0, 1, 64, 9]),        # every expert under a 64-row tile
    (6, 384, 128, [70, 2, 0, 33, 1, 5]),
    (2, 128, 128, [1, 0]),
    (4, 384, 256, [300, 500, 0, 260]),                 # 256-row tiles, ragged last N tile of the down projection
    (32, 256, 256, [3000] + [2] * 31),                 # one hot expert under a low mean: 24 tiles of 128 rows among 64-row tiles
])
def test_grouped_swiglu_vs_oracle(fp8, E, h, I, counts):
    print(f"grouped fp8={fp8} E={E} h={h} I={I} counts={counts}", flush=True)
    y, ref32, refr = run_case(E, h, I, counts, fp8, seed=17)
    assert np.isfinite(y).all()
    e32, er = rel_max(y, ref32), rel_max(y, refr)
    print(f"  max-rel vs fp32 {e32:.3e}  vs reference-rounding {er:.3e}  rms {rel_rms(y, ref32):.3e}", flush=True)
    assert e32 <= TOL
    assert er <= TOL


@pytest.mark.parametrize("E,h,I,counts", [
    (1, 192, 320, [300]),            # three 128-row tiles
    (2, 192, 320, [100, 30]),        # a 128-row tile and a 64-row tile
    (4, 320, 192, [5, 9, 0, 20]),    # 64-row tiles
    (1, 64, 64, [70]),               # a single k-stage
    (4, 384, 320, [300, 500, 0, 260]),   # gate/up: even stage count, ragged last N tile; down: 5 stages
])
def test_grouped_odd_stage_counts(E, h, I, counts):
    """bf16 sizes whose K is an odd multiple of 64: the k loop is unrolled by two and ends in a
    single-stage tail (fp8 sizes are multiples of 128 and never do)."""
    print(f"grouped odd stages E={E} h={h} I={I} counts={counts}", flush=True)
    y, ref32, _ = run_case(E, h, I, counts, False, seed=29)
    assert np.isfinite(y).all() and rel_max(y, ref32) <= TOL


@pytest.mark.parametrize("fp8", [False, True])
def test_tile_height_follows_the_expert(fp8):
    """One launch of the one-workgroup-per-tile kernel alone (mean rows per expert below 128) with experts on both
    sides of every tile-height boundary: a 64-row tile up to 64 rows, one 128-row tile up to 128, one 192-row
    tile up to 192, several 128-row tiles above (those share their weights through one XCD's L2).
    Against the oracle, and an expert's rows bit-for-bit against a launch that holds this expert alone."""
    from moe_gen_amd import ops
    E, h, I = 16, 512, 384
    counts = [3, 64, 65, 128, 129, 300, 0, 17, 257, 1, 192, 193, 1, 2, 0, 5]
    print(f"tile heights fp8={fp8} counts={counts}", flush=True)
    y, ref32, refr = run_case(E, h, I, counts, fp8, seed=61, use_row_map=True)
    assert np.isfinite(y).all() and rel_max(y, ref32) <= TOL and rel_max(y, refr) <= TOL
    # the same experts one at a time (run_case draws x and the weights from the seed alone)
    offsets = np.concatenate([[0], np.cumsum(counts)])
    mats = make_experts(E, h, I, fp8, 62)
    g = torch.Generator().manual_seed(61)
    x = torch.randn(int(offsets[-1]), h, generator=g).to(torch.bfloat16)
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    for e in (1, 2):                                     # 64 and 65 rows: alone they are below a mean of 128 too
        one = [dev(m) for m in mats[e]]
        if fp8:
            ptrs = ops.expert_pointers([one[0][0]], [one[1][0]], [one[2][0]], [one[0][1]], [one[1][1]], [one[2][1]])
        else:
            ptrs = ops.expert_pointers([one[0]], [one[1]], [one[2]])
        a, b = int(offsets[e]), int(offsets[e + 1])
        ye = ops.grouped_swiglu(x[a:b].cuda(), None, ptrs, torch.tensor([0, b - a], dtype=torch.int32, device="cuda"), b - a)
        torch.cuda.synchronize()
        assert np.array_equal(O.bf16_to_f32(bits(ye)), y[a:b]), f"expert {e} differs from its launch alone"


@pytest.mark.parametrize("fp8", [False, True])
def test_experts_split_between_the_two_kernels(fp8):
    """From a mean of 128 rows per expert a launch has both kinds of tiles and every expert goes by its own count.  bf16
    weights: up to 192 rows one tile of a workgroup of its own, more 256-row tiles of the persistent workgroups.
    fp8 weights: the persistent tile space holds an expert's full 256-row tiles, and what they leave over is a tile
    of one workgroup if it is at most 192 rows (300 = 256 + 44, 640 = 512 + 128, 700 = 512 + 188, 512 leaves nothing,
    2000 = 1792 + 208 stays whole).  (At this size the tile space is a short last round, which runs as half tiles of one workgroup.)
    Against the oracle, and every expert's rows bit-for-bit against a call that holds this expert alone, whichever
    kernel and tile its rows fall to there.  (A lone call below a mean of 128 has one-workgroup tiles
    alone, which then walk k from other stages than a call of both kinds, and is left out.)"""
    from moe_gen_amd import ops
    E, h, I = 13, 256, 384
    counts = [700, 3, 192, 193, 64, 0, 129, 2000, 128, 300, 512, 640, 1600]
    print(f"two kernels fp8={fp8} counts={counts}", flush=True)
    y, ref32, refr = run_case(E, h, I, counts, fp8, seed=71, use_row_map=True)
    assert np.isfinite(y).all() and rel_max(y, ref32) <= TOL and rel_max(y, refr) <= TOL
    offsets = np.concatenate([[0], np.cumsum(counts)])
    mats = make_experts(E, h, I, fp8, 72)
    g = torch.Generator().manual_seed(71)
    x = torch.randn(int(offsets[-1]), h, generator=g).to(torch.bfloat16)
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    for e in range(E):
        a, b = int(offsets[e]), int(offsets[e + 1])
        if b - a < 128:
            continue
        one = [dev(m) for m in mats[e]]
        if fp8:
            ptrs = ops.expert_pointers([one[0][0]], [one[1][0]], [one[2][0]], [one[0][1]], [one[1][1]], [one[2][1]])
        else:
            ptrs = ops.expert_pointers([one[0]], [one[1]], [one[2]])
        ye = ops.grouped_swiglu(x[a:b].cuda(), None, ptrs, torch.tensor([0, b - a], dtype=torch.int32, device="cuda"), b - a)
        torch.cuda.synchronize()
        assert np.array_equal(O.bf16_to_f32(bits(ye)), y[a:b]), f"expert {e} ({b - a} rows) differs from its call alone"


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("I,counts", [(1280, [700, 520, 300, 1300, 90]),      # 120 tiles next to 30 of one workgroup (fp8: 100 and 50, halves)
                                      (2048, [700, 520, 300, 1300, 90]),      # 192 and 48 (160 and 80)
                                      (2560, [700, 520, 300, 1300, 90]),      # 240 and 60 (200 and 100, tall: halves)
                                      (1664, [2100, 2300, 2500, 1500, 10]),   # a round, and 186 next to 13 (173, 26)
                                      (896, [700, 520, 300, 90]),             # 42 and 21: halves (35 and 28: halves)
                                      (3072, [700, 520, 300, 160, 170, 180, 90])])      # 144 and 144, tall: halves (120 and 168, too)
def test_rounds_of_the_persistent_kernel_and_its_last_tiles(fp8, I, counts):
    """The persistent workgroups (one per CU) take whole rounds of 256 tiles, the last of them on fewer CUs next to tiles of one workgroup; a
    partial round that leaves too few CUs to these, or costs more than its 128-row halves next to them, becomes such halves.  In the
    comments: the gate and up projection's tiles on 256 CUs, kept unless they say halves, with bf16 (fp8) weights.  The down
    projections of these cases have a few dozen tiles, all of them half tiles.  Against the oracle."""
    from moe_gen_amd import ops
    E, h = len(counts), 256
    print(f"rounds fp8={fp8} I={I} counts={counts}", flush=True)
    y, ref32, refr = run_case(E, h, I, counts, fp8, seed=91, use_row_map=True)
    assert np.isfinite(y).all() and rel_max(y, ref32) <= TOL and rel_max(y, refr) <= TOL


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("h,I", [(128, 1280), (256, 1280), (384, 1280), (512, 1280), (2560, 128), (2688, 256), (2560, 384)])
def test_persistent_kernel_turns_between_tiles_at_short_k(fp8, h, I):
    """More tiles than CUs at 2, 4, 6 and 8 stages of 64 k (gate/up: h; down projection: I), so that workgroups go on from
    tile to tile where a tile's first pair of stages is also its last, or its last but one; 2688: half a column tile at
    the end.  Ragged row counts, gathered rows.  Against the oracle."""
    print(f"turns fp8={fp8} h={h} I={I}", flush=True)
    y, ref32, refr = run_case(5, h, I, [1100, 2047, 1500, 1793, 1750], fp8, seed=97, use_row_map=True)
    assert np.isfinite(y).all() and rel_max(y, ref32) <= TOL and rel_max(y, refr) <= TOL


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("counts", [[300, 640, 129, 70], [2100, 1700], [40, 3, 77]])
def test_a_row_does_not_depend_on_its_place_in_its_expert(fp8, counts):
    """The same rows in another order within every expert give the same output rows, bit for bit, whichever kernel
    and tile a row falls to (with fp8 weights the rows past an expert's last full 256-row tile are computed by the
    other kernel: 300 = 256 + 44)."""
    from moe_gen_amd import ops
    E, h, I = len(counts), 256, 384
    print(f"row order fp8={fp8} counts={counts}", flush=True)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = int(offsets[-1])
    g = torch.Generator().manual_seed(83)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    perm = torch.cat([int(offsets[e]) + torch.randperm(counts[e], generator=g) for e in range(E)])
    mats = make_experts(E, h, I, fp8, 84)
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    dm = [[dev(m) for m in one] for one in mats]
    if fp8:
        ptrs = ops.expert_pointers([o[0][0] for o in dm], [o[1][0] for o in dm], [o[2][0] for o in dm],
                                   [o[0][1] for o in dm], [o[1][1] for o in dm], [o[2][1] for o in dm])
    else:
        ptrs = ops.expert_pointers([o[0] for o in dm], [o[1] for o in dm], [o[2] for o in dm])
    off_d = torch.from_numpy(offsets).cuda()
    y1 = ops.grouped_swiglu(x.cuda(), None, ptrs, off_d, n)
    y2 = ops.grouped_swiglu(x[perm].cuda(), None, ptrs, off_d, n)
    y3 = ops.grouped_swiglu(x.cuda(), perm.to(torch.int32).cuda(), ptrs, off_d, n)       # the same through a row map
    torch.cuda.synchronize()
    assert torch.equal(y2, y1[perm.cuda()])
    assert torch.equal(y3, y2)


@pytest.mark.parametrize("h,I", [(512, 384), (2048, 1024)])
def test_fp8_weight_streamer_rows_do_not_depend_on_the_tile(h, I):
    """fp8 experts of up to 64 rows, in a call below a mean of 128 rows per expert, go through the weight streamer
    (weights by DMA as fp8, one 16/32/48/64-row body per expert).  Eight experts that share one set of weights and
    hold 5 ... 64 rows, each starting with the same five rows: those rows come out bit-identical from every body,
    against the oracle within the layer bound, and the call gives the same bits every time it runs (the buffers of
    a tile are refilled while other waves still multiply; a missing wait shows as run-to-run differences)."""
    from moe_gen_amd import ops
    counts = [5, 16, 17, 32, 33, 48, 49, 64]
    E = len(counts)
    print(f"fp8 streamer h={h} I={I} counts={counts}", flush=True)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = int(offsets[-1])
    g = torch.Generator().manual_seed(97)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    for e in range(1, E):
        x[offsets[e]:offsets[e] + 5] = x[:5]
    one = make_experts(1, h, I, True, 98)[0]
    dm = [tuple(t.cuda() for t in m) for m in one]
    ptrs = ops.expert_pointers([dm[0][0]] * E, [dm[1][0]] * E, [dm[2][0]] * E, [dm[0][1]] * E, [dm[1][1]] * E, [dm[2][1]] * E)
    off_d = torch.from_numpy(offsets).cuda()
    xd = x.cuda()
    ys = [ops.grouped_swiglu(xd, None, ptrs, off_d, n).clone() for _ in range(8)]
    torch.cuda.synchronize()
    for rep in range(1, 8):
        assert torch.equal(ys[rep], ys[0]), f"call {rep} differs from call 0"
    for e in range(1, E):
        assert torch.equal(ys[0][offsets[e]:offsets[e] + 5], ys[0][:5]), f"expert {e} ({counts[e]} rows)"
    wg, wu, wd = (f32_of(m) for m in one)
    ref = O.mlp_f32(O.bf16_to_f32(bits(x)), wg, wu, wd)
    assert rel_max(O.bf16_to_f32(bits(ys[0])), ref) <= TOL


@pytest.mark.parametrize("counts", [
    [5, 16, 17, 32, 33, 64, 65, 80, 81, 96, 112, 128, 129, 144, 160, 176, 192] + [5] * 12,     # mean 59: one kernel
    [192, 181, 170, 160, 150, 140, 130, 129, 257, 300, 384, 600, 5]])                          # mean 215: both kinds of tiles
def test_bf16_weight_streamer_rows_do_not_depend_on_the_tile(counts):
    """bf16 experts of up to 192 rows (and the halves of one of 257 ... 384) go through the bf16 weight streamer: one
    body per number of 16-row groups, two wave layouts (up to 64 rows, above), weights and token rows by DMA.
    Experts that share one set of weights and start with the same five rows: those rows come out bit-identical from
    every body -- in the second list also from the persistent kernel (600 rows) and the halves of a pair --, against
    the oracle within the layer bound, and the call gives the same bits every time it runs (a tile's buffers are
    refilled while other waves still multiply; a missing wait shows as run-to-run differences)."""
    from moe_gen_amd import ops
    E, h, I = len(counts), 448, 640            # 7 / 10 stages of 64 k: 1 / 4 stages after the loop unrolled by six
    print(f"bf16 streamer counts={counts}", flush=True)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = int(offsets[-1])
    g = torch.Generator().manual_seed(197)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    for e in range(1, E):
        x[offsets[e]:offsets[e] + 5] = x[:5]
    one = make_experts(1, h, I, False, 198)[0]
    dm = [m.cuda() for m in one]
    ptrs = ops.expert_pointers([dm[0]] * E, [dm[1]] * E, [dm[2]] * E)
    off_d = torch.from_numpy(offsets).cuda()
    xd = x.cuda()
    ys = [ops.grouped_swiglu(xd, None, ptrs, off_d, n).clone() for _ in range(8)]
    torch.cuda.synchronize()
    for rep in range(1, 8):
        assert torch.equal(ys[rep], ys[0]), f"call {rep} differs from call 0"
    for e in range(1, E):
        assert torch.equal(ys[0][offsets[e]:offsets[e] + 5], ys[0][:5]), f"expert {e} ({counts[e]} rows)"
    wg, wu, wd = (f32_of(m) for m in one)
    ref = O.mlp_f32(O.bf16_to_f32(bits(x)), wg, wu, wd)
    assert rel_max(O.bf16_to_f32(bits(ys[0])), ref) <= TOL


def test_bf16_rows_do_not_depend_on_the_call():
    """With bf16 weights every path adds a column's products in one order, in every call: the same 40
    rows come out bit-identical from a call that the one-workgroup-per-tile kernel serves alone (one expert of 40
    rows) and from a call with both kinds of tiles, where they open an expert of 600 rows (persistent kernel), one
    of 150 (a single tile) and one of 300 (the first of two tiles side by side)."""
    from moe_gen_amd import ops
    h, I, r = 512, 768, 40
    g = torch.Generator().manual_seed(211)
    rows = torch.randn(r, h, generator=g).to(torch.bfloat16)
    one = make_experts(1, h, I, False, 212)[0]
    dm = [m.cuda() for m in one]
    small = ops.grouped_swiglu(rows.cuda(), None, ops.expert_pointers([dm[0]], [dm[1]], [dm[2]]),
                               torch.tensor([0, r], dtype=torch.int32).cuda(), r)
    counts = [600, 150, 300]
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = int(offsets[-1])
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    for e in range(3):
        x[offsets[e]:offsets[e] + r] = rows
    big = ops.grouped_swiglu(x.cuda(), None, ops.expert_pointers([dm[0]] * 3, [dm[1]] * 3, [dm[2]] * 3),
                             torch.from_numpy(offsets).cuda(), n)
    torch.cuda.synchronize()
    for e in range(3):
        assert torch.equal(big[offsets[e]:offsets[e] + r], small), f"expert of {counts[e]} rows"


@pytest.mark.parametrize("h,I", [(448, 512), (576, 640), (704, 384), (384, 448)])   # 7/8, 9/10, 11/6, 6/7 stages of 64 k
def test_bf16_weight_streamer_shapes_and_gather(h, I):
    """The bf16 weight streamer on every token-group count and both sides of each boundary, with stage counts that
    leave 0 ... 5 stages after its loop unrolled by six, rows gathered through row_map, and last N tiles that are
    ragged (down projection: h = 448, 576, 704 of 256 columns; gate/up: I = 448 of 128)."""
    counts = [16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129, 144, 145, 160, 161, 176, 177, 192,
              1, 0, 15, 31, 47, 63] + [2] * 20
    print(f"bf16 streamer shapes h={h} I={I} counts={counts}", flush=True)
    y, ref32, refr = run_case(len(counts), h, I, counts, False, seed=161, use_row_map=True)
    assert np.isfinite(y).all()
    assert rel_max(y, ref32) <= TOL and rel_max(y, refr) <= TOL


@pytest.mark.parametrize("counts", [
    [129, 144, 145, 160, 176, 177, 192, 400, 600, 320, 449, 70],     # mean 255: both kinds of tiles; 400 = 256 + 144 left over
    [129, 150, 192, 170, 64, 65] + [5] * 20])                         # mean 35: the one-workgroup-per-tile kernel alone
@pytest.mark.parametrize("h,I", [(640, 384), (1024, 896)])            # 5 / 3 and 8 / 7 blocks of 128 k (odd and even counts)
def test_fp8_weight_streamer_tiles_of_129_to_192_rows(counts, h, I):
    """fp8 tiles of 129 to 192 rows -- experts of that size, and what the full 256-row tiles of a larger one leave over
    -- run on the streamer form with two weight buffers and 24 KiB of token rows per half.  Experts that share one set
    of weights and start with the same five rows: those rows come out bit-identical from every tile height, in the
    first list also from the persistent kernel (600 = 2 x 256 + 88 rows, 449 = 256 + 193) and the 128-row form (320 =
    256 + 64); the call gives the same bits every time, and the rows are within the layer bound of the oracle."""
    from moe_gen_amd import ops
    E = len(counts)
    print(f"fp8 streamer 129-192 h={h} I={I} counts={counts}", flush=True)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = int(offsets[-1])
    g = torch.Generator().manual_seed(297)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    for e in range(1, E):
        x[offsets[e]:offsets[e] + 5] = x[:5]
    one = make_experts(1, h, I, True, 298)[0]
    dm = [tuple(t.cuda() for t in m) for m in one]
    ptrs = ops.expert_pointers([dm[0][0]] * E, [dm[1][0]] * E, [dm[2][0]] * E, [dm[0][1]] * E, [dm[1][1]] * E, [dm[2][1]] * E)
    off_d = torch.from_numpy(offsets).cuda()
    xd = x.cuda()
    ys = [ops.grouped_swiglu(xd, None, ptrs, off_d, n).clone() for _ in range(6)]
    rm = torch.randperm(n, generator=g).to(torch.int32)
    xin = torch.empty_like(x)
    xin[rm.long()] = x
    y_map = ops.grouped_swiglu(xin.cuda(), rm.cuda(), ptrs, off_d, n)       # the same rows gathered through a row map
    torch.cuda.synchronize()
    for rep in range(1, 6):
        assert torch.equal(ys[rep], ys[0]), f"call {rep} differs from call 0"
    assert torch.equal(y_map, ys[0])
    alone = n // E < 128
    for e in range(1, E):
        if alone and counts[e] <= 64:
            continue        # (alone, up to 64 rows: the streamer form with its own order of summation)
        assert torch.equal(ys[0][offsets[e]:offsets[e] + 5], ys[0][:5]), f"expert {e} ({counts[e]} rows)"
    wg, wu, wd = (f32_of(m) for m in one)
    ref = O.mlp_f32(O.bf16_to_f32(bits(x)), wg, wu, wd)
    assert rel_max(O.bf16_to_f32(bits(ys[0])), ref) <= TOL


@pytest.mark.parametrize("more", [[], [1100]])      # the tile kernel alone; with the persistent kernel next to it
@pytest.mark.parametrize("h,I", [(128, 384), (256, 512), (384, 128), (640, 256)])     # 1 ... 5 blocks of 128 k
def test_fp8_weight_streamer_every_tile_height(h, I, more):
    """Tiles of 1 to 12 groups of 16 rows, first and last row counts of a group, at block counts around the three that a turn of
    the k loop takes.  Against the oracle."""
    counts = [16, 17, 33, 49, 65, 80, 81, 96, 97, 112, 113, 128, 129, 144, 145, 160, 161, 176, 177, 192] + more
    print(f"tile heights h={h} I={I} more={more}", flush=True)
    y, ref32, refr = run_case(len(counts), h, I, counts, True, seed=67, use_row_map=True)
    assert np.isfinite(y).all() and rel_max(y, ref32) <= TOL and rel_max(y, refr) <= TOL


@pytest.mark.parametrize("h,I", [(512, 640), (640, 896), (896, 512)])      # 4 / 5 / 7 blocks of 128 k (gate/up), 5 / 7 / 4 (down)
def test_fp8_weight_streamer_shapes_and_gather(h, I):
    """The fp8 weight streamer on every token-group count and both sides of each boundary, with block counts that
    leave 0, 1 and 2 iterations after its loop unrolled by three, rows gathered through row_map, and a down
    projection whose last N tile is ragged (h = 640, 896)."""
    counts = [16, 17, 32, 33, 48, 49, 64, 1, 0, 15, 31, 47, 63]
    print(f"streamer shapes h={h} I={I} counts={counts}", flush=True)
    y, ref32, refr = run_case(len(counts), h, I, counts, True, seed=61, use_row_map=True)
    assert np.isfinite(y).all()
    assert rel_max(y, ref32) <= TOL and rel_max(y, refr) <= TOL


@pytest.mark.parametrize("fp8", [False, True])
def test_weight_streamer_row_outside_x_reads_zeros(fp8):
    """A row_map entry outside x is a row of zeros for the weight streamers too (their token DMA goes through a
    bounds-checked descriptor; such a row and the rows past an expert's last cost no memory request), and its
    neighbours are untouched: the other rows' bits equal those of a call with valid entries only."""
    from moe_gen_amd import ops
    E, h, I, per = 6, 512, 384, 20
    n = E * per
    mats = make_experts(E, h, I, fp8, 5)
    if fp8:
        dm = [[tuple(t.cuda() for t in m) for m in one] for one in mats]
        ptrs = ops.expert_pointers([o[0][0] for o in dm], [o[1][0] for o in dm], [o[2][0] for o in dm],
                                   [o[0][1] for o in dm], [o[1][1] for o in dm], [o[2][1] for o in dm])
    else:
        dm = [[m.cuda() for m in one] for one in mats]
        ptrs = ops.expert_pointers([o[0] for o in dm], [o[1] for o in dm], [o[2] for o in dm])
    x = torch.randn(n, h, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).cuda()
    off = torch.arange(0, n + 1, per, dtype=torch.int32).cuda()
    rm = torch.arange(n, dtype=torch.int32)
    good = ops.grouped_swiglu(x, rm.cuda(), ptrs, off, n)
    bad = rm.clone()
    for r, v in ((7, n), (45, -1), (119, 2**31 - 1)):
        bad[r] = v
    got = ops.grouped_swiglu(x, bad.cuda(), ptrs, off, n)
    torch.cuda.synchronize()
    keep = torch.ones(n, dtype=torch.bool)
    keep[[7, 45, 119]] = False
    assert torch.equal(bits_t(got)[keep], bits_t(good)[keep])
    assert (got[~keep.cuda()].float() == 0).all()           # SwiGLU of a zero row is zero, and so is its down projection


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("E,mean", [(700, 3), (1024, 2), (600, 200), (400, 200)])
def test_grouped_many_experts(fp8, E, mean):
    """More experts than threads in a workgroup (the M-tile prefix scan takes two passes), up to the
    maximum of 1024, with empty experts sprinkled in; the last two cases have about 200 rows per expert (400
    experts: the persistent kernel with its per-expert tables in LDS; 600: one workgroup per tile, two
    128-row tiles for most experts)."""
    print(f"grouped many experts fp8={fp8} E={E} mean={mean}", flush=True)
    rng = np.random.default_rng(E)
    counts = rng.poisson(mean, E)
    counts[::7] = 0
    y, ref32, _ = run_case(E, 128, 128, counts, fp8, seed=5)
    assert np.isfinite(y).all() and rel_max(y, ref32) <= TOL


def test_grouped_too_many_experts_is_an_error():
    from moe_gen_amd import ops
    E = 1025
    w = torch.zeros(128, 128, dtype=torch.bfloat16, device="cuda")
    ptrs = ops.expert_pointers([w] * E, [w] * E, [w] * E)
    off = torch.zeros(E + 1, dtype=torch.int32, device="cuda")
    off[1:] = 4
    x = torch.zeros(4, 128, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="n_experts"):
        ops.grouped_swiglu(x, None, ptrs, off, 4)


@pytest.mark.parametrize("fp8", [False, True])
def test_grouped_more_tiles_than_cus(fp8):
    """808 gate/up tiles and 404 down tiles of 256 rows on 256 CUs: with fp8 weights every persistent
    workgroup hands its pipeline over from tile to tile (different experts, a ragged last tile, a
    10-row expert in between); rows are gathered through a row map."""
    print(f"grouped more tiles than CUs fp8={fp8}", flush=True)
    y, ref32, _ = run_case(4, 1024, 1024, [9000, 7000, 10, 9000], fp8, seed=31, use_row_map=True)
    assert np.isfinite(y).all()
    err = rel_max(y, ref32)
    print(f"  max-rel vs fp32 {err:.3e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("fp8", [False, True])
def test_grouped_swiglu_row_map(fp8):
    y, ref32, _ = run_case(4, 256, 256, [100, 0, 300, 77], fp8, seed=23, use_row_map=True)
    assert rel_max(y, ref32) <= TOL


def _one_expert(h, I, seed):
    from moe_gen_amd import ops
    g = torch.Generator().manual_seed(seed)
    ws = [(torch.randn(shape, generator=g) * 0.05).to(torch.bfloat16) for shape in ((I, h), (I, h), (h, I))]
    ptrs = ops.expert_pointers(*[[w.cuda()] for w in ws])
    return ws, ptrs


@pytest.mark.parametrize("h,I,n", [(256, 256, 600), (256, 8192, 1100), (192, 256, 600), (256, 256, 100)])
def test_row_map_entry_outside_x_reads_zeros(h, I, n):
    """A row_map entry beyond x_rows stands for a row of zeros (no fault), and every other row is unaffected: the
    persistent kernel fetches gathered rows through a buffer descriptor that ends with x (1100 rows x 64 N tiles:
    a round of its tiles and more), the other kernel checks the entry (600 rows: six tiles, the persistent kernel's
    short last round as half tiles; K = 192 and 100 rows: calls it serves alone)."""
    from moe_gen_amd import ops
    ws, ptrs = _one_expert(h, I, 41)
    g = torch.Generator().manual_seed(42)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    rm = torch.randperm(n, generator=g).to(torch.int32)
    bad = [3, n // 2 + 7, n - 1]
    rm_bad = rm.clone()
    rm_bad[bad] = torch.tensor([n, n + 5, 2 ** 20], dtype=torch.int32)
    off = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    y_ok = ops.grouped_swiglu(x.cuda(), rm.cuda(), ptrs, off, n)
    y_bad = ops.grouped_swiglu(x.cuda(), rm_bad.cuda(), ptrs, off, n)
    torch.cuda.synchronize()
    keep = np.ones(n, bool)
    keep[bad] = False
    assert np.array_equal(bits(y_ok)[keep], bits(y_bad)[keep])
    assert (y_bad[bad].float().cpu().numpy() == 0).all()        # silu(0) * 0 through the down projection


@pytest.mark.parametrize("fp8", [False, True])
def test_gathered_rows_of_an_input_beyond_4_gib(fp8):
    """Gathered rows are addressed with 32-bit byte offsets only while x is smaller than 4 GiB; a larger
    x takes the one-workgroup-per-tile kernel with 64-bit addresses (with fp8 weights its register-staged body: the
    weight streamers address rows through a 32-bit descriptor).  The rows used sit at both ends of x."""
    from moe_gen_amd import ops
    h, I, n = 2048, 256, 512
    x_rows = (1 << 32) // (h * 2) + 4096                          # 4 GiB + 16 MiB of bf16 rows
    if fp8:
        mats = make_experts(1, h, I, True, 43)[0]
        dm = [tuple(t.cuda() for t in m) for m in mats]
        ptrs = ops.expert_pointers([dm[0][0]], [dm[1][0]], [dm[2][0]], [dm[0][1]], [dm[1][1]], [dm[2][1]])
        wg, wu, wd = (f32_of(m) for m in mats)
    else:
        ws, ptrs = _one_expert(h, I, 43)
        wg, wu, wd = (O.bf16_to_f32(bits(w)) for w in ws)
    g = torch.Generator().manual_seed(44)
    rows = torch.randn(n, h, generator=g).to(torch.bfloat16)
    x = torch.zeros(x_rows, h, dtype=torch.bfloat16, device="cuda")
    where = torch.cat([torch.arange(n // 2), torch.arange(x_rows - n // 2, x_rows)]).to(torch.int32)
    where = where[torch.randperm(n, generator=g)]
    x[where.long().cuda()] = rows.cuda()
    off = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    y = ops.grouped_swiglu(x, where.cuda(), ptrs, off, n)
    y_ref = ops.grouped_swiglu(rows.cuda(), None, ptrs, off, n)   # the same rows, sorted: the persistent kernel
    torch.cuda.synchronize()
    del x
    ref32 = O.mlp_f32(O.bf16_to_f32(bits(rows)), wg, wu, wd)
    assert rel_max(O.bf16_to_f32(bits(y)), ref32) <= TOL
    assert rel_max(O.bf16_to_f32(bits(y_ref)), ref32) <= TOL


def test_gathered_rows_beyond_4_gib_at_every_tile_kind_bf16():
    """The register-staged body behind the bf16 weight streamer (4 GiB of gathered rows or more) takes what the
    streamer takes: single tiles of up to 192 rows (above 128 as two passes of 128 rows), the halves of an expert of
    257 to 384 rows, 128-row slices.  Experts that share one set of weights, rows gathered from both ends of a 4 GiB
    x: every row equals, bit for bit, what the same rows give sorted and through the streamer (one order of
    summation for every bf16 path)."""
    from moe_gen_amd import ops
    h, I = 2048, 256
    counts = [150, 192, 300, 40, 129, 70, 384, 500]
    E, n = len(counts), sum(counts)
    x_rows = (1 << 32) // (h * 2) + 4096                          # 4 GiB + 16 MiB of bf16 rows
    ws, _ = _one_expert(h, I, 47)
    dw = [w.cuda() for w in ws]
    ptrs = ops.expert_pointers([dw[0]] * E, [dw[1]] * E, [dw[2]] * E)
    g = torch.Generator().manual_seed(48)
    rows = torch.randn(n, h, generator=g).to(torch.bfloat16)
    x = torch.zeros(x_rows, h, dtype=torch.bfloat16, device="cuda")
    where = torch.cat([torch.arange(n // 2), torch.arange(x_rows - (n - n // 2), x_rows)]).to(torch.int32)
    where = where[torch.randperm(n, generator=g)]
    x[where.long().cuda()] = rows.cuda()
    off = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32, device="cuda")
    print(f"4 GiB gather, bf16, counts={counts}", flush=True)
    y = ops.grouped_swiglu(x, where.cuda(), ptrs, off, n)
    y_ref = ops.grouped_swiglu(rows.cuda(), None, ptrs, off, n)
    torch.cuda.synchronize()
    del x
    wg, wu, wd = (O.bf16_to_f32(bits(w)) for w in ws)
    assert rel_max(O.bf16_to_f32(bits(y_ref)), O.mlp_f32(O.bf16_to_f32(bits(rows)), wg, wu, wd)) <= TOL
    assert torch.equal(y, y_ref)


@pytest.mark.parametrize("fp8", [False, True])
def test_expert_sub_range_through_the_persistent_kernel(fp8):
    """A call on experts [1, 3) of four with absolute row offsets (weights handed out in waves): the rows
    of the other experts stay untouched, the range's rows match the call on all experts."""
    from moe_gen_amd import ops
    E, h, I = 4, 256, 256
    counts = np.array([300, 520, 260, 290], np.int32)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = int(offsets[-1])
    g = torch.Generator().manual_seed(47)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16).cuda()
    mats = make_experts(E, h, I, fp8, 48)
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    dm = [[dev(m) for m in one] for one in mats]

    def pointers(sel):
        if fp8:
            return ops.expert_pointers([dm[e][0][0] for e in sel], [dm[e][1][0] for e in sel], [dm[e][2][0] for e in sel],
                                       [dm[e][0][1] for e in sel], [dm[e][1][1] for e in sel], [dm[e][2][1] for e in sel])
        return ops.expert_pointers([dm[e][0] for e in sel], [dm[e][1] for e in sel], [dm[e][2] for e in sel])

    off_d = torch.from_numpy(offsets).cuda()
    y_all = ops.grouped_swiglu(x, None, pointers(range(E)), off_d, n)
    act = torch.zeros(n, I, dtype=torch.bfloat16, device="cuda")
    y = torch.full((n, h), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.grouped_swiglu(x, None, pointers([1, 2]), off_d[1:4].contiguous(), n, act, y,
                       rows_bound=int(offsets[3] - offsets[1]))
    torch.cuda.synchronize()
    a, b = int(offsets[1]), int(offsets[3])
    assert torch.equal(y[a:b], y_all[a:b])
    assert (y[:a] == 7.0).all() and (y[b:] == 7.0).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("E,h,I,counts", [
    (2, 128, 128, [300, 260]),                # two k-stages: the shortest pipeline the persistent kernel runs
    (2, 128, 384, [513, 256]),                # gate/up: 2 stages; down: 6; a tile of one row
    (3, 256, 128, [700, 0, 300]),             # down projection with 2 stages, an empty expert in between
    (512, 128, 128, [200] * 512),             # as many experts as the kernel keeps tables for
])
def test_persistent_kernel_corner_shapes(fp8, E, h, I, counts):
    """The 256-row persistent kernel (experts above 192 rows, K a multiple of 128) at the ends of what
    it accepts; rows gathered through a row map."""
    print(f"persistent corners fp8={fp8} E={E} h={h} I={I}", flush=True)
    y, ref32, _ = run_case(E, h, I, counts, fp8, seed=37, use_row_map=True)
    assert np.isfinite(y).all() and rel_max(y, ref32) <= TOL


EDGE_COUNTS = [0, 1, 17, 64, 65, 128, 129, 144, 145, 160, 161, 192, 193, 256, 257, 300, 384, 385, 449, 700]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("seed", range(10))
def test_grouped_seeded_mixtures(fp8, seed):
    """Seeded draws of expert count, sizes and per-expert rows from both sides of every tile-height and
    kernel boundary (64 / 128 / 144 / 160 / 192 / 256 / 384 rows), with and without a row map: whichever
    kernels and tile forms the launcher picks for the mixture, every row matches the oracle, and a second
    call returns the same bits."""
    rng = np.random.default_rng(1000 + seed)
    E = int(rng.choice([1, 2, 3, 5, 8, 13]))
    h, I = 128 * int(rng.integers(1, 6)), 128 * int(rng.integers(1, 6))
    kind = ["few", "middle", "edges", "many"][seed % 4]
    counts = {"few": rng.integers(0, 70, E), "middle": rng.integers(100, 400, E),
              "edges": rng.choice(EDGE_COUNTS, E), "many": rng.integers(300, 900, E)}[kind]
    counts = [int(c) for c in counts]
    if sum(counts) == 0:
        counts[0] = 33
    use_map = bool(rng.integers(0, 2))
    print(f"mixture fp8={fp8} seed={seed} E={E} h={h} I={I} {kind} row_map={use_map} counts={counts}", flush=True)
    y, ref32, refr = run_case(E, h, I, counts, fp8, seed=300 + seed, use_row_map=use_map)
    y2, _, _ = run_case(E, h, I, counts, fp8, seed=300 + seed, use_row_map=use_map)
    assert np.isfinite(y).all()
    assert rel_max(y, ref32) <= TOL and rel_max(y, refr) <= TOL
    assert np.array_equal(y, y2)


@pytest.mark.parametrize("n_src,n", [(300, 600), (60, 120)])
def test_row_map_may_repeat_rows(n_src, n):
    """Several sorted rows may name the same source row (a token routed to k experts).  Both launches of a case
    run the same kernel (the persistent kernel / one workgroup per tile): the two walk k from different stages
    and may differ in the last bit."""
    from moe_gen_amd import ops
    h, I = 256, 256
    ws, ptrs = _one_expert(h, I, 51)
    g = torch.Generator().manual_seed(52)
    x = torch.randn(n_src, h, generator=g).to(torch.bfloat16)
    rm = torch.randint(0, n_src, (n,), generator=g, dtype=torch.int32)
    off = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    y = ops.grouped_swiglu(x.cuda(), rm.cuda(), ptrs, off, n)
    y_src = ops.grouped_swiglu(x.cuda(), None, ptrs, torch.tensor([0, n_src], dtype=torch.int32, device="cuda"), n_src)
    torch.cuda.synchronize()
    wg, wu, wd = (O.bf16_to_f32(bits(w)) for w in ws)
    ref32 = O.mlp_f32(O.bf16_to_f32(bits(x)), wg, wu, wd)[rm.long().numpy()]
    assert rel_max(O.bf16_to_f32(bits(y)), ref32) <= TOL
    assert np.array_equal(bits(y), bits(y_src)[rm.long().numpy()])       # a row's result does not depend on its tile


def test_grouped_single_expert_is_plain_mlp():
    """E = 1 reduces to a dense SwiGLU MLP: compare with torch's own bf16 linear layers on the GPU."""
    from moe_gen_amd import DeepseekV3Config, DeepseekV3MLP
    cfg = DeepseekV3Config(hidden_size=512, intermediate_size=768)
    mlp = DeepseekV3MLP(cfg).cuda().to(torch.bfloat16)
    x = torch.randn(3, 70, 512, device="cuda").to(torch.bfloat16)
    y = mlp(x)
    F = torch.nn.functional
    with torch.no_grad():
        ref = F.linear(F.silu(F.linear(x, mlp.gate_proj.weight)) * F.linear(x, mlp.up_proj.weight), mlp.down_proj.weight)
    assert rel_max(y.float().cpu().numpy(), ref.float().cpu().numpy()) <= TOL


@pytest.mark.parametrize("rows,cols", [(128, 128), (130, 200), (1, 16), (257, 1000), (2048, 7168)])
def test_dequant_bit_exact(rows, cols):
    from moe_gen_amd import ops
    g = torch.Generator().manual_seed(rows * 31 + cols)
    q = torch.randint(0, 256, (rows, cols), generator=g, dtype=torch.uint8)
    q[(q & 0x7F) == 0x7F] = 0                   # NaN patterns carry no ordering of payload bits
    s = torch.rand((-(-rows // 128), -(-cols // 128)), generator=g) * 0.01 + 1e-4
    out = ops.dequant_fp8_block128(q.cuda().view(torch.float8_e4m3fn), s.cuda())
    torch.cuda.synchronize()
    ref = O.dequant_block(q.numpy(), s.numpy())
    assert np.array_equal(bits(out), ref)


def test_fp8_decode_table_on_device():
    """All 256 byte values with scale 1: the device conversion is OCP e4m3fn (max 448, no inf)."""
    from moe_gen_amd import ops
    q = torch.arange(256, dtype=torch.uint8).repeat(16).view(16, 256)
    s = torch.ones((1, 2))
    out = ops.dequant_fp8_block128(q.cuda().view(torch.float8_e4m3fn), s.cuda()).float().cpu().numpy()[0]
    tab = O.fp8_table()
    ok = ~np.isnan(tab)
    assert np.array_equal(out[ok], tab[ok]) and np.isnan(out[~ok]).all()


def test_dequant_golden_fixture():
    import os
    from moe_gen_amd import ops
    z = np.load(os.path.join(os.path.dirname(__file__), "golden", "fp8_dequant.npz"))
    out = ops.dequant_fp8_block128(torch.from_numpy(z["q"]).cuda().view(torch.float8_e4m3fn), torch.from_numpy(z["scale"]).cuda())
    assert np.array_equal(bits(out), z["out"])


@pytest.mark.parametrize("fp8", [False, True])
def test_swiglu_epilogue_alone(fp8):
    """The SiLU*mul epilogue pinned on its own: one-hot token rows make every gate and up output a
    single exact product, g[r,c] = Wg[c, r], u[r,c] = Wu[c, r], so `act` (the gate/up launch's
    output) must be bf16(bf16(silu(g)) * u) -- torch's own bf16 silu and bf16 mul on the CPU are the
    witness.  The kernel evaluates silu with the hardware exp and reciprocal (about 1e-6 relative),
    so bf16(silu(g)) may land on the other side of a rounding boundary on a few elements: one bf16
    step there, which the product with u turns into at most two steps of the result (a factor at the
    bottom of its binade, a product at the top of one).  A swapped gate/up role, a missing rounding
    point or a wrong sign fails everywhere."""
    from moe_gen_amd import ops
    from moe_gen_amd.synthetic import quantize_fp8_block128
    h = I = 128
    n = 3 * h                                            # every one-hot row three times, with different scales
    g = torch.Generator().manual_seed(17)
    if fp8:                                              # exactly representable after block quantisation: powers of two times small integers
        wg = (torch.randint(-12, 13, (I, h), generator=g).float() * 0.25)
        wu = (torch.randint(-8, 9, (I, h), generator=g).float() * 0.5)
        wg[0, 0], wu[0, 0] = 28.0, 14.0                 # fixes each block's scale: amax = 28 -> 28/448 = 2^-4, 14/448 = 2^-5
        qg, qu = quantize_fp8_block128(wg), quantize_fp8_block128(wu)
        wg_f = torch.from_numpy(O.bf16_to_f32(O.dequant_block(bits(qg[0]), qg[1].numpy())))
        wu_f = torch.from_numpy(O.bf16_to_f32(O.dequant_block(bits(qu[0]), qu[1].numpy())))
        assert torch.equal(wg_f, wg) and torch.equal(wu_f, wu)
        qd = quantize_fp8_block128(torch.zeros(h, I))
        ptrs = ops.expert_pointers([qg[0].cuda()], [qu[0].cuda()], [qd[0].cuda()], [qg[1].cuda()], [qu[1].cuda()], [qd[1].cuda()])
    else:
        wg = (torch.randn(I, h, generator=g) * 4).to(torch.bfloat16)
        wu = (torch.randn(I, h, generator=g) * 2).to(torch.bfloat16)
        wg_f, wu_f = wg.float(), wu.float()
        ptrs = ops.expert_pointers([wg.cuda()], [wu.cuda()], [torch.zeros(h, I, dtype=torch.bfloat16).cuda()])
    scales = torch.tensor([1.0, 0.5, 4.0])
    x = torch.zeros(n, h, dtype=torch.bfloat16)
    for r in range(n):
        x[r, r % h] = scales[r // h]
    act = torch.empty(n, I, dtype=torch.bfloat16, device="cuda")
    y = torch.empty(n, h, dtype=torch.bfloat16, device="cuda")
    off = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    ops.grouped_swiglu(x.cuda(), None, ptrs, off, n, act, y, ops.PHASE_GATE_UP)
    torch.cuda.synchronize()
    gate = torch.stack([wg_f[:, r % h] * scales[r // h] for r in range(n)]).to(torch.bfloat16)   # exact: one product
    up = torch.stack([wu_f[:, r % h] * scales[r // h] for r in range(n)]).to(torch.bfloat16)
    want = torch.nn.functional.silu(gate) * up                                                    # bf16 modules, as the reference
    got_bits, want_bits = bits(act).astype(np.int32), bits(want).astype(np.int32)
    diff = np.abs(got_bits - want_bits)
    assert diff.max() <= 2, f"epilogue off by {diff.max()} bf16 steps"
    assert (diff > 0).mean() < 0.01, f"{(diff > 0).mean():.2%} of the elements differ"
    assert (diff > 1).mean() < 0.001, f"{(diff > 1).mean():.3%} of the elements differ by two steps"


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("h,I", [(128, 128), (640, 384), (1024, 896), (256, 8320)])    # 1 ... 130 stages; more than 64 fp8 scales per row
def test_thin_kernel_matches_larger_calls(fp8, h, I):
    """Calls whose experts have at most 16 rows run on one wave per 32 weight rows.  Experts of 0 ... 16 rows, empty ones
    in front, between and behind, more experts than a wave scans at once; rows gathered through a row map with an entry
    outside x (zeros).  Against the oracle, and bit for bit against the same rows in a call with an expert of 40 rows
    (the tile kernel: fp8 in its form for up to 64 rows)."""
    from moe_gen_amd import ops
    E = 263
    counts = [0] * E
    for e, c in ((1, 1), (2, 16), (4, 15), (63, 2), (64, 7), (255, 3), (256, 16), (261, 1)):
        counts[e] = c
    print(f"thin fp8={fp8} h={h} I={I}", flush=True)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = int(offsets[-1])
    g = torch.Generator().manual_seed(401)
    x = torch.randn(n + 40, h, generator=g).to(torch.bfloat16)
    mats = make_experts(2, h, I, fp8, 402)                       # experts alternate between two sets of weights
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    dm = [[dev(m) for m in one] for one in mats]
    pick = lambda i, j: [dm[e % 2][i][j] if fp8 else dm[e % 2][i] for e in range(E)]
    ptrs = ops.expert_pointers(*(pick(i, 0) for i in range(3)), *((pick(i, 1) for i in range(3)) if fp8 else ()))
    rm = torch.randperm(n, generator=g).to(torch.int32)
    xd = x.cuda()
    m, _, y = ops.mlp_group(xd, rm.cuda(), ptrs, torch.from_numpy(offsets).cuda(), n, 16)
    ops.grouped_swiglu_joint(m, None, h, fp8)
    bad = rm.clone()
    bad[[0, 20]] = torch.tensor([n + 40, -3], dtype=torch.int32)
    mb, _, yb = ops.mlp_group(xd, bad.cuda(), ptrs, torch.from_numpy(offsets).cuda(), n, 16)
    ops.grouped_swiglu_joint(mb, None, h, fp8)
    big = list(counts)
    big[262] = 40                                                # behind all others: their rows keep their places
    off_big = np.concatenate([[0], np.cumsum(big)]).astype(np.int32)
    rm_big = torch.cat([rm, torch.arange(n, n + 40, dtype=torch.int32)])
    y_big = ops.grouped_swiglu(xd, rm_big.cuda(), ptrs, torch.from_numpy(off_big).cuda(), n + 40)
    torch.cuda.synchronize()
    assert torch.equal(y, y_big[:n])
    keep = torch.ones(n, dtype=torch.bool)
    keep[[0, 20]] = False
    assert torch.equal(yb.cpu()[keep], y.cpu()[keep]) and (yb.cpu()[~keep].float() == 0).all()
    xf = O.bf16_to_f32(bits(x[rm.long()]))
    ref = np.zeros((n, h), np.float32)
    for e in range(E):
        a, b = offsets[e], offsets[e + 1]
        if b > a:
            ref[a:b] = O.mlp_f32(xf[a:b], *(f32_of(w) for w in mats[e % 2]))
    assert rel_max(O.bf16_to_f32(bits(y)), ref) <= TOL


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n,shared_inter", [(1, 256), (16, 768), (17, 256), (100, 768), (192, 256), (193, 512), (300, 256)])
def test_shared_expert_in_the_routed_launches(fp8, n, shared_inter):
    """A shared expert of another intermediate size next to the routed experts: few rows (thin kernel), one tile, two
    halves of 257 ... 384 rows and 128-row slices (tile kernel).  Bit for bit what the two calls give apart; with fp8
    weights too as long as both calls are ones that the tile kernel serves alone (mean rows per expert below 128)."""
    from moe_gen_amd import ops
    E, k, h, I = 12, 2, 384, 256
    print(f"joint fp8={fp8} n={n} shared_inter={shared_inter}", flush=True)
    g = torch.Generator().manual_seed(n)
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    tables = []
    for count, inter, seed in ((E, I, 11), (1, shared_inter, 12)):
        dm = [[dev(m) for m in one] for one in make_experts(count, h, inter, fp8, seed)]
        col = lambda i, j: [o[i][j] if fp8 else o[i] for o in dm]
        tables.append(ops.expert_pointers(*(col(i, 0) for i in range(3)), *((col(i, 1) for i in range(3)) if fp8 else ())))
    idx = torch.rand((n, E), generator=g).topk(k, dim=1).indices.to(torch.int32)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16).cuda()
    d = ops.dispatch(idx.cuda(), E, None, want_row_map=True)
    so = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    r1, _, y1 = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
    s1, _, sh1 = ops.mlp_group(x, None, tables[1], so, n)
    assert ops.shared_joins(r1, s1, h)
    ops.grouped_swiglu_joint(r1, s1, h, fp8)
    r2, _, y2 = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
    s2, _, sh2 = ops.mlp_group(x, None, tables[1], so, n)
    ops.grouped_swiglu_joint(r2, None, h, fp8)
    ops.grouped_swiglu_joint(s2, None, h, fp8)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2)
    if not fp8 or n < 128:
        assert torch.equal(sh1, sh2)
    else:
        a, b = sh1.float(), sh2.float()
        assert (a - b).abs().max().item() <= TOL * b.abs().max().item()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n,E,I,shared_inter", [
    (700, 4, 256, 128),       # the shared expert's k is shorter than the routed experts', every tile of it a half tile
    (1500, 4, 128, 640),      # longer; all of the persistent kernel's tiles are half tiles, the shared expert's among them
    (3000, 8, 1280, 2560),    # rounds of tiles of both
    (2900, 3, 256, 2048),     # mostly the shared expert's
    (200, 2, 256, 384),       # 200 rows each, one 256-row tile
    (150, 2, 256, 384),       # 150 rows each, one tile of up to 192 rows: nothing for the persistent kernel
    (300, 3, 256, 640)])      # bf16: two tiles of up to 192 rows next to a 256-row tile; fp8: 44 rows over a full tile
def test_shared_expert_in_the_launches_of_both_kernels(fp8, n, E, I, shared_inter):
    """From a mean of 128 rows per expert on the shared expert's tiles come first in the launches of the persistent kernel and of
    the other one.  Bit for bit what the calls give apart, with fp8 weights too (both start every tile at k 0 there)."""
    from moe_gen_amd import ops
    k, h = 2, 384
    print(f"joint, both kinds of tiles fp8={fp8} n={n} E={E} I={I} shared_inter={shared_inter}", flush=True)
    g = torch.Generator().manual_seed(n)
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    tables = []
    for count, inter, seed in ((E, I, 11), (1, shared_inter, 12)):
        dm = [[dev(m) for m in one] for one in make_experts(count, h, inter, fp8, seed)]
        col = lambda i, j: [o[i][j] if fp8 else o[i] for o in dm]
        tables.append(ops.expert_pointers(*(col(i, 0) for i in range(3)), *((col(i, 1) for i in range(3)) if fp8 else ())))
    idx = (torch.rand((n, E), generator=g) + 0.2 * torch.arange(E)).topk(k, dim=1).indices.to(torch.int32)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16).cuda()
    d = ops.dispatch(idx.cuda(), E, None, want_row_map=True)
    so = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    r1, _, y1 = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
    s1, _, sh1 = ops.mlp_group(x, None, tables[1], so, n)
    y1.fill_(7.0); sh1.fill_(7.0)
    assert ops.shared_joins(r1, s1, h)
    ops.grouped_swiglu_joint(r1, s1, h, fp8)
    r2, _, y2 = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
    s2, _, sh2 = ops.mlp_group(x, None, tables[1], so, n)
    ops.grouped_swiglu_joint(r2, None, h, fp8)
    ops.grouped_swiglu_joint(s2, None, h, fp8)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2) and torch.equal(sh1, sh2)


@pytest.mark.parametrize("n,E,k,h,I,shared_inter", [
    (1100, 130, 4, 2624, 4096, 384), (1100, 130, 4, 2560, 4160, 384), (1100, 130, 4, 2560, 4096, 448),     # one size an odd multiple of 64
    (1000, 64, 6, 2112, 1408, 384),
    (120, 130, 36, 2560, 4096, 384)])                                                                      # fewer rows than 128
def test_bf16_shared_expert_stays_in_the_launches_where_persistent_tiles_cannot_have_it(n, E, k, h, I, shared_inter):
    """Means of 33 and 93 rows, at which the routed experts' own call has both kinds of tiles where the persistent body can address it:
    a joint call that it cannot serve has one kind.  Bit for bit two calls apart."""
    from moe_gen_amd import ops
    print(f"joint, one kind n={n} E={E} h={h} I={I} shared_inter={shared_inter}", flush=True)
    g = torch.Generator().manual_seed(n)
    tables = []
    for count, inter, seed in ((E, I, 61), (1, shared_inter, 62)):
        one = [m.cuda() for m in make_experts(1, h, inter, False, seed)[0]]
        tables.append(ops.expert_pointers(*([m] * count for m in one)))
    idx = (torch.rand((n, E), generator=g) + 0.004 * torch.arange(E)).topk(k, dim=1).indices.to(torch.int32)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16).cuda()
    d = ops.dispatch(idx.cuda(), E, None, want_row_map=True)
    so = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    r1, _, y1 = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
    s1, _, sh1 = ops.mlp_group(x, None, tables[1], so, n)
    y1.fill_(7.0); sh1.fill_(7.0)
    assert ops.shared_joins(r1, s1, h)
    ops.grouped_swiglu_joint(r1, s1, h, False)
    r2, _, y2 = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
    s2, _, sh2 = ops.mlp_group(x, None, tables[1], so, n)
    ops.grouped_swiglu_joint(r2, None, h, False)
    ops.grouped_swiglu_joint(s2, None, h, False)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2) and torch.equal(sh1, sh2) and torch.isfinite(y1).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("E", [2, 16])          # routed experts of 256 rows (both kinds of tiles) and of 32 (one kind)
@pytest.mark.parametrize("n_rows,rows", [
    (192, 150), (300, 150), (300, 200), (384, 200), (384, 260), (600, 0), (600, 150), (600, 200), (600, 300), (600, 384), (600, 500),
    (1100, 513)])
def test_joint_call_with_fewer_shared_rows_than_its_bound(fp8, E, n_rows, rows):
    """n_rows bounds the shared expert's rows, offsets[] has them: its tiles follow the rows, on both sides of 192, 256 and 384, and
    rows past them are neither read (NaN) nor written.  Bit for bit a call of its own with the same arguments (one kernel, fp8
    weights: the joint call with the exact bound, the call of its own starts its sums elsewhere)."""
    from moe_gen_amd import ops
    n, k, h, I = 256, 2, 256, 384
    print(f"joint, rows below the bound fp8={fp8} E={E} n_rows={n_rows} rows={rows}", flush=True)
    g = torch.Generator().manual_seed(n_rows + rows)
    dev = lambda m: tuple(t.cuda() for t in m) if isinstance(m, tuple) else m.cuda()
    tables = []
    for count, seed in ((E, 21), (1, 22)):
        dm = [[dev(m) for m in one] for one in make_experts(count, h, I, fp8, seed)]
        col = lambda i, j: [o[i][j] if fp8 else o[i] for o in dm]
        tables.append(ops.expert_pointers(*(col(i, 0) for i in range(3)), *((col(i, 1) for i in range(3)) if fp8 else ())))
    idx = torch.rand((n, E), generator=g).topk(k, dim=1).indices.to(torch.int32)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16).cuda()
    xs = torch.randn(n_rows, h, generator=g).to(torch.bfloat16)
    xs[rows:] = float("nan")
    xs = xs.cuda()
    d = ops.dispatch(idx.cuda(), E, None, want_row_map=True)
    so = torch.tensor([0, rows], dtype=torch.int32, device="cuda")
    def call(bound, joint):
        r, _, y = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
        s, _, sh = ops.mlp_group(xs, None, tables[1], so, bound)
        y.fill_(7.0); sh.fill_(7.0)
        if joint:
            assert ops.shared_joins(r, s, h)
            ops.grouped_swiglu_joint(r, s, h, fp8)
        else:
            ops.grouped_swiglu_joint(r, None, h, fp8)
            ops.grouped_swiglu_joint(s, None, h, fp8)
        torch.cuda.synchronize()
        return y, sh
    y1, sh1 = call(n_rows, True)
    y2, sh2 = call(n_rows, False) if E == 2 or not fp8 or rows == 0 else call(rows, True)
    assert torch.equal(y1, y2)
    assert torch.equal(sh1[:rows], sh2[:rows]) and torch.isfinite(sh1[:rows].float()).all()
    assert (sh1[rows:] == 7.0).all()


@pytest.mark.parametrize("n,shared_inter", [(280, 6144), (500, 6144), (700, 4096)])     # the least sizes of the rule
def test_large_fp8_shared_expert_in_a_one_kernel_call_has_the_bits_of_its_own_call(n, shared_inter):
    """Below a mean of 128 rows per routed expert a shared expert of 3/8 of the CUs' worth of 256-row tiles or more is summed as in a
    call of its own, which has both kinds of tiles.  Last tiles of 24, 116 and 60 rows."""
    from moe_gen_amd import ops
    E, k, h, I = 12, 2, 256, 128
    print(f"large shared expert n={n} shared_inter={shared_inter}", flush=True)
    g = torch.Generator().manual_seed(n)
    tables = []
    for count, inter, seed in ((E, I, 41), (1, shared_inter, 42)):
        dm = [[tuple(t.cuda() for t in m) for m in one] for one in make_experts(count, h, inter, True, seed)]
        col = lambda i, j: [o[i][j] for o in dm]
        tables.append(ops.expert_pointers(*(col(i, 0) for i in range(3)), *(col(i, 1) for i in range(3))))
    idx = torch.rand((n, E), generator=g).topk(k, dim=1).indices.to(torch.int32)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16).cuda()
    d = ops.dispatch(idx.cuda(), E, None, want_row_map=True)
    so = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    r1, _, y1 = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
    s1, _, sh1 = ops.mlp_group(x, None, tables[1], so, n)
    assert ops.shared_joins(r1, s1, h)
    ops.grouped_swiglu_joint(r1, s1, h, True)
    r2, _, y2 = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
    s2, _, sh2 = ops.mlp_group(x, None, tables[1], so, n)
    ops.grouped_swiglu_joint(r2, None, h, True)
    ops.grouped_swiglu_joint(s2, None, h, True)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2) and torch.equal(sh1, sh2)


@pytest.mark.parametrize("E,rows,shared_inter,scratch", [
    (12, 17, 12288, True),     # one kernel for the routed experts, slices of k for the shared one
    (2, 300, 4096, True),      # both kinds of tiles
    (2, 100, 640, False)])     # both kinds of tiles, and one that would start its sums elsewhere
def test_joint_call_leaves_apart_what_its_own_call_sums_in_another_way(E, rows, shared_inter, scratch):
    """fp8.  Bit for bit two separate calls on the same groups, scratch included."""
    from moe_gen_amd import _native as N
    from moe_gen_amd import ops
    import ctypes
    n, k, h, I = 256, 2, 512, 128
    print(f"apart E={E} rows={rows} shared_inter={shared_inter} scratch={scratch}", flush=True)
    g = torch.Generator().manual_seed(rows)
    tables = []
    for count, inter, seed in ((E, I, 51), (1, shared_inter, 52)):
        dm = [[tuple(t.cuda() for t in m) for m in one] for one in make_experts(count, h, inter, True, seed)]
        col = lambda i, j: [o[i][j] for o in dm]
        tables.append(ops.expert_pointers(*(col(i, 0) for i in range(3)), *(col(i, 1) for i in range(3))))
    idx = torch.rand((n, E), generator=g).topk(k, dim=1).indices.to(torch.int32)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16).cuda()
    xs = torch.randn(rows, h, generator=g).to(torch.bfloat16).cuda()
    d = ops.dispatch(idx.cuda(), E, None, want_row_map=True)
    so = torch.tensor([0, rows], dtype=torch.int32, device="cuda")
    out = []
    for joint in (True, False):
        r, _, y = ops.mlp_group(x, d.row_map, tables[0], d.offsets, n * k, n)
        s, _, sh = ops.mlp_group(xs, None, tables[1], so, rows)
        if scratch:
            need = N.lib().moe_mlp_workspace_bytes(ctypes.byref(s), h)
            ws = torch.empty(need, dtype=torch.uint8, device="cuda")
            assert need > 0
            s.workspace, s.workspace_bytes = ws.data_ptr(), need
        for a, b in ((r, s),) if joint else ((r, None), (s, None)):
            ops.grouped_swiglu_joint(a, b, h, True)
        torch.cuda.synchronize()
        out.append((y, sh))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("left", [1, 72, 192])
@pytest.mark.parametrize("tiles", [13,      # gate and up: 260 tiles and 20 padded ones, of which 24 run in quarters: the rest of the padded ones persistent
                                   11,      # 220 and 20 of one workgroup beside them; down projection: 12 tiles, the padded one among them, in quarters
                                   1])      # 20 and 20 padded ones, all in quarters
def test_dense_fp8_leftover_rows_as_a_padded_tile(tiles, left):
    """One fp8 MLP whose leftover rows are a padded tile of the persistent kernel's space where the last round then runs in quarters.  The
    rows come out bit for bit as in calls of fewer tiles, where the other kernel serves the leftover, and as in one without it."""
    from moe_gen_amd import ops
    h, I, n = 256, 2560, tiles * 256 + left
    print(f"padded leftover {tiles} {left}", flush=True)
    g = torch.Generator().manual_seed(left)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16).cuda()
    mats = [tuple(t.cuda() for t in m) for m in make_experts(1, h, I, True, 31)[0]]
    ptrs = ops.expert_pointers(*([m[0]] for m in mats), *([m[1]] for m in mats))
    def call(rows):
        return ops.grouped_swiglu(rows, None, ptrs, torch.tensor([0, len(rows)], dtype=torch.int32, device="cuda"), len(rows))
    y = call(x)
    assert torch.isfinite(y).all() and y.any()
    for first in (tiles - 1, max(tiles - 11, 0)):
        assert torch.equal(y[first * 256:], call(x[first * 256:].contiguous())), first
    assert torch.equal(y[:tiles * 256], call(x[:tiles * 256].contiguous()))


@pytest.mark.parametrize("I", [4096, 4224, 18432])      # 32 blocks of 128 k (the rule's least), 33 (a short last slice), DeepSeek-V3's
@pytest.mark.parametrize("h", [128, 768])               # half a column tile; three
def test_dense_fp8_down_projection_in_slices_of_k(h, I):
    """The down projection of one fp8 MLP with its scratch, at the edges of its row tiles: against float64 on the dequantised
    weights, nothing written past the scratch, and a row's bits independent of its place."""
    import ctypes
    from moe_gen_amd import _native as N, ops
    from moe_gen_amd.synthetic import quantize_fp8_block128
    g = torch.Generator(device="cuda").manual_seed(h + I)
    q, sc = quantize_fp8_block128(torch.randn(h, I, generator=g, device="cuda") * 0.02)
    qi = torch.zeros(I, h, device="cuda").to(torch.float8_e4m3fn)      # (gate and up are not run)
    si = torch.ones(I // 128, h // 128, device="cuda")
    ptrs = ops.expert_pointers([qi], [qi], [q], [si], [si], [sc])
    wd = q.double() * sc.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    for n in (1, 16, 17, 63, 64, 65, 80, 81, 128, 129, 160, 161, 256, 257, 384, 512, 513):
        print(f"slices of k h={h} I={I} n={n}", flush=True)
        act = torch.randn(n, I, generator=g, device="cuda").to(torch.bfloat16)
        x = torch.zeros(n, h, dtype=torch.bfloat16, device="cuda")
        off = torch.tensor([0, n], dtype=torch.int32, device="cuda")

        def down(a, need):
            m, _, y = ops.mlp_group(x, None, ptrs, off, n, n, act=a)
            ws = torch.full((need // 4 + 64,), 7.0, device="cuda")
            m.workspace, m.workspace_bytes = (ws.data_ptr(), need) if need else (None, 0)
            ops.grouped_swiglu_joint(m, None, h, True, ops.PHASE_DOWN)
            assert torch.equal(ws[need // 4:], torch.full((64,), 7.0, device="cuda"))
            return y
        m, _, _ = ops.mlp_group(x, None, ptrs, off, n, n, act=act)
        need = N.lib().moe_mlp_workspace_bytes(ctypes.byref(m), h)
        assert need > 0 and need % (4 * n * h) == 0
        y = down(act, need)
        ref = act.double() @ wd.t()
        # weights and result are each rounded to bf16: relative 2^-9 at most, independent per element
        for out in (y, down(act, 0)):
            assert (out.double() - ref).norm() <= 2.0 ** -8 * ref.norm()
        perm = torch.randperm(n, generator=torch.Generator().manual_seed(n)).cuda()
        assert torch.equal(down(act[perm].contiguous(), need), y[perm])


@pytest.mark.parametrize("h,I,n,slices", [
    (1024, 4224, 257, 4),       # the split kernel past 256 rows, its last slice 6 of 9 blocks
    (1024, 4096, 2000, 4),      # sixteen row tiles of it
    (2048, 5632, 900, 4), (4096, 14336, 257, 5), (7168, 18432, 257, 2),
    (7168, 5248, 640, 3),       # 256-row tiles, slices of 14, 14 and 13 blocks
    (4096, 14336, 768, 5), (7168, 18432, 400, 4)])
def test_dense_fp8_slices_past_256_rows(h, I, n, slices):
    """Past 256 rows the down projection of an fp8 MLP is cut on the kernel and into the slices that take least (the number of slices
    is what the scratch is asked for): against float64 on the dequantised weights, nothing past the scratch, and a row's bits
    independent of its place."""
    import ctypes
    from moe_gen_amd import _native as N, ops
    from moe_gen_amd.synthetic import quantize_fp8_block128
    print(f"slices past 256 rows h={h} I={I} n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + h)
    q, sc = quantize_fp8_block128(torch.randn(h, I, generator=g, device="cuda") * 0.02)
    qi, si = torch.zeros(I, h, device="cuda").to(torch.float8_e4m3fn), torch.ones(I // 128, h // 128, device="cuda")
    ptrs = ops.expert_pointers([qi], [qi], [q], [si], [si], [sc])
    off = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    act = torch.randn(n, I, generator=g, device="cuda").to(torch.bfloat16)

    def down(a):
        y = torch.full((n, h), 3.0, dtype=torch.bfloat16, device="cuda")
        m, _, _ = ops.mlp_group(torch.zeros(n, h, dtype=torch.bfloat16, device="cuda"), None, ptrs, off, n, n, act=a, y=y)
        need = N.lib().moe_mlp_workspace_bytes(ctypes.byref(m), h)
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert need == 4 * slices * n * h
        ws = torch.full((need // 4 + 64,), 7.0, device="cuda")
        m.workspace, m.workspace_bytes = ws.data_ptr(), need
        ops.grouped_swiglu_joint(m, None, h, True, ops.PHASE_DOWN)
        assert (ws[need // 4:] == 7.0).all()
        return y
    y = down(act)
    wd = q.double() * sc.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    ref = act.double() @ wd.t()
    # weights and result are each rounded to bf16: relative 2^-9 at most, independent per element
    assert (y.double() - ref).norm() <= 2.0 ** -8 * ref.norm()
    perm = torch.randperm(n, generator=torch.Generator().manual_seed(n)).cuda()
    assert torch.equal(down(act[perm].contiguous()), y[perm])


@pytest.mark.parametrize("n,first,rows", [
    (1300, 0, 1300),        # slices of more than a round of tiles
    (1000, 40, 700),        # fewer rows than the host allows for, behind other rows: fewer row tiles, the last one ragged
    (600, 0, 0)])
def test_dense_fp8_slices_of_k_on_whole_tiles(n, first, rows):
    """The down projection of DeepSeek-V3's dense MLP, 256-row tiles of the persistent kernel once per slice of k: against float64 on the
    dequantised weights, no other row written, nothing past the scratch, and a row's bits independent of its place."""
    import ctypes
    from moe_gen_amd import _native as N, ops
    from moe_gen_amd.synthetic import quantize_fp8_block128
    h, I = 7168, 18432
    print(f"slices on whole tiles n={n} first={first} rows={rows}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    q, sc = quantize_fp8_block128(torch.randn(h, I, generator=g, device="cuda") * 0.02)
    qi, si = torch.zeros(I, h, device="cuda").to(torch.float8_e4m3fn), torch.ones(I // 128, h // 128, device="cuda")
    ptrs = ops.expert_pointers([qi], [qi], [q], [si], [si], [sc])
    off = torch.tensor([first, first + rows], dtype=torch.int32, device="cuda")
    act = torch.randn(n, I, generator=g, device="cuda").to(torch.bfloat16)

    def down(a):
        y = torch.full((n, h), 3.0, dtype=torch.bfloat16, device="cuda")
        m, _, _ = ops.mlp_group(torch.zeros(n, h, dtype=torch.bfloat16, device="cuda"), None, ptrs, off, n, n, act=a, y=y)
        need = N.lib().moe_mlp_workspace_bytes(ctypes.byref(m), h)
        assert need > 4 * n * h and need % (4 * n * h) == 0
        ws = torch.full((need // 4 + 64,), 7.0, device="cuda")
        m.workspace, m.workspace_bytes = ws.data_ptr(), need
        ops.grouped_swiglu_joint(m, None, h, True, ops.PHASE_DOWN)
        assert (ws[need // 4:] == 7.0).all() and (y[:first] == 3.0).all() and (y[first + rows:] == 3.0).all()
        return y[first:first + rows]
    y = down(act)
    if rows == 0:
        return
    wd = q.double() * sc.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    ref = act[first:first + rows].double() @ wd.t()
    # weights and result are each rounded to bf16: relative 2^-9 at most, independent per element
    assert (y.double() - ref).norm() <= 2.0 ** -8 * ref.norm()
    perm = torch.randperm(rows, generator=torch.Generator().manual_seed(n)).cuda()
    moved = act.clone()
    moved[first:first + rows] = act[first:first + rows][perm]
    assert torch.equal(down(moved), y[perm])


@pytest.mark.parametrize("n,inter", [(1, 256), (16, 256), (17, 256), (64, 256), (65, 256), (128, 256), (192, 256), (193, 256), (256, 256),
                                     (1, 4096), (16, 4096), (64, 4096), (65, 4096), (128, 4096)])
def test_fp8_weights_are_dequantised_to_bf16_at_every_row_count(n, inter):
    """A weight is bf16(f32(q) * s) in every kernel (one wave per 32 weight rows, the streamers, the persistent kernel, slices
    of k with scratch from 4096 on), over all finite byte values.  A token row takes the difference of two neighbouring
    codes: both products and their sum are exact in fp32, so the down projection's result is pinned to the bit, and the
    rounding of the two weights is 3 % of it and more.  The up projection is read through a gate of exactly 1: one bf16
    step for silu by the hardware exponential."""
    import ctypes
    from moe_gen_amd import _native as N, ops
    print(f"fp8 rounding n={n} inter={inter}", flush=True)
    h = 384
    codes = torch.tensor([c for c in range(256) if c & 0x7f != 0x7f], dtype=torch.uint8)
    g = torch.Generator().manual_seed(n + inter)

    def weight(rows, cols):
        i = torch.arange(cols).unsqueeze(0) + 37 * torch.arange(rows).unsqueeze(1)
        q = codes[i % len(codes)].view(torch.float8_e4m3fn)
        s = 0.01 + 0.01 * torch.rand(-(-rows // 128), -(-cols // 128), generator=g)
        w = (q.float() * s.repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)[:, :cols]).to(torch.bfloat16).float()
        return q.cuda(), s.cuda(), w

    def rows_of(width):                                  # (+1 at an even k, -1 behind it)
        k = torch.randint(0, width // 2, (n,), generator=g) * 2
        a = torch.zeros(n, width)
        a[torch.arange(n), k], a[torch.arange(n), k + 1] = 1.0, -1.0
        return k, a.to(torch.bfloat16).cuda()

    up, down = weight(inter, h), weight(h, inter)
    one = torch.zeros(inter, h)
    one[:, ::2] = 1.0
    ptrs = ops.expert_pointers([one.to(torch.float8_e4m3fn).cuda()], [up[0]], [down[0]],
                               [torch.ones(inter // 128, h // 128).cuda()], [up[1]], [down[1]])
    off = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    kx, x = rows_of(h)
    m, act, _ = ops.mlp_group(x, None, ptrs, off, n, n)
    ops.grouped_swiglu_joint(m, None, h, True, ops.PHASE_GATE_UP)
    u = (up[2][:, kx] - up[2][:, kx + 1]).t().to(torch.bfloat16)
    want = torch.nn.functional.silu(torch.ones((), dtype=torch.bfloat16)) * u
    assert ((act.cpu().float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs()).all()

    ka, a = rows_of(inter)
    m, _, y = ops.mlp_group(x, None, ptrs, off, n, n, act=a)
    need = N.lib().moe_mlp_workspace_bytes(ctypes.byref(m), h)
    assert (need > 0) == (inter >= 4096)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    m.workspace, m.workspace_bytes = (ws.data_ptr(), need) if need else (None, 0)
    ops.grouped_swiglu_joint(m, None, h, True, ops.PHASE_DOWN)
    assert torch.equal(y.cpu().float(), (down[2][:, ka] - down[2][:, ka + 1]).t().to(torch.bfloat16).float())


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("E,h,I", [(8, 4608, 8192), (40, 512, 384)])     # long k and 144 tiles; short k, whole and part-filled rounds
def test_kernel_choice_for_few_rows_leaves_the_bits(fp8, E, h, I):
    """Calls of at most 16 rows per expert on both sides of three rows per expert, where the rounds of the thin and the tile
    kernel begin to be compared: a row's bits are those of a call that names no bound (the tile kernel) and do not
    depend on how many rows the others have.  All experts share one set of weights."""
    from moe_gen_amd import ops
    print(f"few rows fp8={fp8} E={E} h={h} I={I}", flush=True)
    m = [t if isinstance(t, tuple) else (t,) for t in make_experts(1, h, I, fp8, 21)[0]]
    m = [[t.cuda() for t in one] for one in m]
    ptrs = ops.expert_pointers(*([one[0]] * E for one in m), *(([one[1]] * E for one in m) if fp8 else ()))
    x = torch.randn(E, 16, h, generator=torch.Generator().manual_seed(22)).to(torch.bfloat16).cuda()

    def call(rows, bound):
        xs = x[:, :rows].reshape(-1, h).contiguous()
        off = torch.arange(0, E * rows + 1, rows, dtype=torch.int32, device="cuda")
        g, _, y = ops.mlp_group(xs, None, ptrs, off, E * rows, bound)
        ops.grouped_swiglu_joint(g, None, h, fp8)
        return y.view(E, rows, h)

    want = call(16, 0)
    assert want.float().abs().max() > 0
    for rows in (1, 2, 3, 4, 16):
        assert torch.equal(call(rows, 16), want[:, :rows]), rows


@pytest.mark.parametrize("E,mean,h,I", [        # both sides of the lines of both_kinds
    (8, 127, 384, 320), (8, 128, 384, 320),
    (64, 89, 2048, 1280), (64, 90, 2048, 1280), (63, 90, 2048, 1280),      # mean * mean * weights; experts
    (64, 120, 2048, 1152), (64, 120, 2048, 1280),                          # weights
    (130, 31, 2560, 4096), (130, 32, 2560, 4096)])                         # mean
def test_bf16_skewed_experts_around_the_line_between_one_and_both_kinds(E, mean, h, I):
    """A few experts hold most of the rows: 256-row tiles, pairs and slices next to small ones.  Every expert's rows equal, bit
    for bit, those of a call with that expert alone."""
    from moe_gen_amd import ops
    rows = E * mean
    counts = np.full(E, 3, np.int64)
    counts[[1, 3, 4]] = rows // 4, 300, 190
    counts[6] += rows - counts.sum()
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    print(f"skewed experts E={E} mean={mean} h={h} I={I}", flush=True)
    assert counts.min() > 0 and offsets[-1] == rows
    g = torch.Generator().manual_seed(E + mean)
    x = torch.randn(rows, h, generator=g).to(torch.bfloat16).cuda()
    few = [[m.cuda() for m in one] for one in make_experts(3, h, I, False, E)]
    mats = [few[e % 3] for e in range(E)]
    call = lambda xs, ms, off: ops.grouped_swiglu(xs, None, ops.expert_pointers(*([m[j] for m in ms] for j in range(3))),
                                                  torch.tensor(off, dtype=torch.int32, device="cuda"), xs.shape[0])
    y = call(x, mats, offsets.tolist())
    for e in (0, 1, 3, 4, 5, 6, E - 1):
        a, b = int(offsets[e]), int(offsets[e + 1])
        assert torch.equal(y[a:b], call(x[a:b].contiguous(), [mats[e]], [0, b - a])), f"expert {e} ({b - a} rows)"


@pytest.mark.parametrize("h,E,counts", [(2048, 6, [192, 97, 96, 1, 200, 130]),      # 8 column tiles an expert, 88 tiles of up to 96 rows
                                        (4096, 8, [97, 97, 97, 97, 97, 97, 97, 97]),   # 16: as many tiles as CUs
                                        (4096, 16, [300, 20, 700, 60, 257]),        # 16: too many of 96 rows for 256 CUs, 14 of 128
                                        (4096, 16, [900, 3, 1, 385, 384]),          # 16: too many of 128 as well
                                        (256, 24, [1000, 161, 64, 17])])            # one column tile, rows in up to 11 tiles
def test_bf16_down_projection_of_few_tiles_is_cut_in_rows(h, E, counts):
    """Heights that the call's own counts choose: rows equal, bit for bit, those of calls with 64 rows of their expert alone."""
    from moe_gen_amd import ops
    I = 320
    counts = counts + [0] * (E - len(counts))
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    print(f"few tiles h={h} {counts}", flush=True)
    g = torch.Generator().manual_seed(h + E)
    act = torch.randn(int(offsets[-1]), I, generator=g).to(torch.bfloat16).cuda()
    downs = [(torch.randn(h, I, generator=g) * 0.05).to(torch.bfloat16).cuda() for _ in counts]
    other = torch.zeros(I, h, dtype=torch.bfloat16, device="cuda")

    def down(rows, mats, off):
        ptrs = ops.expert_pointers([other] * len(mats), [other] * len(mats), mats)
        y = torch.full((rows.shape[0], h), 7.0, dtype=torch.bfloat16, device="cuda")
        x = torch.zeros(rows.shape[0], h, dtype=torch.bfloat16, device="cuda")
        m, _, _ = ops.mlp_group(x, None, ptrs, torch.tensor(off, dtype=torch.int32, device="cuda"), rows.shape[0], rows.shape[0], act=rows, y=y)
        ops.grouped_swiglu_joint(m, None, h, False, ops.PHASE_DOWN)
        return y

    assert offsets[-1] // E < 128                      # (tiles of one workgroup alone)
    y = down(act, downs, offsets.tolist())
    for e in range(E):
        if counts[e] == 0:
            continue
        a, b = int(offsets[e]), int(offsets[e + 1])
        parts = [down(act[i:min(i + 64, b)].contiguous(), [downs[e]], [0, min(i + 64, b) - i]) for i in range(a, b, 64)]
        assert torch.equal(y[a:b], torch.cat(parts)), f"expert {e} ({b - a} rows)"


@pytest.mark.parametrize("n,I", [(1, 18432), (16, 14464), (17, 16384), (33, 16512), (48, 18432), (64, 20480), (65, 18432), (80, 20480), (81, 16384), (96, 16512), (97, 14464),
                                 (113, 20480), (128, 18432)])       # 8, 9 and 10 waves a workgroup on 256 CUs, last tiles whole and ragged; past 96 rows
@pytest.mark.parametrize("h", [128, 640])                           # 1 and 5 blocks of 128 k, for rings of 3 (65 rows and more) to 6 stages (up to 16)
def test_wide_fp8_mlp_of_few_rows(n, I, h):
    """Gate and up projection of one wide fp8 MLP.  A token row that is 1 at one k reads a column of both matrices exactly, so that
    act is pinned to one bf16 step (silu by the hardware exponential); dense rows against the oracle, also gathered in another
    order with an entry outside x, bit for bit the same where the row is."""
    from moe_gen_amd import ops
    print(f"wide mlp n={n} I={I} h={h}", flush=True)
    mats = make_experts(1, h, I, True, 7)[0]
    dm = [tuple(t.cuda() for t in m) for m in mats]
    ptrs = ops.expert_pointers(*([m[0]] for m in dm), *([m[1]] for m in dm))
    off = torch.tensor([0, n], dtype=torch.int32, device="cuda")

    def gate_up(x, row_map=None):
        m, act, _ = ops.mlp_group(x, row_map, ptrs, off, n, n)
        act.fill_(7.0)
        ops.grouped_swiglu_joint(m, None, h, True, ops.PHASE_GATE_UP)
        return act

    g = torch.Generator().manual_seed(n + I)
    k = torch.randint(0, h, (n,), generator=g)
    one = torch.zeros(n, h)
    one[torch.arange(n), k] = 1.0
    gate, up = (torch.from_numpy(f32_of(m)) for m in mats[:2])
    want = torch.nn.functional.silu(gate[:, k].t().to(torch.bfloat16)).float() * up[:, k].t().to(torch.bfloat16).float()
    got = gate_up(one.to(torch.bfloat16).cuda()).cpu().float()
    assert ((got - want).abs() <= 2.0 ** -6 * want.abs()).all()

    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    y = gate_up(x.cuda())
    a = x.float() @ gate.t()
    ref = torch.nn.functional.silu(a) * (x.float() @ up.t())
    assert rel_max(O.bf16_to_f32(bits(y)), ref.numpy()) <= TOL
    rm = torch.randperm(n, generator=g).to(torch.int32)
    bad = rm.clone()
    bad[n // 2] = n + 5
    z = gate_up(x.cuda(), bad.cuda())
    keep = torch.arange(n) != n // 2
    assert torch.equal(z.cpu()[keep], y.cpu()[rm.long()][keep]) and (z.cpu()[n // 2].float() == 0).all()


@pytest.mark.parametrize("n,I,h", [(1, 18432, 2048), (16, 14464, 2048), (17, 16384, 2048), (32, 20480, 2048), (48, 14464, 2048), (96, 18432, 2048),
                                   (1, 14464, 8320), (16, 16512, 8320), (32, 18432, 8320), (64, 14464, 8320), (96, 14464, 8320)])
def test_wide_fp8_mlp_of_few_rows_at_long_k(n, I, h):
    """16 blocks of 128 k: every ring turns several times, whatever its stages; 65: the block scales, 64 of which a wave holds, are
    loaded again.  Rows that are 1 at one k pin a column of both matrices, and so its block's scales; dense rows against float64."""
    from moe_gen_amd import ops
    from moe_gen_amd.synthetic import quantize_fp8_block128
    print(f"wide mlp n={n} I={I} h={h}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + h)
    mats = [quantize_fp8_block128(torch.randn(I, h, generator=g, device="cuda") * (0.02 + 0.02 * torch.rand(1, h, generator=g, device="cuda"))) for _ in range(2)]
    down = (torch.zeros(h, I, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn), torch.ones(h // 128, I // 128, device="cuda"))
    ptrs = ops.expert_pointers(*([m[0]] for m in (*mats, down)), *([m[1]] for m in (*mats, down)))
    off = torch.tensor([0, n], dtype=torch.int32, device="cuda")

    def gate_up(x):
        m, act, _ = ops.mlp_group(x, None, ptrs, off, n, n)
        act.fill_(7.0)
        ops.grouped_swiglu_joint(m, None, h, True, ops.PHASE_GATE_UP)
        return act

    full = [(q.float() * s.repeat_interleave(128, 0).repeat_interleave(128, 1)).to(torch.bfloat16) for q, s in mats]
    k = torch.randint(0, h, (n,), generator=g, device="cuda")
    k[: min(n, 2)] = torch.tensor([h - 1, 64 * 128 if h > 64 * 128 else 0], device="cuda")[: min(n, 2)]
    one = torch.zeros(n, h, device="cuda")
    one[torch.arange(n, device="cuda"), k] = 1.0
    want = torch.nn.functional.silu(full[0][:, k].t()).float() * full[1][:, k].t().float()
    assert ((gate_up(one.to(torch.bfloat16)).float() - want).abs() <= 2.0 ** -6 * want.abs()).all()
    x = torch.randn(n, h, generator=g, device="cuda").to(torch.bfloat16)
    a, b = (x.double() @ w.double().t() for w in full)
    y, ref = gate_up(x).double(), torch.nn.functional.silu(a) * b
    assert ((y - ref).abs().max() / ref.abs().max()).item() <= TOL


@pytest.mark.parametrize("h,I,E,counts", [
    (192, 320, 12, [1, 0, 16, 17, 63, 64, 65, 100, 128, 3, 33, 48]),      # a ragged last half tile, 5 stages of 64 k; up to two slices
    (4096, 64, 8, [48, 47, 1, 129, 90, 0, 60, 9]),                        # 128 whole tiles: half a round; one stage; three slices
    (2048, 704, 40, [5] * 20 + [0] * 10 + [40, 64, 65, 130, 1, 2, 17, 33, 9, 20]),     # 320 whole tiles: a part-filled second round
    (64, 448, 1, [40])])                                                  # half of a half tile
def test_bf16_half_tiles_of_a_down_projection(h, I, E, counts):
    """Tiles of 128 columns and up to 64 rows: rows equal, bit for bit, those of a call with 192-row tiles and persistent ones (an
    expert of many rows behind them)."""
    from moe_gen_amd import ops
    print(f"half tiles h={h} I={I} {counts}", flush=True)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n, more = int(offsets[-1]), 130 * (E + 1)
    g = torch.Generator().manual_seed(h + I)
    act = torch.randn(n + more, I, generator=g).to(torch.bfloat16).cuda()
    downs = [(torch.randn(h, I, generator=g) * 0.05).to(torch.bfloat16).cuda() for _ in range(E + 1)]
    other = torch.zeros(I, h, dtype=torch.bfloat16, device="cuda")

    def down(rows, mats, off):
        ptrs = ops.expert_pointers([other] * len(mats), [other] * len(mats), mats)
        y = torch.full((rows.shape[0], h), 7.0, dtype=torch.bfloat16, device="cuda")
        x = torch.zeros(rows.shape[0], h, dtype=torch.bfloat16, device="cuda")
        m, _, _ = ops.mlp_group(x, None, ptrs, torch.tensor(off, dtype=torch.int32, device="cuda"), rows.shape[0], rows.shape[0], act=rows, y=y)
        ops.grouped_swiglu_joint(m, None, h, False, ops.PHASE_DOWN)
        return y

    y = down(act[:n].contiguous(), downs[:E], offsets.tolist())
    big = down(act, downs, offsets.tolist() + [n + more])
    assert torch.equal(y, big[:n])
    ref = act[:n].float().cpu()
    for e in range(E):
        a, b = int(offsets[e]), int(offsets[e + 1])
        if b > a:
            assert rel_max(O.bf16_to_f32(bits(y[a:b])), (ref[a:b] @ downs[e].float().cpu().t()).numpy()) <= TOL


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("h,I", [(3072, 1536),      # 60 tiles both ways: quarters
                                 (4352, 2176),      # 85: thirds, one workgroup less than CUs
                                 (4608, 2304),      # 90: too many for thirds
                                 (256, 6912)])      # gate/up: a round and 14 tiles in quarters
def test_last_tiles_in_three_and_four_pieces(fp8, h, I):
    """Experts of persistent tiles alone, ragged ones (230 and 193 rows) with pieces of few rows or none.  Rows equal, bit for bit, those of
    a call that ends with an expert of 12 tiles more, where the persistent workgroups hold these."""
    from moe_gen_amd import ops
    counts = [512, 230, 449, 3072]
    n, E = sum(counts[:3]), 3
    print(f"pieces fp8={fp8} h={h} I={I}", flush=True)
    g = torch.Generator().manual_seed(h + I)
    x = torch.randn(sum(counts), h, generator=g).to(torch.bfloat16).cuda()
    mats = [[[t.cuda() for t in (m if fp8 else [m])] for m in one] for one in make_experts(E + 1, h, I, fp8, I)]

    def call(e, rows):
        ptrs = ops.expert_pointers(*([m[j][part] for m in mats[:e]] for part in range(1 + fp8) for j in range(3)))
        off = np.concatenate([[0], np.cumsum(counts[:e])]).astype(np.int32)
        return ops.grouped_swiglu(rows, None, ptrs, torch.from_numpy(off).cuda(), rows.shape[0])

    y = call(E, x[:n].contiguous())
    assert torch.isfinite(y).all() and y.any() and torch.equal(y, call(E + 1, x)[:n])
