"""The batched expert GEMV and the kernel-mode Mixture-of-Experts block on the GPU
(reference tests/test_moe.py:283-399)."""

import numpy as np
import pytest
import torch

import llmq_oracle as oracle
from conftest import rel_l2, to_np
from test_moe_host import expert_block, mixtral_model, routing

from llmquant import QuantConfig, oneshot

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    from llmquant.hip import load_extension

    return load_extension()


def kernel_block(bits="int8", **kw):
    """hidden and intermediate 512: four groups of 128, the smallest rows the matrix-core kernels
    take (shorter ones go to the fallback kernels, whose summation order is another)."""
    from llmquant.quantizers import KernelQuantExperts, RealQuantExperts

    kw.setdefault("hidden", 512)
    kw.setdefault("inter", 512)
    block, cfg = expert_block(**kw)
    block = block.cuda()
    scheme = QuantConfig(mlp_weight=bits).scheme("mlp_weight")
    return block, KernelQuantExperts.from_experts(block, scheme).cuda().eval(), \
        RealQuantExperts.from_experts(block, scheme).cuda().eval(), cfg


@pytest.mark.parametrize("bits", ["int8", "int4"])
@pytest.mark.parametrize("tokens", [1, 4, 8])
def test_the_batched_kernel_is_bit_exact_per_row_against_single_launches(ext, bits, tokens):
    _, quant, _, cfg = kernel_block(bits)
    torch.manual_seed(tokens)
    hidden = torch.randn(tokens, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, _ = routing(tokens, cfg.num_local_experts, cfg.num_experts_per_tok, seed=tokens)
    index = index.cuda()
    with torch.no_grad():
        order, plan = quant._plan(index)
        rows = hidden[order // cfg.num_experts_per_tok]
        batched = quant._batched(rows, quant.gate_up_data, quant.sgate_up, plan, quant.hidden_dim, quant._gate_up_padded)
        flat = index.reshape(-1)
        looped = torch.empty_like(batched)
        for expert in flat.unique().tolist():
            sel = (flat[order] == expert).nonzero().flatten()
            for r in sel.tolist():  # one row per launch: the single-row kernel is the yardstick
                looped[r] = ext.wq_gemv(rows[r:r + 1], quant.gate_up_data[expert], quant.sgate_up[expert], 0)[0]
    assert torch.equal(batched, looped)
    assert all(part.is_cuda for part in plan) and order.is_cuda  # nothing came back to the host


@pytest.mark.parametrize("bits", [8, 4])
def test_runs_of_every_length_and_entries_that_must_be_ignored(ext, bits):
    """The op on a hand-made plan: runs of 1..8 rows, an empty entry, an entry pointing past the
    rows and one naming an expert that does not exist (both ignored, their rows left zero)."""
    gen = torch.Generator().manual_seed(0)
    experts, n, k = 5, 96, 512
    w = (torch.randn(experts, n, k, generator=gen) * 0.02).to(torch.bfloat16)
    stacks = [oracle.canonical_weight(to_np(w[e]), bits, 128) for e in range(experts)]
    codes = np.stack([c for c, _ in stacks])
    q = torch.from_numpy(oracle.pack_int4(codes) if bits == 4 else codes).cuda()
    s = torch.from_numpy(np.stack([sc for _, sc in stacks])).cuda()
    lengths = [1, 2, 3, 4, 5, 6, 7, 8]
    rows = sum(lengths) + 3
    x = torch.randn(rows, k, generator=gen).to(torch.bfloat16).cuda()
    block_expert = [i % experts for i in range(len(lengths))] + [2, 1, 7]
    block_row0 = list(np.cumsum([0] + lengths[:-1])) + [0, rows - 2, 0]
    block_rows = lengths + [0, 5, 2]  # empty; runs past the last row; no such expert
    plan = [torch.tensor(v, dtype=torch.int32, device="cuda") for v in (block_expert, block_row0, block_rows)]
    got = ext.wq_gemv_batched(x, q, s, *plan, 0)
    assert got.shape == (rows, n)
    for e, r0, length in zip(block_expert[:8], block_row0[:8], lengths):
        want = oracle.gemv_float64(to_np(x[r0:r0 + length]), codes[e], stacks[e][1])
        assert rel_l2(to_np(got[r0:r0 + length]), want) <= 1e-2
        for r in range(r0, r0 + length):
            assert torch.equal(got[r], ext.wq_gemv(x[r:r + 1], q[e], s[e], 0)[0])
    assert not got[sum(lengths):].any()
    assert ext.wq_gemv_batched_max_rows() == 8


def test_unusual_group_size_takes_the_fallback_kernel(ext):
    gen = torch.Generator().manual_seed(1)
    experts, n, k, gs = 3, 40, 192, 64
    w = (torch.randn(experts, n, k, generator=gen) * 0.02).to(torch.bfloat16)
    stacks = [oracle.canonical_weight(to_np(w[e]), 8, gs) for e in range(experts)]
    q = torch.from_numpy(np.stack([c for c, _ in stacks])).cuda()
    s = torch.from_numpy(np.stack([sc for _, sc in stacks])).cuda()
    x = torch.randn(5, k, generator=gen).cuda()
    plan = [torch.tensor(v, dtype=torch.int32, device="cuda") for v in ([2, 0], [0, 3], [3, 2])]
    got = ext.wq_gemv_batched(x, q, s, *plan, 0)
    want = np.concatenate([oracle.gemv_float64(to_np(x[:3]), *stacks[2]), oracle.gemv_float64(to_np(x[3:]), *stacks[0])])
    assert rel_l2(to_np(got), want) <= 1e-5


@pytest.mark.parametrize("bits", ["int8", "int4"])
@pytest.mark.parametrize("tokens", [1, 2, 8])
def test_kernel_block_agrees_with_real_mode_and_the_oracle(bits, tokens):
    dense, quant, real, cfg = kernel_block(bits)
    torch.manual_seed(0)
    hidden = torch.randn(tokens, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, weights = routing(tokens, cfg.num_local_experts, cfg.num_experts_per_tok, seed=5)
    index, weights = index.cuda(), weights.cuda()
    with torch.no_grad():
        got, want_real, want_dense = quant(hidden, index, weights), real(hidden, index, weights), dense(hidden, index, weights)
    want = oracle.moe_experts_real(to_np(hidden), to_np(index), to_np(weights), to_np(quant.qgate_up),
                                   to_np(quant.sgate_up), to_np(quant.qdown), to_np(quant.sdown))
    assert rel_l2(to_np(got), want) <= 1e-2            # bf16 outputs, summed in an order atomics choose
    assert rel_l2(to_np(got), to_np(want_real)) <= 1e-2
    assert (got.float() - want_dense.float()).abs().max() < want_dense.float().abs().max() * (0.1 if bits == "int8" else 0.5)


def test_short_rows_fall_back_and_stay_within_tolerance():
    """hidden 256 / intermediate 128 (the reference's test block): two groups and one group per
    row, below what the matrix-core kernel takes."""
    dense, quant, real, cfg = kernel_block(hidden=256, inter=128)
    hidden = torch.randn(3, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, weights = routing(3, cfg.num_local_experts, cfg.num_experts_per_tok, seed=7)
    with torch.no_grad():
        got, want = quant(hidden, index.cuda(), weights.cuda()), real(hidden, index.cuda(), weights.cuda())
    assert rel_l2(to_np(got), to_np(want)) <= 1e-2


def test_wide_batches_take_the_per_expert_path():
    _, quant, real, cfg = kernel_block(experts=2, top_k=2)
    tokens = 64
    assert tokens > quant._batched_max_rows
    hidden = torch.randn(tokens, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, weights = routing(tokens, cfg.num_local_experts, cfg.num_experts_per_tok)
    with torch.no_grad():
        out = quant(hidden, index.cuda(), weights.cuda())
        looped = quant._forward_looped(hidden, index.cuda(), weights.cuda())   # (where the grouped GEMMs do not apply)
        want = real(hidden, index.cuda(), weights.cuda())
    for got in (out, looped):
        assert got.shape == hidden.shape and rel_l2(to_np(got), to_np(want)) <= 2e-2
    quant.act_fn = torch.nn.GELU()
    quant._act_is_silu = quant._probe_silu()
    with torch.no_grad():
        assert not quant._takes_gemm(hidden, index.cuda(), weights.cuda())
        assert torch.isfinite(quant(hidden, index.cuda(), weights.cuda())).all()


def test_the_expert_block_replays_from_a_graph():
    _, quant, _, cfg = kernel_block()
    hidden = torch.randn(1, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, weights = routing(1, cfg.num_local_experts, cfg.num_experts_per_tok)
    index, weights = index.cuda(), weights.cuda()
    with torch.no_grad():
        eager = quant(hidden, index, weights)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(3):
                quant(hidden, index, weights)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = quant(hidden, index, weights)
        for _ in range(3):  # replays, each checked, with other work in between
            captured.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, eager)
            quant(torch.randn_like(hidden), index, weights)
        index.copy_(torch.roll(index, 1, dims=1))  # the plan is rebuilt on the device inside the graph
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, quant(hidden, index, weights))


def test_a_small_mixtral_in_kernel_mode_and_through_a_packed_file(tmp_path):
    from transformers import MixtralForCausalLM

    from llmquant.packing import load_packed_model, save_packed_model
    from llmquant.quantizers import KernelQuantExperts

    recipe = QuantConfig(attn_weight="int8", mlp_weight="int4", head_weight="int8")
    real = oneshot(mixtral_model().cuda(), recipe.to_modifier(mode="real"))
    kernel = oneshot(mixtral_model().cuda(), recipe.to_modifier(mode="kernel"))
    block = kernel.model.layers[0].mlp.experts
    assert isinstance(block, KernelQuantExperts) and block.gate_up_data.dtype == torch.uint8
    ids = torch.randint(0, 1000, (1, 6), generator=torch.Generator().manual_seed(3)).cuda()
    with torch.no_grad():
        want, got = real(ids).logits.float(), kernel(ids).logits.float()
    assert rel_l2(to_np(got), to_np(want)) <= 3e-2
    path = save_packed_model(kernel, tmp_path / "moe.llmq", "local-mixtral")
    loaded = load_packed_model(path, device="cuda", config=kernel.config)
    again = loaded.model.layers[0].mlp.experts
    assert isinstance(again, KernelQuantExperts)
    assert torch.equal(again.gate_up_data, block.gate_up_data) and torch.equal(again.sdown, block.sdown)
    with torch.no_grad():
        assert torch.equal(loaded(ids).logits, kernel(ids).logits)


@pytest.mark.parametrize("tokens,top_k,experts,limit", [(1, 8, 64, 8), (8, 8, 64, 8), (3, 2, 8, 8), (5, 4, 60, 3),
                                                         (64, 8, 64, 8), (1, 1, 1, 8), (700, 8, 128, 8), (9, 2, 1000, 4)])
def test_route_plan_kernel_matches_the_pytorch_form(tokens, top_k, experts, limit):
    """One launch against the argsort / scatter_add / cumsum form (itself pinned to the oracle on the CPU):
    the same order and the same blocks, for one token, many tokens, experts nobody picked, runs longer than
    the limit and a limit that does not divide them."""
    from llmquant.hip import load_extension
    from llmquant.quantizers import route_plan

    ext = load_extension()
    gen = torch.Generator().manual_seed(tokens * 131 + experts)
    index = torch.stack([torch.randperm(experts, generator=gen)[:top_k] for _ in range(tokens)]).cuda()
    assert ext.route_plan_supported(index.numel(), experts)
    for idx in (index, index.to(torch.int32)):
        order, be, r0, rows = ext.route_plan(idx, experts, limit)
        want_order, (want_be, want_r0, want_rows) = route_plan(index, experts, limit)
        assert order.dtype == torch.int64 and be.dtype == torch.int32
        assert torch.equal(order, want_order)
        assert torch.equal(be, want_be) and torch.equal(r0, want_r0) and torch.equal(rows, want_rows)
    # a skewed routing: every token picks the same experts, so their runs exceed the limit
    same = torch.arange(top_k).repeat(tokens, 1).cuda() % experts
    order, be, r0, rows = ext.route_plan(same, experts, limit)
    want_order, want = route_plan(same, experts, limit)
    assert torch.equal(order, want_order)
    assert all(torch.equal(a, b) for a, b in zip((be, r0, rows), want))


def test_route_plan_kernel_limits():
    from llmquant.hip import load_extension

    ext = load_extension()
    assert not ext.route_plan_supported(8193, 64)
    assert not ext.route_plan_supported(8, 1025)
    with pytest.raises(RuntimeError, match="does not take"):
        ext.route_plan(torch.zeros(8193, dtype=torch.int64, device="cuda"), 64, 8)
    with pytest.raises(RuntimeError, match="limit must be positive"):
        ext.route_plan(torch.zeros(8, dtype=torch.int64, device="cuda"), 64, 0)
    order, be, r0, rows = ext.route_plan(torch.zeros(0, dtype=torch.int64, device="cuda"), 4, 8)
    assert order.numel() == 0 and be.tolist() == [0, 1, 2, 3] and rows.tolist() == [0, 0, 0, 0]


@pytest.mark.parametrize("bits", ["int8", "int4"])
@pytest.mark.parametrize("tokens", [1, 3, 8])
def test_fused_forward_pieces_equal_the_operation_by_operation_form(ext, bits, tokens):
    """gate|up with act(gate) * up in its store, the one-token form that skips the row gather, and the
    weighted sum per token, each against the PyTorch steps of KernelQuantExperts.forward."""
    _, quant, _, cfg = kernel_block(bits)
    top_k = cfg.num_experts_per_tok
    torch.manual_seed(10 + tokens)
    hidden = torch.randn(tokens, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, weights = routing(tokens, cfg.num_local_experts, top_k, seed=tokens)
    index, weights = index.cuda(), weights.to(torch.bfloat16).cuda()
    assert quant._fusable(hidden, index, weights)
    with torch.no_grad():
        order, plan = quant._plan(index)
        rows = hidden[order // top_k]
        plain = quant._batched(rows, quant.gate_up_data, quant.sgate_up, plan, quant.hidden_dim, quant._gate_up_padded)
        gate, up = plain.chunk(2, dim=-1)
        want_act = torch.nn.functional.silu(gate) * up
        act = ext.wq_gemv_batched_fused(rows, False, rows.shape[0], quant.gate_up_data, quant.sgate_up, *plan, True)
        assert torch.equal(act, want_act)
        if tokens == 1:
            again = ext.wq_gemv_batched_fused(hidden, True, rows.shape[0], quant.gate_up_data, quant.sgate_up, *plan, True)
            assert torch.equal(again, want_act)
        out = ext.wq_gemv_batched_fused(act, False, rows.shape[0], quant.down_data, quant.sdown, *plan, False)
        assert torch.equal(out, quant._batched(act, quant.down_data, quant.sdown, plan, quant.intermediate_dim,
                                               quant._down_padded))
        # index_add_ on a bf16 tensor rounds after every addition, in no fixed order; the kernel takes the
        # order of the sorted rows
        final = torch.zeros_like(hidden)
        flat_w = weights.reshape(-1)
        for i, src in enumerate(order.tolist()):
            final[src // top_k] = final[src // top_k] + out[i] * flat_w[src]
        got = ext.moe_combine(out, order, weights, tokens)
        assert torch.equal(got, final)
        assert torch.equal(quant._forward_fused(hidden, index, weights), final)
        loose = quant._forward_unfused(hidden, index, weights)
        assert rel_l2(to_np(got), to_np(loose)) <= 1e-2


def test_experts_that_are_not_silu_keep_the_unfused_forward(ext):
    _, quant, _, cfg = kernel_block("int8")
    assert quant._probe_silu()
    quant.act_fn = torch.nn.GELU()
    quant._act_is_silu = quant._probe_silu()
    hidden = torch.randn(2, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, weights = routing(2, cfg.num_local_experts, cfg.num_experts_per_tok, seed=3)
    index, weights = index.cuda(), weights.to(torch.bfloat16).cuda()
    assert not quant._fusable(hidden, index, weights)
    assert torch.isfinite(quant(hidden, index, weights)).all()


@pytest.mark.parametrize("bits,dtype", [("int4", torch.bfloat16), ("int8", torch.bfloat16), ("int4", torch.float16),
                                        ("int8", torch.float32)])
@pytest.mark.parametrize("tokens,hidden,inter,experts,top_k", [
    (1, 512, 512, 4, 1),       # one unit: a workgroup of one wave; sixteen-row tiles that fill half the chip
    (3, 512, 512, 4, 2),
    (1, 2048, 1024, 64, 8),    # a unit a wave, tiles of eight rows
    (8, 2048, 1024, 64, 8),
    (2, 512, 1536, 20, 16),    # 48 units on 16 waves, the largest top_k
    (2, 512, 3072, 8, 6),      # int4: the down launch's LDS passes 64 KB only with the products it holds beside the rows
    (1, 8704, 8192, 3, 2),     # gate|up rows of more chunks than waves, down rows of sixteen chunks
])
def test_direct_launches_equal_the_planned_ones(ext, bits, dtype, tokens, hidden, inter, experts, top_k):
    """Every row's own expert id instead of a plan: the same arithmetic, so the same bits, also for ids that one token
    holds twice and ids outside the layer (counted with the nearest valid one by both)."""
    from llmquant.quantizers import KernelQuantExperts

    gen = torch.Generator(device="cuda").manual_seed(hidden + inter)
    source = torch.nn.Module()
    source.act_fn = torch.nn.SiLU()
    for name, shape in (("gate_up_proj", (experts, 2 * inter, hidden)), ("down_proj", (experts, hidden, inter))):
        weight = torch.randn(shape, device="cuda", generator=gen) * 0.05
        setattr(source, name, torch.nn.Parameter(weight.to(dtype), requires_grad=False))
    quant = KernelQuantExperts.from_experts(source, QuantConfig(mlp_weight=bits).scheme("mlp_weight"))
    x = torch.randn(tokens, hidden, device="cuda", generator=gen).to(dtype)
    weights, index = torch.randn(tokens, experts, device="cuda", generator=gen).softmax(-1).topk(top_k, dim=-1)
    weights = weights.to(dtype)
    odd = index.clone()
    odd[0, 0], odd[-1, -1] = -3, experts + 5
    if top_k > 1:
        odd[0, 1] = odd[-1, 0]
    assert quant._takes_direct(x, index, weights)
    with torch.no_grad():
        for ids in (index, odd, index.int()):
            assert torch.equal(quant(x, ids, weights), quant._forward_fused(x, ids, weights))


def tile_rows(bits, tokens, hidden, inter, experts, top_k):
    from llmquant.hip.build import load_capi

    return load_capi().llmq_wq_experts_tile_rows(tokens, top_k, experts, hidden, inter, 4 if bits == "int4" else 8)


@pytest.mark.parametrize("bits,dtype", [("int4", torch.bfloat16), ("int8", torch.bfloat16), ("int4", torch.float16),
                                        ("int8", torch.float16)])
@pytest.mark.parametrize("tokens,hidden,inter,experts,top_k,skew", [
    (9, 128, 128, 4, 2, False),      # one group a row, one column tile, runs of a few rows
    (33, 384, 256, 3, 1, True),      # a run of 33 rows: one more than a row tile; columns that fill half a tile
    (64, 512, 384, 8, 8, False),     # every expert takes every token: two full tiles each
    (150, 512, 512, 2, 2, True),     # 150 rows an expert: five tiles, the last of 22
    (40, 2048, 1024, 64, 8, False),  # experts that nobody picked among many
])
def test_grouped_gemms_against_real_mode(ext, bits, dtype, tokens, hidden, inter, experts, top_k, skew):
    """A prompt's tokens through the grouped GEMMs, against RealQuantExperts with fp32 throughout: what differs is the
    16-bit rounding of gate, up, silu(gate), their product, each expert's row, its weighted row and the partial sums,
    each within half a unit (2^-9 relative in bf16, 2^-12 in fp16); seven of them in a row stay below 1e-2 / 1.5e-3."""
    from llmquant.quantizers import KernelQuantExperts, RealQuantExperts

    gen = torch.Generator(device="cuda").manual_seed(tokens)
    source = torch.nn.Module()
    source.act_fn = torch.nn.SiLU()
    for name, shape in (("gate_up_proj", (experts, 2 * inter, hidden)), ("down_proj", (experts, hidden, inter))):
        weight = torch.randn(shape, device="cuda", generator=gen) * 0.05
        setattr(source, name, torch.nn.Parameter(weight.to(dtype), requires_grad=False))
    scheme = QuantConfig(mlp_weight=bits).scheme("mlp_weight")
    quant, real = KernelQuantExperts.from_experts(source, scheme), RealQuantExperts.from_experts(source, scheme)
    x = torch.randn(tokens, hidden, device="cuda", generator=gen).to(dtype)
    scores = torch.randn(tokens, experts, device="cuda", generator=gen)
    if skew:
        scores[:, 0] += 10.0
    weights, index = scores.softmax(-1).topk(top_k, dim=-1)
    weights = weights.to(dtype)
    assert quant._takes_gemm(x, index, weights)
    with torch.no_grad():
        got, want = quant(x, index, weights), real(x.float(), index, weights.float())
        assert torch.equal(got, quant(x, index, weights))   # whatever order the rows were placed in
    assert rel_l2(to_np(got), to_np(want)) <= (1e-2 if dtype == torch.bfloat16 else 1.5e-3)


@pytest.mark.parametrize("tokens,hidden,inter,experts,top_k,skew", [
    (641, 128, 128, 16, 8, False),   # 5128 rows: eight more than the plan's threads keep in registers
    (512, 128, 128, 80, 10, True),   # 5120, all kept; two experts a lane of the scan; ten rows a token: eight and two
    (20, 256, 128, 24, 16, False),   # two whole runs of eight rows a token
])
def test_a_prompt_past_what_the_plan_and_the_combination_hold_at_once(ext, tokens, hidden, inter, experts, top_k, skew):
    test_grouped_gemms_against_real_mode(ext, "int4", torch.bfloat16, tokens, hidden, inter, experts, top_k, skew)


@pytest.mark.parametrize("bits,dtype", [("int4", torch.bfloat16), ("int8", torch.bfloat16), ("int4", torch.float16)])
@pytest.mark.parametrize("tokens,hidden,inter,experts,top_k,skew", [
    (20, 640, 768, 4, 2, False),     # five and six groups: the second run of four groups' scales holds one and two
    (90, 896, 1152, 2, 2, False),    # seven and nine
    (90, 1536, 1920, 2, 2, False),   # twelve and fifteen: three and almost four whole runs
])
def test_scales_of_a_last_run_of_groups(ext, bits, dtype, tokens, hidden, inter, experts, top_k, skew):
    assert tile_rows(bits, tokens, hidden, inter, experts, top_k) == 32
    test_grouped_gemms_against_real_mode(ext, bits, dtype, tokens, hidden, inter, experts, top_k, skew)


@pytest.mark.parametrize("bits,dtype", [("int4", torch.bfloat16), ("int8", torch.bfloat16), ("int4", torch.float16),
                                        ("int8", torch.float16)])
@pytest.mark.parametrize("tokens,hidden,inter,experts,top_k,skew,heights", [
    (601, 896, 2176, 2, 2, False, (64, 64)),   # nine 64-row tiles an expert and one of 25; seven and seventeen groups
    (400, 1536, 4736, 2, 2, True, (64, 64)),   # six and one of 16; twelve and thirty-seven
    (333, 640, 4096, 3, 2, True, (32, 64)),    # the first expert takes every token, the others what is left
    (190, 1024, 512, 40, 8, False, (64, 64)),  # 38 rows an expert: one or two tiles each, most of them not full
    (150, 768, 1664, 3, 2, False, (32, 32)),   # about a hundred rows each: four 32-row tiles; six and thirteen groups
])
def test_prompts_by_the_height_of_their_row_tiles(ext, bits, dtype, tokens, hidden, inter, experts, top_k, skew, heights):
    """Shapes on both sides of the line between the heights, ragged in rows and in groups (heights: int4, int8)."""
    assert tile_rows(bits, tokens, hidden, inter, experts, top_k) == heights[bits == "int8"]
    test_grouped_gemms_against_real_mode(ext, bits, dtype, tokens, hidden, inter, experts, top_k, skew)


@pytest.mark.parametrize("tokens", [2, 12])
def test_an_activation_that_starts_inside_a_packet(ext, tokens):
    """A contiguous view at an odd storage offset, through the two-launch form and the grouped GEMMs: the bits of the
    same values in a tensor of their own."""
    from llmquant.quantizers import KernelQuantExperts

    gen = torch.Generator(device="cuda").manual_seed(tokens)
    source = torch.nn.Module()
    source.act_fn = torch.nn.SiLU()
    for name, shape in (("gate_up_proj", (4, 1024, 512)), ("down_proj", (4, 512, 512))):
        weight = torch.randn(shape, device="cuda", generator=gen) * 0.05
        setattr(source, name, torch.nn.Parameter(weight.to(torch.bfloat16), requires_grad=False))
    quant = KernelQuantExperts.from_experts(source, QuantConfig(mlp_weight="int4").scheme("mlp_weight"))
    x = torch.randn(tokens * 512 + 1, device="cuda", generator=gen).to(torch.bfloat16)[1:].view(tokens, 512)
    assert x.data_ptr() % 16 and x.is_contiguous()
    weights, index = torch.randn(tokens, 4, device="cuda", generator=gen).softmax(-1).topk(2, dim=-1)
    weights = weights.to(torch.bfloat16)
    with torch.no_grad():
        assert torch.equal(quant(x, index, weights), quant(x.clone(), index, weights))


def test_a_prompt_carries_the_derivative_of_its_routing_weights(ext):
    """Beyond eight tokens, reverse and forward mode: d out / d weight is the expert's row. In float32 from the real-mode
    block; here its rows are rounded to bfloat16 a few times (each 2^-9), as in the forward pass."""
    from torch.autograd import forward_ad

    _, quant, real, cfg = kernel_block("int8", experts=4, top_k=2)
    gen = torch.Generator(device="cuda").manual_seed(2)
    hidden = torch.randn(20, cfg.hidden_size, device="cuda", generator=gen).to(torch.bfloat16)
    weights, index = torch.randn(20, 4, device="cuda", generator=gen).softmax(-1).topk(2, dim=-1)
    weights = weights.to(torch.bfloat16)
    cotangent = torch.randn(20, cfg.hidden_size, device="cuda", generator=gen)
    with torch.no_grad():
        assert quant._takes_gemm(hidden, index, weights)
    mine, theirs = weights.clone().requires_grad_(), weights.float().requires_grad_()
    out = quant(hidden, index, mine)
    assert out.requires_grad and not quant(hidden, index, weights).requires_grad
    out.backward(cotangent.to(torch.bfloat16))
    real(hidden.float(), index, theirs).backward(cotangent)
    assert rel_l2(to_np(mine.grad), to_np(theirs.grad)) <= 2e-2
    with torch.no_grad(), forward_ad.dual_level():
        tangent = torch.randn(20, 2, device="cuda", generator=gen).to(torch.bfloat16)
        along = forward_ad.unpack_dual(quant(hidden, index, forward_ad.make_dual(weights, tangent))).tangent
        assert rel_l2(to_np(along), to_np(real(hidden.float(), index, tangent.float()))) <= 1e-2


@pytest.mark.parametrize("bits,dtype", [("int4", torch.bfloat16), ("int8", torch.float16)])
def test_a_prompt_with_ids_outside_the_layer(ext, bits, dtype):
    """Beyond eight tokens: tokens that hold such an id get a row of NaN, the others the bits they have without them; ids
    that are not int64 are refused."""
    from llmquant.quantizers import KernelQuantExperts

    gen = torch.Generator(device="cuda").manual_seed(4)
    source = torch.nn.Module()
    source.act_fn = torch.nn.SiLU()
    for name, shape in (("gate_up_proj", (3, 512, 128)), ("down_proj", (3, 128, 256))):
        weight = torch.randn(shape, device="cuda", generator=gen) * 0.05
        setattr(source, name, torch.nn.Parameter(weight.to(dtype), requires_grad=False))
    quant = KernelQuantExperts.from_experts(source, QuantConfig(mlp_weight=bits).scheme("mlp_weight"))
    x = torch.randn(40, 128, device="cuda", generator=gen).to(dtype)
    weights, index = torch.randn(40, 3, device="cuda", generator=gen).softmax(-1).topk(2, dim=-1)
    weights = weights.to(dtype)
    odd, bad = index.clone(), [0, 7, 39]
    odd[0, 0], odd[7, 1], odd[39, 0] = 3, -1, 2 ** 40
    with torch.no_grad():
        assert quant._takes_gemm(x, odd, weights)
        want, got = quant(x, index, weights), quant(x, odd, weights)
        assert got[bad].isnan().all()
        rest = [t for t in range(40) if t not in bad]
        assert torch.equal(got[rest], want[rest]) and want.isfinite().all()
        with pytest.raises(RuntimeError, match="LongTensor"):
            quant(x, index.int(), weights)


def test_a_prompt_too_long_for_the_grouped_gemms_goes_through_the_loop_unless_captured(ext):
    _, quant, _, cfg = kernel_block("int4", experts=4, top_k=2)
    hidden = torch.randn(20, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, weights = routing(20, 4, 2, seed=1)
    index, weights = index.cuda(), weights.cuda()
    with torch.no_grad():
        grouped = quant(hidden, index, weights)
        quant._grouped_pays = lambda rows: False
        assert not quant._takes_gemm(hidden, index, weights)
        assert rel_l2(to_np(quant(hidden, index, weights)), to_np(grouped)) <= 1e-2
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = quant(hidden, index, weights)
        for _ in range(3):
            captured.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, grouped)


def test_a_copied_and_a_pickled_block_give_the_same_rows(ext):
    import copy
    import io

    _, quant, _, cfg = kernel_block("int4")
    hidden = torch.randn(3, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    index, weights = routing(3, cfg.num_local_experts, cfg.num_experts_per_tok, seed=2)
    index, weights = index.cuda(), weights.cuda()
    file = io.BytesIO()
    torch.save(quant, file)
    file.seek(0)
    with torch.no_grad():
        want = quant(hidden, index, weights)
        for other in (copy.deepcopy(quant), torch.load(file, weights_only=False)):
            assert torch.equal(other(hidden, index, weights), want)
