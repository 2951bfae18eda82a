"""Block parity: MoEBlock(implementation="cuda_fused") against the CPU oracle.

Stage by stage, each stage fed the kernels' own inputs:
  * routing: ids equal the oracle's on exact fp32 logits wherever the K-th /
    (K+1)-th margin is not a near-tie (the fused router sums its dot products
    in its own order; selection on the kernel's logits is bit-exact in
    test_gpu_router.py); the downstream oracle uses the kernel's routing;
  * dispatch: counts, offsets, inverse and packed rows bit-exact (when the
    gate/up GEMM gathers its rows from x, which the block does from top-3 on
    with hidden a multiple of 64, the row table instead: each used row's
    token, -1 for padding; the GEMM oracle then reads x through it);
  * gate/up + SwiGLU and down GEMM: at least 99.99% of elements identical to
    the MFMA-order oracle, the rest within 2 bf16 steps;
  * combine: bit-exact.
End to end: max-abs <= 1.6e-2 and relative L2 <= 5e-4
against the expert-major oracle with the kernels' accumulation order (at the
full sizes C3 T=4096, C4 T=4096 and C5 on a token sample, whose routing and
k-order combine the oracle replays), and
against the independent token-major oracle with exact float64 dot products
(at I=14336 that last bound is 2e-3: two fp32 summation orders disagree there
by ~1e-3, because a few one-step bf16 flips of the activation perturb every
expert output element of their token and flip ~6% of its bf16 roundings).
The reference's own gate (tests/test_gpu.py:43-48 -> check_forward, rtol = atol
= 3e-2, rel-L2 <= 2e-2) is implied by these bounds.
"""

import numpy as np
import pytest
import torch

from moe_dispatch.layer import GATE_UP_ROW_PADDING, MoEBlock, MoEConfig, make_weights, padded_weight
from oracle import moe_oracle as oracle
from tests._helpers import LazyExpertWeights, assert_near_bit_exact, gpu, rel_l2, route_margin, to_np

pytestmark = gpu

MAX_ABS = 1.6e-2
REL_L2 = 5e-4
REL_L2_LARGE_I = 2e-3  # exact-arithmetic comparison at I=14336 (see module docstring)


def _run_block(cfg, tokens, pattern, seed, bias=None):
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=seed)
    if bias is not None:
        block.set_routing_bias(torch.tensor(bias))
    else:
        block.set_routing_pattern(pattern)
    x = torch.randn(tokens, cfg.hidden, generator=torch.Generator().manual_seed(seed + 1)).bfloat16().cuda()
    out = block(x).clone()
    ids32, _, weights = block._route_buffers[(tokens, x.device)]
    state = block.workspace(x)
    torch.cuda.synchronize()
    return block, x, out, ids32, weights, state


def _gate_up_rows(block, x, transport, layout, topk):
    """The rows the gate/up GEMM read: the packed copy, or for a gathered forward
    (no copy) x through the row table, which must map every used row to its
    token and every padding row to -1."""
    used = int(layout["offsets"][-1])
    if not block._launches[(x.shape[0], x.device)].gathered:
        return transport.packed
    src = transport.row_src[:used]
    expected = np.full(used, -1, np.int64)
    inverse = layout["inverse"].reshape(-1)
    expected[inverse] = np.arange(inverse.size) // topk
    np.testing.assert_array_equal(to_np(src), expected)
    rows = torch.zeros_like(transport.packed)
    ok = src >= 0
    rows[:used][ok] = x.index_select(0, src[ok].long())
    return rows


def _check_block(cfg, tokens, pattern="balanced", seed=0, bias=None, large_i=False):
    block, x, out, ids32, weights, state = _run_block(cfg, tokens, pattern, seed, bias)
    xf = to_np(x)
    router_w = to_np(block.router_weight)
    bias_np = to_np(block.routing_bias)
    gate_up = LazyExpertWeights(block.gate_up_weight)
    down = LazyExpertWeights(block.down_weight)
    ids = to_np(ids32)
    w = to_np(weights)
    # Routing against exact logits (near-ties excepted).
    logits = oracle.router_logits(xf, router_w)
    ids_ref, w_ref, _ = oracle.topk_route(logits, bias_np, cfg.topk)
    safe = route_margin(logits, bias_np, cfg.topk) > 1e-4
    # Near-ties are rare: at most 1% of the tokens (or one) are left out.
    assert (~safe).sum() <= max(1, 0.01 * tokens) or tokens < 20
    np.testing.assert_array_equal(ids[safe], ids_ref[safe])
    np.testing.assert_allclose(w[safe], w_ref[safe], rtol=0, atol=2e-5)
    # Dispatch, bit-exact.
    transport = state.transport
    layout = oracle.dispatch_layout(ids, cfg.experts, cfg.alignment)
    np.testing.assert_array_equal(to_np(transport.counts), layout["counts"])
    np.testing.assert_array_equal(to_np(transport.offsets), layout["offsets"])
    np.testing.assert_array_equal(to_np(transport.inverse), layout["inverse"])
    used = int(layout["offsets"][-1])
    rows = transport.capacity_rows
    packed_ref, _ = oracle.pack(xf, layout, cfg.topk, rows)
    packed = to_np(_gate_up_rows(block, x, transport, layout, cfg.topk))
    np.testing.assert_array_equal(packed[:used], packed_ref[:used])
    offsets = layout["offsets"]
    # Expert GEMMs, each on the kernels' own input.
    act = to_np(state.activated)
    proj_ref = oracle.bf16_round(oracle.grouped_gemm(packed[:used], gate_up, offsets))
    assert_near_bit_exact(act[:used], oracle.swiglu(proj_ref, used), max_fraction=2e-4, max_steps=2.0)
    eo = to_np(state.expert_output)
    eo_ref = oracle.bf16_round(oracle.grouped_gemm(act[:used], down, offsets))
    assert_near_bit_exact(eo[:used], eo_ref, max_fraction=1e-4)
    # Combine, bit-exact on the kernels' expert output.
    got = to_np(out)
    np.testing.assert_array_equal(got, oracle.combine(eo, layout["inverse"], w))
    # End to end.
    ref = oracle.block_forward(xf, router_w, bias_np, gate_up, down, cfg.topk, cfg.alignment, ids=ids, weights=w)
    expect = ref["output"]
    assert float(np.abs(got - expect).max()) <= MAX_ABS
    assert rel_l2(got, expect) <= REL_L2
    dense = oracle.token_major_forward(xf, gate_up, down, ids, w, order="exact")
    assert float(np.abs(got - dense).max()) <= MAX_ABS
    assert rel_l2(got, dense) <= (REL_L2_LARGE_I if large_i else REL_L2)
    return layout["counts"]


@pytest.mark.parametrize("tokens", [1, 13, 33, 200])
@pytest.mark.parametrize("pattern", ["balanced", "skewed"])
@pytest.mark.parametrize("topk", [1, 2])
def test_small_blocks(tokens, pattern, topk):
    _check_block(MoEConfig(32, 64, 8, topk), tokens, pattern)


@pytest.mark.parametrize("cfg,tokens", [
    ((64, 128, 1, 1), 50),         # one expert, top-1
    ((128, 64, 8, 8), 40),         # top-8 of 8: every token on every expert (row table)
    ((72, 136, 12, 3), 60),        # hidden and intermediate not multiples of 64: packed rows
    ((64, 64, 64, 8), 30),         # E=64, top-8, few tokens: most experts empty (row table)
    ((128, 128, 4, 2, 128), 100),  # alignment 128: most packed rows are padding
    ((128, 256, 8, 2), 2048),      # H=128: the down GEMM's 128-column halves past its last column
])
def test_block_edge_configurations(cfg, tokens):
    _check_block(MoEConfig(*cfg), tokens, seed=tokens)


def test_config1_cpu_reference_shape():
    """T=128, H=512, I=1024, E=8, top-2 (the reference's CPU-runnable case)."""
    _check_block(MoEConfig(512, 1024, 8, 2), 128, seed=0)


@pytest.mark.parametrize("tokens", [256, 1024])
def test_config3_sweep(tokens):
    """H=1024, I=2048, E=16, top-2."""
    _check_block(MoEConfig(1024, 2048, 16, 2), tokens, seed=tokens)


def test_config5_fine_grained_skewed_small():
    """E=64, top-6, Zipf router bias (empty and hot experts), at a reduced token count."""
    bias = oracle.zipf_bias(64, exponent=1.2, scale=1.75, seed=0)
    counts = _check_block(MoEConfig(256, 128, 64, 6), 512, bias=bias)
    assert (counts == 0).sum() >= 3


def test_block_is_deterministic():
    cfg = MoEConfig(256, 512, 16, 2)
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    x = torch.randn(777, 256, device="cuda").bfloat16()
    first = block(x).clone()
    second = block(x).clone()
    assert torch.equal(first, second)


def test_router_weight_updates_are_seen():
    """The fused router keeps the bf16 split of its weights between calls; an
    in-place update or a new tensor must still route with the new weights."""
    cfg = MoEConfig(256, 512, 16, 2)
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    twin = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    x = torch.randn(300, 256, device="cuda").bfloat16()
    block(x)
    block(x)
    gen = torch.Generator(device="cuda").manual_seed(9)
    for replace in (False, True):
        new_w = torch.randn(16, 256, device="cuda", generator=gen) / 16
        if replace:
            block.router_weight = new_w.clone()
        else:
            block.router_weight.copy_(new_w)
        twin.router_weight = new_w.clone()
        assert torch.equal(block(x), twin(x))


def test_fast_path_rechecks_a_replaced_router_weight():
    """After the pre-validated launches are in use, a router weight of another dtype,
    shape or layout is caught by the validating path (RuntimeError), never read as
    fp32 [E,H]; putting the original back restores the same output."""
    cfg = MoEConfig(256, 512, 8, 2)
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    x = torch.randn(100, 256, device="cuda").bfloat16()
    first = block(x).clone()
    assert torch.equal(block(x), first) and (100, x.device) in block._launches
    good = block.router_weight
    wrong = [good.bfloat16(), torch.randn(8, 264, device="cuda"), torch.randn(9, 256, device="cuda"),
             good.t().contiguous().t()]
    for bad in wrong:
        block.router_weight = bad
        with pytest.raises(RuntimeError):
            block(x)
    block.router_weight = good
    assert torch.equal(block(x), first)
    torch.cuda.synchronize()


def test_capture_right_after_a_router_update_leaves_eager_calls_correct():
    """A capture records the router split without running it; the next eager forward
    must split again rather than trust planes the capture never wrote."""
    cfg = MoEConfig(256, 512, 8, 2)
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=4)
    twin = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=4)
    gen = torch.Generator(device="cuda").manual_seed(8)
    x = torch.randn(64, 256, device="cuda", generator=gen).bfloat16()
    block(x)
    block(x)
    new_w = torch.randn(8, 256, device="cuda", generator=gen) / 16
    block.router_weight.copy_(new_w)
    twin.router_weight = new_w.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        block(x)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    assert torch.equal(block(x).clone(), twin(x))
    del graph


@pytest.mark.parametrize("cfg,tokens,bias", [
    (MoEConfig(512, 1024, 8, 2), 128, None),
    (MoEConfig(256, 512, 16, 2), 777, "skewed"),
    (MoEConfig(256, 128, 64, 6), 300, "zipf"),
])
def test_repeat_calls_match_validated_calls(cfg, tokens, bias):
    """After its first (validated) forward a block reuses the checked launch
    arguments; those forwards must equal a fresh block's validated forward."""
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=5)
    if bias == "skewed":
        block.set_routing_pattern("skewed")
    elif bias == "zipf":
        block.set_routing_bias(torch.tensor(oracle.zipf_bias(cfg.experts, exponent=1.2, scale=1.75, seed=0)))
    gen = torch.Generator(device="cuda").manual_seed(7)
    inputs = [torch.randn(tokens, cfg.hidden, device="cuda", generator=gen).bfloat16() for _ in range(3)]
    first = block(inputs[0]).clone()
    assert (tokens, inputs[0].device) in block._launches
    assert torch.equal(block(inputs[0]), first)
    for x in inputs[1:]:
        fresh = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=5)
        fresh.routing_bias.copy_(block.routing_bias)
        assert torch.equal(block(x).clone(), fresh(x))


def test_repeat_calls_follow_weight_changes_and_streams():
    cfg = MoEConfig(256, 512, 8, 2)
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=2)
    twin = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=2)
    x = torch.randn(200, 256, device="cuda").bfloat16()
    block(x)
    block(x)
    gen = torch.Generator(device="cuda").manual_seed(4)
    # A new expert weight tensor (another address): the launches are rebuilt.
    new_gate_up = (torch.randn(8, 1024, 256, device="cuda", generator=gen) / 16).bfloat16()
    block.gate_up_weight = new_gate_up.clone()
    twin.gate_up_weight = new_gate_up.clone()
    assert torch.equal(block(x).clone(), twin(x))
    # In-place updates of the down weights and the bias keep the addresses.
    new_down = (torch.randn(8, 256, 512, device="cuda", generator=gen) / 22).bfloat16()
    block.down_weight.copy_(new_down)
    twin.down_weight.copy_(new_down)
    block.set_routing_pattern("skewed")
    twin.set_routing_pattern("skewed")
    assert torch.equal(block(x).clone(), twin(x))
    # Launches go to the current stream.
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = block(x).clone()
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(out, twin(x))


@pytest.mark.parametrize("cfg", [MoEConfig(4096, 256, 8, 2), MoEConfig(4096, 192, 16, 6)])
def test_padded_gate_up_rows_equal_contiguous_weights(cfg):
    """H = 4096: the fused block keeps its gate/up rows padded (8 KiB rows). Its
    forward equals a twin's whose gate/up weights are a contiguous copy, bit for
    bit, on the weight-streaming and persistent paths (and at top-6 the gathered
    gate/up GEMM); in-place updates through the padded view reach the kernels."""
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    assert block.gate_up_weight.stride(1) == cfg.hidden + GATE_UP_ROW_PADDING
    twin = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    twin.gate_up_weight = block.gate_up_weight.contiguous()
    gen = torch.Generator(device="cuda").manual_seed(5)
    for tokens in (1, 16, 700):
        x = torch.randn(tokens, cfg.hidden, device="cuda", generator=gen).bfloat16()
        assert torch.equal(block(x).clone(), twin(x)), tokens
    new = (torch.randn(block.gate_up_weight.shape, device="cuda", generator=gen) / 45).bfloat16()
    block.gate_up_weight.copy_(new)
    twin.gate_up_weight.copy_(new)
    x = torch.randn(300, cfg.hidden, device="cuda", generator=gen).bfloat16()
    assert torch.equal(block(x).clone(), twin(x))


@pytest.mark.parametrize("cfg", [MoEConfig(2048, 256, 8, 2), MoEConfig(128, 4096, 8, 2), MoEConfig(2048, 2048, 16, 6)])
def test_padded_weight_rows_equal_contiguous_weights(cfg):
    """Gate/up or down rows of a multiple of 4 KiB moved to row-padded storage: the forward
    equals that of a twin with contiguous copies, bit for bit, and in-place updates reach
    the kernels."""
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    twin = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    for name, k in (("gate_up_weight", cfg.hidden), ("down_weight", cfg.intermediate)):
        setattr(block, name, padded_weight(getattr(block, name)))
        assert getattr(block, name).stride(1) == (k + GATE_UP_ROW_PADDING if k % 2048 == 0 else k)
        setattr(twin, name, getattr(block, name).contiguous())
    gen = torch.Generator(device="cuda").manual_seed(5)
    for tokens in (1, 20, 700):
        x = torch.randn(tokens, cfg.hidden, device="cuda", generator=gen).bfloat16()
        assert torch.equal(block(x).clone(), twin(x)), tokens
    new = (torch.randn(block.down_weight.shape, device="cuda", generator=gen) / 45).bfloat16()
    block.down_weight.copy_(new)
    twin.down_weight.copy_(new)
    x = torch.randn(300, cfg.hidden, device="cuda", generator=gen).bfloat16()
    assert torch.equal(block(x).clone(), twin(x))


@pytest.mark.parametrize("cfg", [MoEConfig(2048, 256, 8, 2), MoEConfig(4096, 2048, 8, 2), MoEConfig(6144, 512, 4, 1)])
def test_given_weights_are_shared(cfg):
    """A fused block keeps the storage of the weights it is given (gate/up rows of a power
    of two bytes of at least 8 KiB aside, which it pads): no second copy, and the owner's
    in-place updates reach the kernels, also between blocks that share them."""
    weights = make_weights(cfg, "cuda", torch.bfloat16, 3)
    blocks = [MoEBlock(cfg, device="cuda", implementation="cuda_fused", weights=weights) for _ in range(2)]
    shared = ["router", "down"] + (["gate_up"] if cfg.hidden != 4096 else [])
    for block in blocks:
        for name in shared:
            tensor = getattr(block, name + "_weight")
            assert tensor.data_ptr() == getattr(weights, name).data_ptr() and tensor.is_contiguous(), name
    x = torch.randn(20, cfg.hidden, device="cuda").bfloat16()
    first = [block(x).clone() for block in blocks]
    for name in shared[1:]:
        getattr(weights, name).mul_(-0.5)
    twin = MoEBlock(cfg, device="cuda", implementation="cuda_fused", weights=weights)
    if "gate_up" not in shared:
        twin.gate_up_weight = blocks[0].gate_up_weight
    want = twin(x).clone()
    assert not torch.equal(want, first[0])
    for block in blocks:
        assert torch.equal(block(x), want)


def test_native_forward_follows_replaced_parameters():
    """The one-call forward is used while the tensors are the bound ones: a parameter set
    over a buffer, a resized storage and a wrong input go back through the checks."""
    cfg = MoEConfig(128, 192, 8, 2)
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    x = torch.randn(40, 128, device="cuda").bfloat16()
    block(x)
    down = (torch.randn(8, 128, 192, device="cuda") / 14).bfloat16()
    block.down_weight = torch.nn.Parameter(down, requires_grad=False)
    twin = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=3)
    twin.down_weight.copy_(down)
    want = twin(x).clone()
    for _ in range(3):
        assert torch.equal(block(x), want)
    assert block._launches[(40, x.device)].still_valid(block)
    block.down_weight.data = torch.zeros_like(down)
    assert torch.all(block(x) == 0)
    for bad in (x[:, :64], x.float(), x.t().contiguous().t(), x.cpu()):
        with pytest.raises(ValueError):
            block(bad)


def test_empty_batch():
    block = MoEBlock(MoEConfig(64, 128, 8, 2), device="cuda", implementation="cuda_fused")
    out = block(torch.empty(0, 64, device="cuda", dtype=torch.bfloat16))
    assert out.shape == (0, 64)


def test_variants_agree():
    """The three implementations share weights; outputs agree within bf16 tolerance."""
    cfg = MoEConfig(128, 256, 8, 2)
    fused = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=5)
    weights = None
    from moe_dispatch.layer import MoEWeights

    weights = MoEWeights(fused.router_weight, fused.gate_up_weight, fused.down_weight)
    x = torch.randn(300, 128, device="cuda").bfloat16()
    outs = {"cuda_fused": fused(x).clone()}
    for impl in ("cuda", "torch"):
        block = MoEBlock(cfg, device="cuda", implementation=impl, weights=weights,
                         expert_backend="hip" if impl == "cuda" else "torch")
        outs[impl] = block(x).clone()
    for impl in ("cuda", "torch"):
        diff = (outs[impl].float() - outs["cuda_fused"].float())
        assert float(diff.abs().max()) <= 3e-2
        assert float(diff.norm() / outs["cuda_fused"].float().norm()) <= 2e-2


@pytest.mark.parametrize("tokens", [1, 16])
def test_config4_decode_sizes_full_model_shape(tokens):
    """H=4096, I=14336, E=8, top-2 at decode token counts, full weights."""
    _check_block(MoEConfig(4096, 14336, 8, 2), tokens, seed=1, large_i=True)
    torch.cuda.empty_cache()


def _sample_rows(offsets, counts, per_expert, rng):
    """First, last and random rows of every non-empty expert span; sample offsets."""
    rows, sample_offsets = [], [0]
    for e in range(len(counts)):
        s, n = int(offsets[e]), int(counts[e])
        if n:
            pick = {0, n - 1} | set(rng.integers(0, n, size=max(per_expert - 2, 0)).tolist())
            rows.extend(s + r for r in sorted(pick))
        sample_offsets.append(len(rows))
    return np.asarray(rows, dtype=np.int64), np.asarray(sample_offsets, dtype=np.int64)


def _check_expert_span(state, block, packed_rows, offsets, counts, expert):
    """Both GEMMs over one whole expert span (every row, every column) against the
    MFMA-order oracle (the C checker), each on the kernels' own input."""
    lo, n = int(offsets[expert]), int(counts[expert])
    packed = to_np(packed_rows[lo:lo + n])
    act = to_np(state.activated[lo:lo + n])
    eo = to_np(state.expert_output[lo:lo + n])
    span = np.array([0, n])
    gate_up = to_np(block.gate_up_weight[expert])[None]
    proj_ref = oracle.bf16_round(oracle.grouped_gemm(packed, gate_up, span))
    del gate_up
    assert_near_bit_exact(act, oracle.swiglu(proj_ref, n), max_fraction=2e-4, max_steps=2.0)
    down = to_np(block.down_weight[expert])[None]
    eo_ref = oracle.bf16_round(oracle.grouped_gemm(act, down, span))
    assert_near_bit_exact(eo, eo_ref, max_fraction=1e-4)


def _check_block_sampled(cfg, tokens, bias=None, large_i=False, per_expert=6, token_sample=48, seed=0,
                         full_span=False):
    """Full-size block: exact layout and permutation over all tokens; GEMMs, combine and
    end-to-end output on sampled rows/tokens (rows of a GEMM are independent); with
    ``full_span``, both GEMMs over the whole span of the expert with the fewest rows."""
    block, x, out, ids32, weights, state = _run_block(cfg, tokens, "balanced", seed, bias)
    rng = np.random.default_rng(seed)
    transport = state.transport
    ids, w = to_np(ids32), to_np(weights)
    # Routing on a token sample against exact logits (near-ties excepted).
    tsample = np.sort(rng.choice(tokens, size=min(token_sample, tokens), replace=False))
    router_w, bias_np = to_np(block.router_weight), to_np(block.routing_bias)
    xs = to_np(x[torch.from_numpy(tsample).cuda()])
    logits = oracle.router_logits(xs, router_w)
    ids_ref, w_ref, _ = oracle.topk_route(logits, bias_np, cfg.topk)
    safe = route_margin(logits, bias_np, cfg.topk) > 1e-4
    np.testing.assert_array_equal(ids[tsample][safe], ids_ref[safe])
    np.testing.assert_allclose(w[tsample][safe], w_ref[safe], rtol=0, atol=2e-5)
    # Dispatch over every token: layout bit-exact, permutation and padding.
    layout = oracle.dispatch_layout(ids, cfg.experts, cfg.alignment)
    np.testing.assert_array_equal(to_np(transport.counts), layout["counts"])
    np.testing.assert_array_equal(to_np(transport.offsets), layout["offsets"])
    np.testing.assert_array_equal(to_np(transport.inverse), layout["inverse"])
    np.testing.assert_array_equal(to_np(transport.slots).reshape(-1), layout["slots"])
    packed_rows = _gate_up_rows(block, x, transport, layout, cfg.topk)
    inv = transport.inverse.reshape(-1).long()
    gathered = packed_rows.index_select(0, inv).view(tokens, cfg.topk, cfg.hidden)
    assert torch.equal(gathered, x[:, None, :].expand_as(gathered))
    offsets, counts = layout["offsets"], layout["counts"]
    for e in range(cfg.experts):
        pad = packed_rows[int(offsets[e]) + int(counts[e]):int(offsets[e + 1])]
        assert int(torch.count_nonzero(pad)) == 0
    # Expert GEMMs on sampled rows of every expert, each on the kernels' own input.
    rows, sample_offsets = _sample_rows(offsets, counts, per_expert, rng)
    rows_t = torch.from_numpy(rows).cuda()
    gate_up, down = LazyExpertWeights(block.gate_up_weight), LazyExpertWeights(block.down_weight)
    packed_s = to_np(packed_rows.index_select(0, rows_t))
    act_s = to_np(state.activated.index_select(0, rows_t))
    proj_ref = oracle.bf16_round(oracle.grouped_gemm(packed_s, gate_up, sample_offsets))
    assert_near_bit_exact(act_s, oracle.swiglu(proj_ref, len(rows)), max_fraction=2e-4, max_steps=2.0)
    eo_s = to_np(state.expert_output.index_select(0, rows_t))
    eo_ref = oracle.bf16_round(oracle.grouped_gemm(act_s, down, sample_offsets))
    assert_near_bit_exact(eo_s, eo_ref, max_fraction=1e-4)
    # Combine on sampled tokens, bit-exact on the kernels' expert output.
    inv_s = layout["inverse"][tsample]
    needed = np.unique(inv_s)
    eo_rows = np.zeros((transport.capacity_rows, cfg.hidden), np.float32)
    eo_rows[needed] = to_np(state.expert_output.index_select(0, torch.from_numpy(needed).cuda()))
    got = to_np(out)[tsample]
    np.testing.assert_array_equal(got, oracle.combine(eo_rows, inv_s, w[tsample]))
    # End to end on the token sample, the north-star bounds against the oracle with
    # the kernels' rounding points and accumulation order (the sampled tokens'
    # routing, k-order combine) ...
    xs_all = to_np(x)[tsample]
    ordered = oracle.block_forward(xs_all, router_w, bias_np, gate_up, down, cfg.topk, 1, ids=ids[tsample],
                                   weights=w[tsample])["output"]
    assert float(np.abs(got - ordered).max()) <= MAX_ABS
    assert rel_l2(got, ordered) <= REL_L2
    # ... and against the exact-arithmetic token-major oracle (see the module docstring).
    dense = oracle.token_major_forward(to_np(x), gate_up, down, ids, w, token_index=tsample, order="exact")
    assert float(np.abs(got - dense).max()) <= MAX_ABS
    assert rel_l2(got, dense) <= (REL_L2_LARGE_I if large_i else REL_L2)
    if full_span:
        # The expert with the fewest rows, and (when there is one) the smallest
        # of more than 256 rows: several full-height row tiles of one expert.
        nonempty = [e for e in range(cfg.experts) if counts[e] > 0]
        spans = {min(nonempty, key=lambda e: counts[e])}
        tall = [e for e in nonempty if counts[e] > 256]
        if tall:
            spans.add(min(tall, key=lambda e: counts[e]))
        for e in sorted(spans):
            _check_expert_span(state, block, packed_rows, offsets, counts, e)
    return counts


def test_config4_prefill_full_size_sampled():
    """C4 at T=4096 (the benchmark workload): full layout, sampled GEMM rows and tokens,
    and one whole expert span of both GEMMs."""
    _check_block_sampled(MoEConfig(4096, 14336, 8, 2), 4096, large_i=True, full_span=True)


def test_config3_t4096_full_size_sampled():
    _check_block_sampled(MoEConfig(1024, 2048, 16, 2), 4096)


def test_config5_full_size_zipf_skew():
    """C5: T=8192, H=2048, I=1408, E=64, top-6 with the Zipf router bias: several experts
    get no tokens and a few take more than 15% of the assignments. Whole expert spans
    of both GEMMs (the gate/up one gathering its rows from x) are checked too."""
    cfg = MoEConfig(2048, 1408, 64, 6)
    counts = _check_block_sampled(cfg, 8192, bias=oracle.zipf_bias(64), full_span=True)
    assert int((counts == 0).sum()) >= 3
    assert int((counts > 0.15 * 8192 * 6).sum()) >= 2


def test_first_forward_of_a_token_count_asks_the_library_once(monkeypatch):
    """A new token count pays for its buffers, its operators and one argument struct: one
    query of the one-pass route, and no argument tuples for the stages (stage_calls
    makes those for whoever times them)."""
    cfg = MoEConfig(512, 256, 64, 6)
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=0)
    lib = block._extension.lib
    real, calls = lib.moe_route_rows_scratch_bytes, []
    monkeypatch.setattr(lib, "moe_route_rows_scratch_bytes", lambda *a: calls.append(a) or real(*a))
    for tokens in (5, 300):
        x = torch.randn(tokens, cfg.hidden, device="cuda").bfloat16()
        calls.clear()
        block(x)
        block(x)
        assert calls == [(tokens, cfg.hidden, cfg.experts, cfg.topk)]
        launches = block._launches[(tokens, x.device)]
        pairs = {name: value for name, value in vars(launches).items() if isinstance(value, tuple)}
        assert set(pairs) == {"fingerprint", "keep"}, set(pairs)
        # Every field of the packed arguments under its name in the header.
        args, state = launches.args, block.workspace(x)
        t, (ids32, ids64, weights) = state.transport, block._route_buffers[(tokens, x.device)]
        pointers = {"bias": block.routing_bias, "ids32": ids32, "ids64": ids64, "weights": weights,
                    "router_scratch": block._router_scratch, "counts": t.counts, "offsets": t.offsets,
                    "slots": t.slots, "inverse": t.inverse, "row_src": t.row_src, "packed": t.packed,
                    "dispatch_scratch": t.scratch, "ranks": t.tile_ranks, "tile_counts": t.tile_counts,
                    "sums": state.plane_sums, "gate_up": block.gate_up_weight, "down": block.down_weight,
                    "activated": state.activated, "expert_output": state.expert_output, "output": t.output}
        sizes = {"struct_bytes": 8 * len(args._ORDER), "router_scratch_bytes": block._router_scratch.numel(),
                 "dispatch_scratch_bytes": t.scratch.numel(), "tile_counts_bytes": 4 * t.tile_counts.numel(),
                 "tile_tokens": t.rank_tile, "sums_bytes": 0 if state.plane_sums is None else state.plane_sums.numel(),
                 "gate_up_row_stride": cfg.hidden, "down_row_stride": cfg.intermediate, "tokens": tokens,
                 "hidden": cfg.hidden, "intermediate": cfg.intermediate, "experts": cfg.experts, "topk": cfg.topk,
                 "alignment": cfg.alignment, "packed_rows": t.capacity_rows, "vectorized": 1,
                 "gathered": 1, "one_pass": int(tokens == 5)}
        want = {name: v.data_ptr() if v is not None else None for name, v in pointers.items()} | sizes
        assert {name: getattr(args, name) for name in args._ORDER} == want


@pytest.mark.parametrize("cfg,tokens,first", [
    (MoEConfig(512, 256, 64, 6), 40, ["route"]),              # one-pass route with plane sums
    (MoEConfig(512, 256, 8, 2), 7, ["route"]),                # one-pass route in one workgroup
    (MoEConfig(512, 256, 8, 2), 200, ["router", "dispatch"]),  # ranked, packed
    (MoEConfig(512, 256, 8, 4), 200, ["router", "dispatch"]),  # ranked, gathered
    (MoEConfig(128, 64, 64, 2), 3000, ["router", "dispatch"]),  # counted, packed
    (MoEConfig(128, 64, 64, 6), 3000, ["router", "dispatch"]),  # counted, gathered
])
def test_stage_calls_are_the_forwards_own(monkeypatch, cfg, tokens, first):
    """The timed stages make the calls that the forward makes, in its order and with its
    arguments: run one after another on cleared buffers they give its output."""
    block = MoEBlock(cfg, device="cuda", implementation="cuda_fused", seed=0)
    x = torch.randn(tokens, cfg.hidden, device="cuda").bfloat16()
    block(x)
    want = block(x).clone()
    launches = block._launches[(tokens, x.device)]
    assert (launches.args.one_pass == 1) == (first == ["route"])
    stages = launches.stage_calls(x)
    assert list(stages) == first + ["gateup_swiglu", "down", "combine"]
    state = block.workspace(x)
    with torch.inference_mode():
        buffers = [t for t in vars(state.transport).values() if isinstance(t, torch.Tensor)]
        for t in buffers + [state.activated, state.expert_output, *block._route_buffers[(tokens, x.device)]]:
            t.zero_()
    for run in stages.values():
        run()
    assert torch.equal(launches.output, want)
