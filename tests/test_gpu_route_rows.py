"""moe_route_rows (small batches: routing and the row-table dispatch in one pass)
against moe_router_fused followed by moe_dispatch_rows, bit for bit: ids, weights,
counts, offsets, slots, inverse and row table, at the edges of both its forms (one
workgroup for E <= 16; plane sums and a finishing workgroup above)."""

import pytest
import torch

from moe_dispatch.workspace import CudaWorkspace
from tests._helpers import gpu

pytestmark = gpu

CASES = [
    # tokens, hidden, experts, topk, alignment
    (1, 8, 1, 1, 1), (1, 4096, 8, 2, 8), (16, 4096, 8, 2, 8), (5, 72, 5, 3, 128), (16, 8192, 16, 8, 8),
    (15, 1032, 10, 4, 16), (2, 2048, 3, 2, 8), (16, 320, 12, 8, 1),
    (1, 2048, 64, 6, 8), (8, 2048, 64, 8, 8), (9, 1000, 17, 3, 8), (128, 4096, 64, 8, 128), (17, 8, 24, 1, 1),
    (100, 256, 33, 2, 8), (128, 2048, 48, 6, 64), (16, 1088, 32, 4, 8),
    # five fragments at the longest range; one token group at the shortest and longest ranges
    (13, 6152, 13, 4, 8), (5, 640, 20, 2, 8), (3, 4096, 40, 4, 16),
]


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("tokens,hidden,experts,topk,alignment", CASES)
def test_equals_router_and_row_dispatch(ext, tokens, hidden, experts, topk, alignment, ties):
    gen = torch.Generator(device="cuda").manual_seed(tokens * hidden + experts)
    x = torch.randn(tokens, hidden, device="cuda", generator=gen).bfloat16()
    if ties:  # zero logits: a bias of repeated values decides, ties to the lower expert
        x.zero_()
    w = torch.randn(experts, hidden, device="cuda", generator=gen) / hidden**0.5
    bias = torch.randint(0, 3, (experts,), device="cuda", generator=gen).float()
    scratch = torch.empty(ext.router_scratch_bytes(experts, hidden), dtype=torch.uint8, device="cuda")

    def buffers():
        ws = CudaWorkspace(tokens, hidden, experts, topk, torch.bfloat16, alignment=alignment, extension=ext)
        index = {n: getattr(ws, n).fill_(-7) for n in ("counts", "offsets", "slots", "inverse", "row_src")}
        return ws, index, [torch.full((tokens, topk), -7, device="cuda", dtype=d)
                           for d in (torch.int32, torch.int64, torch.float32)]

    ws_a, index_a, route_a = buffers()
    ext.router_fused_out(x, w, bias, *route_a, scratch=scratch)
    ws_a.dispatch_rows(route_a[0])
    ws_b, index_b, route_b = buffers()
    lib = ext.lib
    need = lib.moe_route_rows_scratch_bytes(tokens, hidden, experts, topk)
    assert (need == 0) == (experts <= 16) and need >= 0
    sums = torch.full((need + 16,), 0x5A, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for weight in (w.data_ptr(), None):  # with the split, then on the split the scratch holds
        for t in (*index_b.values(), *route_b):
            t.fill_(-7)
        status = lib.moe_route_rows(
            x.data_ptr(), weight, bias.data_ptr(), *[t.data_ptr() for t in route_b], scratch.data_ptr(),
            scratch.numel(), *[t.data_ptr() for t in index_b.values()], sums.data_ptr(), need, tokens, hidden,
            experts, topk, alignment, ws_b.capacity_rows, stream)
        lib.check(status, "moe_route_rows")
        for a, b in zip(route_a, route_b):
            assert torch.equal(a, b)
        for name in index_a:
            assert torch.equal(index_a[name], index_b[name]), name
    assert torch.all(sums[need:] == 0x5A)


def test_shapes_without_a_one_pass_route(ext):
    need = ext.lib.moe_route_rows_scratch_bytes
    assert need(17, 512, 16, 2) == -1 and need(1, 8200, 8, 2) == -1
    assert need(129, 512, 17, 2) == -1 and need(1, 4104, 17, 2) == -1 and need(128, 4096, 17, 8) > 0


# One call per selection form: E <= 16 in one workgroup, by direct loads, and
# E > 16. The logits are the biases (x is zero), so the selection is known exactly.
@pytest.mark.parametrize("tokens,experts", [(3, 8), (16, 16), (200, 8), (3, 40), (200, 64)])
@pytest.mark.parametrize("topk", [1, 2, 4, 7])
@pytest.mark.parametrize("kind", ["plus_inf", "minus_inf", "nan"])
def test_infinite_and_nan_logits(ext, tokens, experts, topk, kind):
    hidden = 256
    x = torch.zeros(tokens, hidden, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(experts, hidden, device="cuda")
    bias = torch.arange(experts, 0, -1, dtype=torch.float32) / 16  # the lower expert is the larger
    per_lane = 2 if experts <= 16 else 8
    if kind == "plus_inf":  # a pinned expert
        bias[experts - 1] = float("inf")
    elif kind == "minus_inf":  # masked experts, at least topk others left in use
        bias[: experts - topk] = float("-inf")
    else:  # the first expert of the second lane: never the largest in a comparison
        bias[per_lane] = float("nan")
    order = torch.where(bias.isnan(), torch.full_like(bias, float("-inf")), bias)
    want_ids = torch.sort(order, descending=True, stable=True).indices[:topk]
    picked = bias[want_ids].double()
    if topk <= 2 and kind == "plus_inf":
        want = torch.tensor([1.0, 0.0], dtype=torch.float64)[:topk]
    else:  # from top-3 on an infinite winner's own term is exp(inf - inf)
        want = torch.exp(picked - picked[0])
        want = want / want.sum()
    ids32 = torch.empty(tokens, topk, device="cuda", dtype=torch.int32)
    ids64, weights = ids32.long(), ids32.float()
    scratch = torch.empty(ext.router_scratch_bytes(experts, hidden), dtype=torch.uint8, device="cuda")
    ext.router_fused_out(x, w, bias.cuda(), ids32, ids64, weights, scratch=scratch)
    assert torch.equal(ids64.cpu(), want_ids.expand(tokens, topk))
    assert torch.equal(ids32.cpu().long(), ids64.cpu())
    # 32-bit exp, sum and product: a few units in the last place.
    torch.testing.assert_close(weights.cpu().double(), want.expand(tokens, topk), rtol=1e-6, atol=1e-9, equal_nan=True)
