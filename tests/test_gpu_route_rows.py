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
