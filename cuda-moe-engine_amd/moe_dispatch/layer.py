"""A complete single-GPU MoE feed-forward block with matched implementation variants.

Mirrors ``src/moe_dispatch/layer.py:12-214``: ``MoEConfig``, ``MoEWeights``,
``make_weights``, ``LayerWorkspace``, ``MoEBlock`` (``route``, ``workspace``,
``experts_forward``, ``forward``, ``set_routing_pattern``) and
``token_major_oracle``. Implementations:

* ``cuda_fused``: HIP fused router (fp32 logits + bias + top-k + softmax),
  HIP dispatch, HIP gate/up GEMM with the SwiGLU epilogue, HIP down GEMM, HIP
  combine. The drop-in for the reference's ``cuda_fused``.
* ``cuda``: PyTorch router, HIP transport, HIP GEMMs with a separate
  PyTorch SwiGLU.
* ``torch``: the PyTorch variant (CPU or GPU), used as the baseline.

Top-k may be 1..8 (the reference allows 1 or 2); ``set_routing_bias`` sets an
arbitrary router bias.
"""

from array import array
from dataclasses import dataclass
import math

import torch

from . import _lib
from ._extension import current_stream_handle, get_extension, weight_row_stride
from .experts import grouped_linear, resolve_backend, swiglu_reference
from .reference import TorchWorkspace
from .workspace import MAX_EXPERTS, MAX_TOPK, CudaWorkspace

IMPLEMENTATIONS = ("torch", "cuda", "cuda_fused")


@dataclass(frozen=True)
class MoEConfig:
    hidden: int = 512
    intermediate: int = 1024
    experts: int = 8
    topk: int = 2
    alignment: int = 8

    def __post_init__(self):
        if self.hidden < 8 or self.intermediate < 8:
            raise ValueError("hidden/intermediate must be at least 8")
        if self.hidden % 8 or self.intermediate % 8:
            raise ValueError("grouped GEMM dimensions must be multiples of 8")
        if (
            not 1 <= self.experts <= MAX_EXPERTS
            or not 1 <= self.topk <= MAX_TOPK
            or self.topk > self.experts
        ):
            raise ValueError("invalid expert/topk configuration")
        if not 8 <= self.alignment <= 128 or self.alignment % 8:
            raise ValueError("full-block grouped GEMM alignment must be a multiple of 8 up to 128")


@dataclass
class MoEWeights:
    router: torch.Tensor
    gate_up: torch.Tensor
    down: torch.Tensor


def _capturing():
    return torch.cuda.is_available() and torch.cuda.is_current_stream_capturing()


def make_weights(config, device, dtype, seed=42):
    """Seeded weights, drawn in the reference's order (``layer.py:38-59``).

    router ``[E,H]`` fp32 ~ N(0,1/H); gate_up ``[E,2I,H]`` ~ N(0,1/H) and down
    ``[E,H,I]`` ~ N(0,1/I), both cast to ``dtype``.
    """
    generator = torch.Generator(device=device).manual_seed(seed)
    e, h, i = config.experts, config.hidden, config.intermediate
    router = torch.randn(e, h, device=device, generator=generator) / math.sqrt(h)
    gate_up = (torch.randn(e, 2 * i, h, device=device, generator=generator) / math.sqrt(h)).to(dtype)
    down = (torch.randn(e, h, i, device=device, generator=generator) / math.sqrt(i)).to(dtype)
    return MoEWeights(router, gate_up, down)


# Elements of padding after each row of a row-padded expert weight. The GEMMs read
# every row of a tile, on every CU, at the same k offset at once, and rows a
# multiple of WEIGHT_ROW_CONFLICT bytes apart then fall on the same memory
# channels. Measured, padded against contiguous rows: gate/up at H=2048, I=4096,
# 16 experts, 128 rows 121.6 -> 93.0 us (4.4 -> 5.8 TB/s) and at H=2048, I=1408, 64
# experts, 288 rows 139.2 -> 125.2; at H=4096, I=14336, 8 experts, 2 rows 90.0 ->
# 80.3 and 32 rows 338 -> 302; down at I=14336 (7 x 4 KiB) with 32 rows 182 -> 158
# and 666 rows 217 -> 206. Full prefill is unchanged (4096 tokens at H=4096: 1447
# and 1441 us). Rows of 2 KiB multiples gained 1-8% at H=1024 with few rows and
# nothing with many; rows of other lengths do not conflict. The results are the
# same bit for bit (each output is the same MFMA chain).
GATE_UP_ROW_PADDING = 64
WEIGHT_ROW_CONFLICT = 4096


def _row_padded(weight):
    e, n, k = weight.shape
    storage = torch.zeros(e, n, k + GATE_UP_ROW_PADDING, device=weight.device, dtype=weight.dtype)
    storage[:, :, :k].copy_(weight)
    return storage[:, :, :k]


def padded_gate_up(weight):
    """``weight`` ([E, 2I, H]) as a ``[:, :, :H]`` view of row-padded storage when its
    rows are a power of two bytes of at least 8 KiB, else contiguous: the layout the
    fused block gives its gate/up weights. Every other weight keeps the storage it
    was given, which its owner may share between blocks or update in place."""
    row_bytes = weight.shape[2] * weight.element_size()
    if row_bytes < 8192 or row_bytes & (row_bytes - 1):
        return weight.contiguous()
    return _row_padded(weight)


def padded_weight(weight):
    """``weight`` ([E, N, K]) as a ``[:, :, :K]`` view of row-padded storage when its
    rows are a multiple of WEIGHT_ROW_CONFLICT bytes and one expert stays below the
    GEMMs' 4 GiB with the padding, else contiguous. For a program that has no other
    use of the tensor: ``block.down_weight = padded_weight(block.down_weight)`` (and
    ``gate_up_weight``) moves a fused block's weights to storage of their own."""
    _, n, k = weight.shape
    size = weight.element_size()
    if k * size % WEIGHT_ROW_CONFLICT or n * (k + GATE_UP_ROW_PADDING) * size >= 2**32:
        return weight.contiguous()
    return _row_padded(weight)


@dataclass
class LayerWorkspace:
    transport: object
    projection: torch.Tensor
    activated: torch.Tensor
    expert_output: torch.Tensor
    one_pass: bool = False  # the fused forward routes through moe_route_rows
    # Its plane sums, where the shape needs any: a captured graph holds their address,
    # so like every buffer here they live as long as the block.
    plane_sums: torch.Tensor | None = None


class MoEBlock(torch.nn.Module):
    """Inference-only top-k MoE: router, dispatch, two grouped GEMMs, SwiGLU, combine.

    Output is a reusable view: clone it before the next call.
    """

    def __init__(
        self,
        config=None,
        *,
        device="cuda",
        dtype=torch.bfloat16,
        implementation="cuda_fused",
        expert_backend="auto",
        seed=42,
        weights=None,
    ):
        super().__init__()
        self.config = config or MoEConfig()
        if implementation not in IMPLEMENTATIONS:
            raise ValueError("implementation must be torch, cuda, or cuda_fused")
        device = torch.device(device)
        if implementation != "torch" and device.type != "cuda":
            raise RuntimeError("HIP implementations require a GPU")
        if device.type == "cuda" and dtype != torch.bfloat16:
            raise ValueError("full GPU block uses BF16 grouped GEMMs")
        self.implementation = implementation
        backend = resolve_backend(device, expert_backend)
        if implementation != "torch" and backend != "hip":
            raise ValueError("HIP implementations use the HIP grouped GEMM (expert_backend='hip')")
        self.expert_backend = backend
        weights = weights or make_weights(self.config, device, dtype, seed)
        cfg = self.config
        if weights.gate_up.shape != (cfg.experts, 2 * cfg.intermediate, cfg.hidden) or (
            weights.down.shape != (cfg.experts, cfg.hidden, cfg.intermediate)
        ):
            raise ValueError("expert weights do not match the block configuration")
        if weights.router.shape != (cfg.experts, cfg.hidden):
            raise ValueError("router weights do not match the block configuration")
        self.register_buffer("router_weight", weights.router.contiguous())
        # The fused block pads power-of-two gate/up rows (padded_gate_up); the tensor is a
        # view of that storage, so in-place updates of it reach the kernels.
        gate_up = padded_gate_up(weights.gate_up) if implementation == "cuda_fused" else weights.gate_up.contiguous()
        self.register_buffer("gate_up_weight", gate_up)
        self.register_buffer("down_weight", weights.down.contiguous())
        self.register_buffer("routing_bias", torch.zeros(cfg.experts, device=device))
        self._workspaces = {}
        self._route_buffers = {}
        self._router_scratch = None  # bf16 split of the router weights (fused router)
        self._router_split_of = None  # _router_split_key() of the weights the split holds
        self._split_in_capture = True  # record the router split into captured graphs
        self._launches = {}  # cuda_fused: pre-validated launches per input signature
        self._extension = get_extension() if implementation != "torch" else None

    def set_routing_pattern(self, pattern):
        if pattern not in ("balanced", "skewed"):
            raise ValueError("routing pattern must be balanced or skewed")
        self.routing_bias.zero_()
        if pattern == "skewed":
            self.routing_bias[: self.config.topk] = 5.0

    def set_routing_bias(self, bias):
        """Set an arbitrary fp32 router bias ``[E]`` (e.g. a Zipf-shaped skew)."""
        bias = torch.as_tensor(bias, dtype=torch.float32)
        if bias.shape != (self.config.experts,):
            raise ValueError("routing bias must have shape [experts]")
        self.routing_bias.copy_(bias)

    def route(self, x):
        return self._route(x)

    def _route(self, x, ranked_into=None):
        """route(); with a CudaWorkspace whose shape has a ranked route
        (``rank_tile`` > 0), the fused router also writes that workspace's
        in-tile ranks and tile counts for its ``dispatch_ranked``."""
        if self.implementation == "cuda_fused":
            key = (x.shape[0], x.device)
            if key not in self._route_buffers:
                shape = (x.shape[0], self.config.topk)
                self._route_buffers[key] = (
                    torch.empty(shape, device=x.device, dtype=torch.int32),
                    torch.empty(shape, device=x.device, dtype=torch.int64),
                    torch.empty(shape, device=x.device, dtype=torch.float32),
                )
            ids32, ids64, weights = self._route_buffers[key]
            if self._router_scratch is None or self._router_scratch.device != x.device:
                need = self._extension.router_scratch_bytes(self.config.experts, self.config.hidden)
                self._router_scratch = torch.empty(need, dtype=torch.uint8, device=x.device)
                self._router_split_of = None
            router_weight, split_of = self._router_split_plan()
            weight = None if router_weight is None else self.router_weight
            if ranked_into is None:
                self._extension.router_fused_out(x, weight, self.routing_bias, ids32, ids64, weights,
                                                 scratch=self._router_scratch)
            else:
                self._extension.router_fused_ranked_out(x, weight, self.routing_bias, ids32, ids64, weights,
                                                        ranked_into.tile_ranks, ranked_into.tile_counts,
                                                        scratch=self._router_scratch)
            self._router_split_of = split_of
            return ids32, ids64, weights
        logits = torch.nn.functional.linear(x.float(), self.router_weight) + self.routing_bias
        selected, ids64 = torch.topk(logits, self.config.topk, dim=-1)
        weights = torch.softmax(selected, dim=-1).contiguous()
        return ids64.to(torch.int32).contiguous(), ids64.contiguous(), weights

    def _router_split_key(self):
        """Identity of the router weights the bf16 split was taken from.

        The key holds the tensor itself (so its storage cannot be freed and
        reused by another tensor at the same address while the key is kept),
        its address, version counter, dtype, shape and device. None when the
        tensor has no version counter (inference tensors): then every call splits.
        """
        w = self.router_weight
        try:
            version = w._version
        except RuntimeError:  # inference tensors do not count versions
            return None
        return (w, w.data_ptr(), version, w.dtype, tuple(w.shape), w.device)

    @staticmethod
    def _same_split(a, b):
        return a is not None and b is not None and a[0] is b[0] and a[1:] == b[1:]

    def _router_split_plan(self):
        """(router weight pointer or None, split key to record) for the next fused-router call.

        The bf16 split of the router weights is redone only when they may have
        changed (another tensor, or an in-place write, which bumps the version
        counter). Inside a graph capture it is recorded into the graph, so that
        every replay reads the weights as they are then, unless the capture is
        ``capture_forward``'s: its graph's replay() re-splits beforehand, and only
        when the weights changed. A recorded split runs only when the graph is
        replayed, so after recording one the split counts as stale.
        """
        split_of = self._router_split_key()
        capturing = _capturing()
        current = self._same_split(split_of, self._router_split_of)
        if current and not (capturing and self._split_in_capture):
            return None, split_of
        return self.router_weight.data_ptr(), (None if capturing else split_of)

    def workspace(self, x):
        key = (x.shape[0], x.dtype, x.device)
        if key not in self._workspaces:
            cfg = self.config
            common = (x.shape[0], cfg.hidden, cfg.experts, cfg.topk, x.dtype)
            if self.implementation == "torch":
                transport = TorchWorkspace(*common, device=x.device, alignment=cfg.alignment)
            else:
                transport = CudaWorkspace(
                    *common, device=x.device, alignment=cfg.alignment, extension=self._extension
                )
            rows = transport.capacity_rows
            # The fused gate/up kernel never materialises the [R, 2I] projection.
            fused = self.implementation == "cuda_fused"
            proj_rows = 0 if fused else rows
            sums_bytes = _one_pass_bytes(self._extension.lib, x.shape[0], cfg) if fused else None
            self._workspaces[key] = LayerWorkspace(
                transport,
                torch.empty((proj_rows, 2 * cfg.intermediate), device=x.device, dtype=x.dtype),
                torch.empty((rows, cfg.intermediate), device=x.device, dtype=x.dtype),
                torch.empty((rows, cfg.hidden), device=x.device, dtype=x.dtype),
                sums_bytes is not None,
                torch.empty(sums_bytes, device=x.device, dtype=torch.uint8) if sums_bytes else None,
            )
        return self._workspaces[key]

    def _experts_gathered(self, state, x):
        """experts_forward() with the gate/up GEMM reading x through
        ``transport.row_src`` (after dispatch_rows), not the packed rows."""
        transport = state.transport
        ext = self._extension
        ext.gateup_swiglu_gathered_out(x, transport.row_src, self.gate_up_weight, transport.offsets, state.activated)
        ext.grouped_gemm_out(state.activated, self.down_weight, transport.offsets, state.expert_output)
        return state.expert_output

    def experts_forward(self, state):
        transport = state.transport
        offsets = transport.offsets
        if self.implementation == "cuda_fused":
            ext = self._extension
            ext.gateup_swiglu_out(transport.packed, self.gate_up_weight, offsets, state.activated)
            ext.grouped_gemm_out(state.activated, self.down_weight, offsets, state.expert_output)
            return state.expert_output
        ends = offsets[1:]
        grouped_linear(
            transport.packed, self.gate_up_weight, ends, backend=self.expert_backend,
            output=state.projection, offsets=offsets,
        )
        state.activated.copy_(swiglu_reference(state.projection))
        grouped_linear(
            state.activated, self.down_weight, ends, backend=self.expert_backend,
            output=state.expert_output, offsets=offsets,
        )
        return state.expert_output

    def forward(self, x):
        if self.implementation == "cuda_fused" and x.ndim == 2:
            # No torch operator runs on this path, so it needs no inference mode.
            launches = self._launches.get((x.shape[0], x.device))
            if launches is not None and launches.accepts(x) and launches.still_valid(self):
                return launches(self, x)
        return self._validated_forward(x)

    @torch.inference_mode()
    def _validated_forward(self, x):
        if x.ndim != 2 or x.shape[1] != self.config.hidden or not x.is_contiguous():
            raise ValueError("expected contiguous x[T,hidden]")
        if x.dtype != self.gate_up_weight.dtype or x.device != self.gate_up_weight.device:
            raise ValueError("input dtype/device must match expert weights")
        if x.shape[0] == 0:
            return torch.empty_like(x)
        state = self.workspace(x)
        fused = self.implementation == "cuda_fused"
        # The fused router does the dispatch's counting pass when the shape allows.
        ranked = fused and state.transport.rank_tile > 0
        gathered = fused and (state.one_pass or _gathers(x, self.config.topk))
        ids32, ids64, weights = self._route(x, state.transport if ranked else None)
        transport = state.transport
        if gathered:
            # No packed copy: the gate/up GEMM reads x through the row table.
            if ranked:
                transport.dispatch_ranked_rows(ids32)
            else:
                transport.dispatch_rows(ids32)
            output = self._experts_gathered(state, x)
        else:
            if ranked:
                transport.dispatch_ranked(x, ids32)
            else:
                transport.dispatch(x, ids32, ids64)
            output = self.experts_forward(state)
        transport.combine(output, weights)
        if self.implementation == "cuda_fused":
            # Every operator above validated its tensors; later calls of this
            # shape reuse the checked arguments.
            self._launches[(x.shape[0], x.device)] = _FusedLaunches(self, x, state)
        return state.transport.output


def _can_gather(tokens, hidden):
    """Whether the gate/up GEMM can read its rows from bf16 x (hidden a multiple of 64, x below 2 GiB)."""
    return hidden % 64 == 0 and tokens * hidden * 2 < 2**31


def _gathers(x, topk):
    """Whether the fused forward skips the packed copy, the gate/up GEMM reading
    x through the dispatch's row table. It needs the ring kernels (hidden a
    multiple of 64) and x below 2 GiB, and pays off from top-3 on: the gathered
    GEMM is 1-2% slower than the packed one (H=4096, I=14336, E=8: 1510 against
    1489 us; H=1024, I=2048, E=16: +2.2%), which at top-2 costs about what the
    copy does, while with K rows per token the copy it saves grows with K
    (H=2048, I=1408, E=64, top-6: dispatch 39 -> 7 us, forward -3.8%). With
    that configuration's Zipf routing the gathered GEMM is itself faster than
    the packed one (560 against 638 us): it reads x's 33.6 MB where the packed
    kernel reads a 201 MB copy."""
    return topk >= 3 and _can_gather(*x.shape)


def _one_pass_bytes(lib, tokens, cfg):
    """Plane-sum bytes of the small-batch route that also writes the row table
    (``moe_route_rows``), or None where the shape has none. It replaces the router
    and the dispatch whatever top-k is: H=4096, E=8, top-2: 12.6 -> 6.6 us at one
    token, 13.8 -> 7.5 at 16; H=2048, E=64, top-6, 48 tokens: 33.6 -> 10.5 us."""
    need = lib.moe_route_rows_scratch_bytes(tokens, cfg.hidden, cfg.experts, cfg.topk)
    return need if need >= 0 and _can_gather(tokens, cfg.hidden) else None


class _FusedLaunches:
    """The C-ABI calls of one validated cuda_fused forward, for reuse.

    A forward through the validating operators (router_fused_out, dispatch,
    the two grouped GEMMs, combine) fixes every argument but x's address and
    the stream: workspace and weight pointers, sizes, the dtype code. Later
    forwards of the same token count on the same device make the same launches
    through one native call (``moe_block_forward``) on those arguments while every
    parameter tensor the kernels read is
    the object it was, at the same address, with the same dtype, shape and
    layout (an in-place update keeps all of these; the router split follows
    the weights' version as in ``MoEBlock.route``). Anything else sends the
    forward back through the validating path, which raises on a bad tensor.
    Host work per forward at 128 tokens of 512, where the kernels take about 22 us: 68 us
    through the operators, 31 with one foreign call per launch, 24 with one.
    """

    _PARAMETERS = ("router_weight", "gate_up_weight", "down_weight", "routing_bias", "_router_scratch")

    def __init__(self, block, x, state):
        cfg = block.config
        t = state.transport
        ids32, ids64, weights = block._route_buffers[(x.shape[0], x.device)]
        self.lib = block._extension.lib
        self.device_index = x.device.index if x.device.index is not None else torch.cuda.current_device()
        self.fingerprint = self._fingerprint(block)
        self.keep = (ids32, ids64, weights, t, state)  # the buffers below stay allocated
        self.output = t.output
        tokens, hidden = x.shape
        scratch = block._router_scratch
        # A ranked route (the router counts for the dispatch) whenever the shape
        # has one, and the row table instead of the packed copy whenever the
        # gate/up GEMM gathers, as in forward().
        self.ranked = t.rank_tile > 0
        self.gathered = state.one_pass or _gathers(x, cfg.topk)
        # The weights' row strides (contiguous, or gate/up rows padded); anything
        # else was refused by the validating forward that built these launches.
        gate_up_stride = weight_row_stride(block.gate_up_weight)
        down_stride = weight_row_stride(block.down_weight)
        if gate_up_stride is None or down_stride is None:
            raise RuntimeError("expert weights must be contiguous or row-padded")
        if x.dtype != torch.bfloat16:
            raise RuntimeError("cuda_fused launches are bf16")
        sums = state.plane_sums
        # The whole forward as one call (moe_block_forward): moe_block_args as its 64-bit
        # fields, in the header's order (``args`` names them; null pointers are 0). Every new
        # token count pays for this, and names for the fields, in a dictionary or a structure's
        # keywords, are allocations outside the interpreter's small ones: 10-45 us more.
        self.packed_args = array("q", (
            _lib.BLOCK_ARGS_BYTES, block.routing_bias.data_ptr(), ids32.data_ptr(), ids64.data_ptr(),
            weights.data_ptr(), scratch.data_ptr(), scratch.numel(),
            t.counts.data_ptr(), t.offsets.data_ptr(), t.slots.data_ptr(), t.inverse.data_ptr(), t.row_src.data_ptr(),
            t.packed.data_ptr(), t.scratch.data_ptr(), t.scratch.numel(),
            t.tile_ranks.data_ptr(), t.tile_counts.data_ptr(), t.tile_counts.numel() * 4, t.rank_tile,
            0 if sums is None else sums.data_ptr(), 0 if sums is None else sums.numel(),
            block.gate_up_weight.data_ptr(), gate_up_stride, block.down_weight.data_ptr(), down_stride,
            state.activated.data_ptr(), state.expert_output.data_ptr(), t.output.data_ptr(),
            tokens, hidden, cfg.intermediate, cfg.experts, cfg.topk, t.alignment, t.capacity_rows,
            bool(t.vectorized), self.gathered, state.one_pass))
        self.args_address = self.packed_args.buffer_info()[0]
        self.hidden = hidden

    @property
    def args(self):
        """The packed arguments by their names in the header (a view)."""
        return _lib.BlockArgs.from_buffer(self.packed_args)

    @classmethod
    def _fingerprint(cls, block):
        tensors = tuple(getattr(block, name) for name in cls._PARAMETERS)
        return tuple((name, v, v.data_ptr(), v.dtype, v.shape, v.stride()) for name, v in zip(cls._PARAMETERS, tensors))

    def still_valid(self, block):
        buffers, plain = block._buffers, block.__dict__
        for name, v, address, dtype, shape, stride in self.fingerprint:
            current = plain.get(name)
            if current is None:  # getattr's other places: buffers, and parameters set over one
                current = buffers.get(name)
                if current is None:
                    current = block._parameters.get(name)
            if current is not v or v.data_ptr() != address or v.shape != shape or v.stride() != stride \
                    or v.dtype != dtype:
                return False
        return True

    def accepts(self, x):
        """The caller's half of the checks (the key these launches are kept under has its
        token count and device; the weights' device and dtype are theirs)."""
        return x.dtype == torch.bfloat16 and x.shape[1] == self.hidden and x.is_contiguous()

    def __call__(self, block, x):
        router_weight, split_of = block._router_split_plan()
        status = self.lib.moe_block_forward(self.args_address, x.data_ptr(), router_weight,
                                            current_stream_handle(self.device_index))
        if status:
            self.lib.check(status, "forward")
        if router_weight is not None:  # else the split it holds is the one it has on record
            block._router_split_of = split_of
        return self.output

    def stage_calls(self, x):
        """Each stage of __call__ as a zero-argument callable on the current
        stream (the router with the split it holds), for per-stage timing: router
        and dispatch, or for a small batch the one-pass ``route`` in their place."""
        lib, a, x_ptr = self.lib, self.args, x.data_ptr()

        def bind(name, *args):
            def run():
                lib.check(getattr(lib, name)(*args, current_stream_handle(self.device_index)), name)
            return run

        index = (a.ids32, a.counts, a.offsets, a.slots)
        layout = (a.experts, a.topk, a.alignment, a.packed_rows)
        stages = {}
        if a.one_pass:
            stages["route"] = bind("moe_route_rows", x_ptr, None, a.bias, a.ids32, a.ids64, a.weights, a.router_scratch,
                                   a.router_scratch_bytes, *index[1:], a.inverse, a.row_src, a.sums, a.sums_bytes,
                                   a.tokens, a.hidden, *layout)
        else:
            table = (a.dispatch_scratch, a.dispatch_scratch_bytes)
            router = (x_ptr, None, a.bias, a.ids32, a.ids64, a.weights, None, a.router_scratch, a.router_scratch_bytes,
                      a.tokens, a.hidden, a.experts, a.topk)
            name = ""
            if self.ranked:
                name, table = "_ranked", (a.ranks, a.tile_counts, a.tile_counts_bytes, a.tile_tokens)
                router += table[:3]
            stages["router"] = bind("moe_router_fused" + name, *router)
            if self.gathered:
                stages["dispatch"] = bind(f"moe_dispatch{name}_rows", *index, a.inverse, a.row_src, *table, a.tokens,
                                          *layout)
            else:
                stages["dispatch"] = bind("moe_dispatch" + name, x_ptr, _lib.DTYPE_BF16, *index, a.packed, a.inverse,
                                          *table, a.tokens, a.hidden, *layout, a.vectorized)
        gemm = (a.activated, a.offsets, a.packed_rows, a.hidden, a.intermediate, a.experts)
        if self.gathered:
            stages["gateup_swiglu"] = bind("moe_grouped_gateup_swiglu_gathered_strided", x_ptr, a.row_src, a.tokens,
                                           a.gate_up, a.gate_up_row_stride, *gemm)
        else:
            stages["gateup_swiglu"] = bind("moe_grouped_gateup_swiglu_strided", a.packed, a.gate_up,
                                           a.gate_up_row_stride, *gemm)
        stages["down"] = bind("moe_grouped_gemm_strided", a.activated, a.down, a.down_row_stride, a.expert_output,
                              *gemm[1:])
        stages["combine"] = bind("moe_combine", a.expert_output, _lib.DTYPE_BF16, a.inverse, a.weights, a.output,
                                 a.tokens, a.hidden, a.topk, a.packed_rows)
        return stages


@torch.inference_mode()
def token_major_oracle(block, x):
    """Routed tokens evaluated token by token, independent of the packed layout.

    The check the reference's benchmark harness runs on every forward
    (``layer.py:200-214``), with the same policy: fp32 router logits plus bias,
    top-k, softmax of the selected logits, each expert's gate/up projection,
    SwiGLU and down projection in the block's dtype (torch's own GEMMs), and the
    weighted sum in fp32 cast once. Here each expert evaluates only the
    (token, slot) pairs routed to it, gathered straight from the top-k ids, and
    adds them back by token index; no dispatch buffer, offset or permutation of
    the engine is used. Excluded from timings.
    """
    cfg = block.config
    logits = torch.nn.functional.linear(x.float(), block.router_weight) + block.routing_bias
    top = torch.topk(logits, cfg.topk, dim=-1)
    weights = torch.softmax(top.values, dim=-1)
    total = torch.zeros(x.shape, device=x.device, dtype=torch.float32)
    for expert in range(cfg.experts):
        tokens, slots = torch.nonzero(top.indices == expert, as_tuple=True)
        if tokens.numel() == 0:
            continue
        rows = x.index_select(0, tokens)
        hidden_state = swiglu_reference(torch.nn.functional.linear(rows, block.gate_up_weight[expert]))
        y = torch.nn.functional.linear(hidden_state, block.down_weight[expert]).float()
        total.index_add_(0, tokens, y * weights[tokens, slots].unsqueeze(1))
    return total.to(x.dtype)
