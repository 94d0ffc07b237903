"""Autograd wiring of the expert region and registration of the reference's operator.

Two ways in:

* ``expert_region(...)``: the whole region (gate -> top-k -> sort -> grouped SwiGLU with the permute
  fused into the operand load -> unpermute+combine) as ONE autograd node with a hand-written
  backward.  This is what ``piper_amd.moe.AnnotatedMoE`` runs.
* the piecewise operators the reference model code calls one by one
  (examples/models/qwen3.py:237-283): ``router``, ``reorder``, ``permute``, ``bmm_experts``,
  ``combine``.  ``bmm_experts`` is also registered as ``torch.ops.piper_artifact.bmm_experts`` with
  the reference's schema (examples/models/qwen3_bmm_experts_patch.py:63-72), so reference model
  code that looks the op up by name gets the HIP implementation.
"""
from __future__ import annotations

import torch
from torch.overrides import has_torch_function_variadic

from . import ops
from ._lib import host

_ROUTE_TOPK = ops.route_topk
_is_tracing = torch._C._is_tracing          # torch.jit.is_tracing() without its check for scripted code


def _replaced_route():
    """ops.route_topk where somebody has put another function in its place (to record or force the
    routing); None otherwise, and the host path launches the kernel itself."""
    return None if ops.route_topk is _ROUTE_TOPK else ops.route_topk


# --------------------------------------------------------------------------- piecewise operators


def _sorted_tables(top_idx: torch.Tensor, num_experts: int):
    """(counts, starts, perm, inv_perm) of the counting sort of `top_idx`, computed once per routing
    result: the tables ride on the index tensor, and the inverse permutation rides on `perm`, so the
    piecewise operators that follow (reorder, permute backward, combine) launch no second sort."""
    # valid for this tensor object, these contents (autograd's version counter moves with every
    # in-place write) and this expert count; a view or a clone is another object and is sorted again
    key = (top_idx._version, int(num_experts))
    cached = getattr(top_idx, "_pk_sorted", None)
    if cached is None or cached[0] != key:
        tables = host().sort_by_expert(top_idx, int(num_experts))
        tables[2]._pk_inverse = (tables[2]._version, tables[3])
        cached = (key, tables)
        top_idx._pk_sorted = cached
    return cached[1]


def _inverse_of(perm: torch.Tensor) -> torch.Tensor:
    """inv_perm for a permutation produced by `reorder` (cached there); any other permutation is
    inverted once and remembered on the tensor."""
    cached = getattr(perm, "_pk_inverse", None)
    if cached is None or cached[0] != perm._version:
        inv = torch.empty_like(perm)
        inv[perm.long()] = torch.arange(perm.numel(), dtype=perm.dtype, device=perm.device)
        cached = (perm._version, inv)
        perm._pk_inverse = cached
    return cached[1]


def _router(x, w_gate, gate_bias, top_k, route_norm, route_scale):
    return host().router(x, w_gate, gate_bias, top_k, route_norm, route_scale, _replaced_route())


def router(x, w_gate, gate_bias=None, *, top_k: int, route_norm: bool, route_scale: float = 1.0):
    """(top_scores [T,K] f32, selected_experts_indices [T,K] i32, num_tokens_per_expert [E] i32).
    The call `self.router(x, self.expert_bias)` of qwen3.py:237-241.  The histogram is the one the
    counting sort produces (no host sync, no second pass over the indices)."""
    call = torch.ops.piper_amd.router if _is_tracing() else _router
    top_scores, top_idx = call(x, w_gate, gate_bias, int(top_k), bool(route_norm), float(route_scale))
    counts = _sorted_tables(top_idx, w_gate.shape[0])[0]
    return top_scores, top_idx, counts


def reorder(top_scores: torch.Tensor, top_idx: torch.Tensor, num_experts: int):
    """The reorderer of qwen3.py:243-247.  Returns (top_scores_experts_sorted [A],
    token_indices_experts_sorted [A] i32, num_tokens_per_expert [E] i32)."""
    counts, _starts, perm, _inv = _sorted_tables(top_idx, num_experts)
    scores_sorted = top_scores.reshape(-1).index_select(0, perm)
    return scores_sorted, perm, counts


def _permute(x, perm, top_k):
    return host().permute(x, perm, _inverse_of(perm), top_k)


def permute(x: torch.Tensor, token_indices_experts_sorted: torch.Tensor, top_k: int) -> torch.Tensor:
    """routed_input = x[token_indices_experts_sorted // top_k]  (qwen3.py:250)."""
    call = torch.ops.piper_amd.permute if _is_tracing() else _permute
    return call(x, token_indices_experts_sorted, int(top_k))


def _traced_without_data(*tensors) -> bool:
    """True under fake-tensor propagation (Dynamo, make_fx) or on the meta device: the call is only
    asked for the output's shape, dtype and whether it takes part in autograd."""
    from torch._subclasses.fake_tensor import FakeTensor
    return any(t.is_meta or isinstance(t, FakeTensor) for t in tensors)


def _bmm_experts_shape_only(w1, w2, w3, x):
    out = torch.empty_like(x)
    if torch.is_grad_enabled() and any(t.requires_grad for t in (w1, w2, w3, x)):
        out.requires_grad_(True)
    return out


def _bmm_experts_autograd(w1, w2, w3, x, num_tokens_per_expert):
    # The reference binds one traceable Python function to every dispatch key, the Autograd key
    # included (qwen3_bmm_experts_patch.py:67-75), so Dynamo's fake-tensor propagation runs this
    # kernel too: it must not touch device pointers then.
    if _traced_without_data(w1, w2, w3, x, num_tokens_per_expert):
        return _bmm_experts_shape_only(w1, w2, w3, x)
    return host().bmm_experts(w1, w2, w3, x, num_tokens_per_expert, False)


def _bmm_experts_forward_only(w1, w2, w3, x, num_tokens_per_expert):
    if _traced_without_data(w1, w2, w3, x, num_tokens_per_expert):
        return torch.empty_like(x)
    with torch.no_grad():
        return host().bmm_experts(w1, w2, w3, x, num_tokens_per_expert, False)


def _bmm_experts_meta(w1, w2, w3, x, num_tokens_per_expert):
    return torch.empty_like(x)


_LIBS = []


def register_reference_op() -> bool:
    """Define ``piper_artifact::bmm_experts`` (same schema as qwen3_bmm_experts_patch.py:63-65) on
    the CUDA(=HIP)/Autograd/Meta keys.  If the op already exists (the reference patch was imported
    first) only the CUDA and AutogradCUDA kernels are overridden.  Returns True when this call
    registered something."""
    if _LIBS:
        return False
    exists = hasattr(torch.ops, "piper_artifact") and hasattr(torch.ops.piper_artifact, "bmm_experts")
    if not exists:
        def_lib = torch.library.Library("piper_artifact", "DEF")
        def_lib.define(
            "bmm_experts(Tensor w1, Tensor w2, Tensor w3, Tensor x, Tensor num_tokens_per_expert) -> Tensor"
        )
        _LIBS.append(def_lib)
    impl = torch.library.Library("piper_artifact", "IMPL")
    impl.impl("bmm_experts", _bmm_experts_forward_only, "CUDA")
    impl.impl("bmm_experts", _bmm_experts_autograd, "AutogradCUDA")
    if not exists:
        impl.impl("bmm_experts", _bmm_experts_meta, "Meta")
    _LIBS.append(impl)
    return True


def _direct(*tensors) -> bool:
    """Whether a call may go to the kernels without the operator in between (the native side looks at the
    tensors themselves and at dispatch modes): nothing is being compiled, and no tensor subclass, FX proxy
    or torch-function mode waits for the operator's name."""
    return not torch.compiler.is_compiling() and not has_torch_function_variadic(*tensors)


def bmm_experts(w1, w2, w3, x, num_tokens_per_expert):
    """Same call as the reference's ``bmm_experts`` (qwen3_bmm_experts_patch.py:78-87)."""
    register_reference_op()
    if _direct(w1, w2, w3, x, num_tokens_per_expert):     # ordinary tensors: the operator's kernel without the dispatcher
        out = host().bmm_experts(w1, w2, w3, x, num_tokens_per_expert, True) if x.is_cuda else None
        if out is not None:
            return out
    return torch.ops.piper_artifact.bmm_experts(w1, w2, w3, x, num_tokens_per_expert)


def _combine(y, perm, top_scores):
    return host().combine(y, perm, _inverse_of(perm), top_scores)


def combine(gathered_output, token_indices_experts_sorted, top_scores):
    """Unpermute scatter + fp32 weighted sum over k (qwen3.py:265-283), fused."""
    call = torch.ops.piper_amd.combine if _is_tracing() else _combine
    return call(gathered_output, token_indices_experts_sorted, top_scores)


# --------------------------------------------------------------------------- split backward
class WeightGradQueue:
    """Weight-gradient work postponed by a backward-input pass (Piper's BWD_I / BWD_W split,
    src/executors.py:353-476).  ``run()`` launches the postponed kernels and accumulates their
    results into ``param.grad`` as the reference's weight pass does (src/executors.py:333-343)."""

    def __init__(self):
        self._work = []

    def push(self, fn) -> None:
        self._work.append(fn)

    def __len__(self) -> int:
        return len(self._work)

    def run(self) -> None:
        work, self._work = self._work, []
        for fn in work:
            fn()


_WGRAD_QUEUE: WeightGradQueue | None = None


class defer_weight_grads:
    """Context manager: backward passes run inside it compute input gradients only; the weight
    gradients of leaf parameters are queued on the returned WeightGradQueue."""

    def __enter__(self) -> WeightGradQueue:
        global _WGRAD_QUEUE
        self._prev = _WGRAD_QUEUE
        _WGRAD_QUEUE = WeightGradQueue()
        host().set_queue(_WGRAD_QUEUE)
        return _WGRAD_QUEUE

    def __exit__(self, *exc) -> None:
        global _WGRAD_QUEUE
        _WGRAD_QUEUE = self._prev
        host().set_queue(self._prev)


class accumulate_weight_grads:
    """Context manager for backward passes that accumulate into ``.grad`` (``torch.autograd.backward``
    / ``Tensor.backward``, the way the reference's executor runs a backward task,
    src/executors.py:257-296): inside it the fused expert region adds the gradients of leaf
    parameters whose ``.grad`` already exists to that buffer in the epilogue of the weight-gradient
    kernels and hands autograd no gradient for them, instead of writing fresh tensors that
    AccumulateGrad then adds in a separate pass over 3 x E x I x H elements.  Gradient accumulation
    over microbatches as in src/executors.py:333-343.  Not for ``torch.autograd.grad``, which must
    return the gradients and leave ``.grad`` alone."""

    def __enter__(self):
        self._prev = host().set_accumulate(True)
        return self

    def __exit__(self, *exc) -> None:
        host().set_accumulate(self._prev)


# --------------------------------------------------------------------------- fused region
# Measured on MI355X: running the weight gradient next to the input gradient gains ~1.5 % (both
# kernels are throughput-bound), so it is opt-in; per-kernel timings are only meaningful with it off.
def set_overlap_wgrad(on: bool) -> None:
    """Run the weight-gradient kernel on a second stream, concurrently with the input gradient."""
    host().set_overlap(bool(on))


# The fused region and the RMSNorm are torch.library operators too (namespace piper_amd), for the same
# reason the reference wraps its expert segment in one (qwen3_bmm_experts_patch.py:56-75): the model
# is captured by Dynamo with fullgraph=True (src/compile.py:273), which cannot look inside a
# function that launches kernels through a C ABI.  As graph nodes they are opaque calls whose
# output shape comes from the fake-tensor branch of their kernels.
_REGION_LIBS = []


def _expert_region_autograd(x, w_gate, gate_bias, w1, w2, w3, top_k, route_norm, route_scale, residual):
    ts = [t for t in (x, w_gate, gate_bias, w1, w2, w3, residual) if t is not None]
    if _traced_without_data(*ts):
        out = torch.empty_like(x)
        if torch.is_grad_enabled() and any(t.requires_grad for t in ts):
            out.requires_grad_(True)
        return out
    return host().expert_region(x, w_gate, gate_bias, w1, w2, w3, top_k, route_norm, route_scale, residual, None, 0.0,
                                _replaced_route(), False)


def _expert_region_forward_only(x, w_gate, gate_bias, w1, w2, w3, top_k, route_norm, route_scale, residual):
    with torch.no_grad():
        return _expert_region_autograd(x, w_gate, gate_bias, w1, w2, w3, top_k, route_norm, route_scale, residual)


def _rmsnorm_autograd(x, weight, eps):
    if _traced_without_data(x, weight):
        out = torch.empty_like(x)
        if torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad):
            out.requires_grad_(True)
        return out
    return host().rmsnorm(x, weight, eps, False)


def _rmsnorm_forward_only(x, weight, eps):
    with torch.no_grad():
        return _rmsnorm_autograd(x, weight, eps)


def register_region_ops() -> bool:
    """Define ``piper_amd::expert_region`` and ``piper_amd::rmsnorm`` (done when this module is
    imported: a registration cannot happen inside a function Dynamo is tracing).  Returns True when
    this call registered them."""
    if _REGION_LIBS:
        return False
    lib = torch.library.Library("piper_amd", "DEF")
    lib.define("expert_region(Tensor x, Tensor w_gate, Tensor? gate_bias, Tensor w1, Tensor w2, Tensor w3, "
               "int top_k, bool route_norm, float route_scale, Tensor? residual) -> Tensor")
    lib.define("rmsnorm(Tensor x, Tensor weight, float eps) -> Tensor")
    for name, fwd, auto in (("expert_region", _expert_region_forward_only, _expert_region_autograd),
                            ("rmsnorm", _rmsnorm_forward_only, _rmsnorm_autograd)):
        lib.impl(name, fwd, "CUDA")
        lib.impl(name, auto, "AutogradCUDA")
        lib.impl(name, fwd, "Meta")
        # CPU tensors reach the kernels' own check and are refused there; fake CPU tensors get a shape
        lib.impl(name, fwd, "CPU")
        lib.impl(name, auto, "AutogradCPU")
    # what torch.jit.trace records of the piecewise operators that otherwise go to the kernels directly
    lib.define("router(Tensor x, Tensor w_gate, Tensor? gate_bias, int top_k, bool route_norm, float route_scale) -> (Tensor, Tensor)")
    lib.define("permute(Tensor x, Tensor perm, int top_k) -> Tensor")
    lib.define("combine(Tensor y, Tensor perm, Tensor top_scores) -> Tensor")
    for name, fn in (("router", _router), ("permute", _permute), ("combine", _combine)):
        for key in ("CUDA", "AutogradCUDA", "CPU", "AutogradCPU"):
            lib.impl(name, fn, key)
    _REGION_LIBS.append(lib)
    return True


def expert_region(x, w_gate, gate_bias, w1, w2, w3, *, top_k: int, route_norm: bool, route_scale: float = 1.0,
                  residual=None):
    """The whole MoE expert region of AnnotatedMoE.forward (qwen3.py:233-289) on x [T,H].
    `residual` [T,H] is added to the result in the combine kernel."""
    if _direct(x, w_gate, gate_bias, w1, w2, w3, residual):     # ordinary tensors: the operator's kernel without the dispatcher
        out = host().expert_region(x, w_gate, gate_bias, w1, w2, w3, int(top_k), bool(route_norm), float(route_scale),
                                   residual, None, 0.0, _replaced_route(), True)
        if out is not None:
            return out
    return torch.ops.piper_amd.expert_region(x, w_gate, gate_bias, w1, w2, w3, int(top_k), bool(route_norm),
                                             float(route_scale), residual)


def rmsnorm(x, weight, eps: float = 1e-6):
    """RMSNorm over the last dimension (the block's ffn_norm, qwen3.py:313-314)."""
    shape = x.shape
    if _direct(x, weight):
        out = host().rmsnorm(x.reshape(-1, shape[-1]), weight, float(eps), True)
        if out is not None:
            return out.reshape(shape)
    return torch.ops.piper_amd.rmsnorm(x.reshape(-1, shape[-1]), weight, float(eps)).reshape(shape)


def moe_block(h, norm_weight, w_gate, gate_bias, w1, w2, w3, *, top_k: int, route_norm: bool,
              route_scale: float = 1.0, norm_eps: float = 1e-6):
    """h + moe(ffn_norm(h)) on h [T,H] (qwen3.py:313-314): RMSNorm kernel, expert region, residual
    added in the combine kernel.  One autograd node: its backward adds the residual branch's gradient
    inside the norm's backward kernel."""
    if _direct(h, norm_weight, w_gate, gate_bias, w1, w2, w3):
        out = host().expert_region(h, w_gate, gate_bias, w1, w2, w3, int(top_k), bool(route_norm), float(route_scale), None,
                                   norm_weight, float(norm_eps), _replaced_route(), True)
        if out is not None:
            return out
    return expert_region(rmsnorm(h, norm_weight, norm_eps), w_gate, gate_bias, w1, w2, w3, top_k=top_k,
                         route_norm=route_norm, route_scale=route_scale, residual=h)


register_region_ops()
