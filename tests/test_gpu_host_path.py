"""The native host path of the operators where autograd, the split backward and the bucket path meet
tensors and callers other than the ordinary ones: saved-tensor hooks, forward-mode tangents, strided
gradients, what a postponed weight pass keeps alive, inputs past one launch's grid, and whoever looks for
the operators by name (tracers, torch-function modes and subclasses, the profiler)."""
import gc
import warnings

import pytest
import torch
import torch.autograd.forward_ad as fwAD
from torch.overrides import TorchFunctionMode
from torch.utils.checkpoint import checkpoint

from conftest import BF16_TOL, rel_err
from piper_amd import functional as F_
from piper_amd import ops
from piper_amd._lib import host, on_stream, wait_stream
from piper_amd.moe import AnnotatedMoE, MoEArgs, MoEFeedForwardBlock, RMSNorm

pytestmark = pytest.mark.gpu

T, H, E, K, I = 96, 256, 8, 2, 128


def _params(dev, dtype=torch.bfloat16, seed=0, hidden=H, experts=E, inter=I):
    g = torch.Generator().manual_seed(seed)

    def rnd(*shape, scale, dt=dtype):
        return (torch.randn(*shape, generator=g) * scale).to(dt).to(dev).requires_grad_(True)

    return dict(norm=(1 + 0.1 * torch.randn(hidden, generator=g)).to(dtype).to(dev).requires_grad_(True),
                w_gate=rnd(experts, hidden, scale=0.05, dt=torch.float32), bias=rnd(experts, scale=0.1, dt=torch.float32),
                w1=rnd(experts, inter, hidden, scale=0.05), w2=rnd(experts, hidden, inter, scale=0.05),
                w3=rnd(experts, inter, hidden, scale=0.05))


def _activations(dev, tokens, dtype=torch.bfloat16, seed=1, hidden=H):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(tokens, hidden, generator=g).to(dtype).to(dev) for _ in range(2))


def _region(x, p):
    return F_.expert_region(x, p["w_gate"], p["bias"], p["w1"], p["w2"], p["w3"], top_k=K, route_norm=True)


def _block(x, p):
    return F_.moe_block(x, p["norm"], p["w_gate"], p["bias"], p["w1"], p["w2"], p["w3"], top_k=K, route_norm=True)


def _experts(x, p):
    n = x.shape[0]
    counts = torch.full((p["w1"].shape[0],), n // p["w1"].shape[0], dtype=torch.int32, device=x.device)
    return F_.bmm_experts(p["w1"], p["w2"], p["w3"], x, counts)


FLOWS = {"region": (_region, ("w_gate", "bias", "w1", "w2", "w3")),
         "block": (_block, ("norm", "w_gate", "bias", "w1", "w2", "w3")),
         "experts": (_experts, ("w1", "w2", "w3"))}


def _under(hooks, fn, x):
    if hooks == "none":
        return fn(x)
    if hooks == "checkpoint":
        return checkpoint(fn, x, use_reentrant=False)
    ctx = torch.autograd.graph.save_on_cpu() if hooks == "save_on_cpu" else \
        torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t)
    with ctx:
        return fn(x)


@pytest.mark.parametrize("hooks", ["identity", "save_on_cpu", "checkpoint"])
@pytest.mark.parametrize("flow", FLOWS)
def test_postponed_weight_gradients_reach_the_parameters_under_saved_tensor_hooks(dev, flow, hooks):
    """A hook's unpacked tensor is a copy: the gradients belong to the parameters themselves, and are
    those of the same pass without hooks, bit for bit."""
    print(f"[case] postponed weight gradients, {flow}, {hooks}", flush=True)
    fn, names = FLOWS[flow]
    x0, d = _activations(dev, T)

    def run(how):
        p = _params(dev)
        x = x0.clone().requires_grad_(True)
        out = _under(how, lambda t: fn(t, p), x)
        with F_.defer_weight_grads() as queue:
            out.backward(d)
        queue.run()
        return {"x": x.grad, **{n: p[n].grad for n in names}}

    want, got = run("none"), run(hooks)
    for n in want:
        assert got[n] is not None, f"{n} has no gradient"
        assert torch.equal(got[n], want[n]), n


def test_gate_weight_that_is_a_transposed_view(dev):
    """The postponed gate gradient of a non-contiguous gate weight has the weight's elements in their places."""
    x, d = _activations(dev, T)

    def run(postponed):
        p = _params(dev)
        p["w_gate"] = torch.nn.Parameter(p["w_gate"].detach().t().contiguous().t())
        assert not p["w_gate"].is_contiguous()
        out = _region(x, p)
        if postponed:
            with F_.defer_weight_grads() as queue:
                out.backward(d)
            queue.run()
        else:
            out.backward(d)
        return p["w_gate"].grad

    assert torch.equal(run(True), run(False))


def _strided(values):
    """`values` in a tensor whose last two dimensions (or whose only one) are not laid out contiguously."""
    if values.dim() == 1:
        t = torch.zeros(2 * values.numel(), dtype=values.dtype, device=values.device)[::2]
    else:
        t = torch.zeros(values.transpose(-1, -2).shape, dtype=values.dtype, device=values.device).transpose(-1, -2)
    t.copy_(values)
    assert not t.is_contiguous()
    return t


@pytest.mark.parametrize("mode", ["postponed", "accumulate"])
@pytest.mark.parametrize("flow,strided", [("region", ("w1",)), ("region", ("w1", "w2", "w3")), ("region", ("w_gate",)), ("region", ("bias",)),
                                          ("region", ("w_gate", "bias", "w2")), ("experts", ("w1",)), ("experts", ("w1", "w2", "w3"))],
                         ids=lambda v: v if isinstance(v, str) else "-".join(v))
def test_gradients_are_added_to_strided_grad_buffers(dev, flow, strided, mode):
    """A `.grad` that is not contiguous receives the sum autograd would leave in it: the kernels, which
    write contiguous tensors, are not pointed at it."""
    fn, names = FLOWS[flow]
    print(f"[case] strided .grad, {flow}, {mode}, {strided}", flush=True)
    x, d = _activations(dev, T)
    p0 = _params(dev)
    fn(x, p0).backward(d)
    fresh = {n: p0[n].grad for n in names}

    p = _params(dev)
    before = {n: torch.randn_like(p[n]) for n in names}
    for n in names:
        p[n].grad = _strided(before[n]) if n in strided else before[n].clone()
    held = {n: p[n].grad for n in strided}
    out = fn(x, p)
    if mode == "postponed":
        with F_.defer_weight_grads() as queue:
            out.backward(d)
        queue.run()
    else:
        with F_.accumulate_weight_grads():
            out.backward(d)
    for n in names:
        want = before[n].float() + fresh[n].float()
        # one rounding to the buffer's type, of the sum or of the gradient and then the sum
        tol = 2.0 ** -7 if p[n].dtype == torch.bfloat16 else 1e-6
        assert rel_err(p[n].grad, want) <= tol, (n, rel_err(p[n].grad, want))
    for n in strided:
        assert rel_err(held[n], p[n].grad) == 0.0 and held[n].stride() == _strided(before[n]).stride(), n


def test_expanded_grad_is_refused(dev):
    """Several elements of an expanded `.grad` share one place in memory: an error, and nothing written past it."""
    x, d = _activations(dev, T)
    p = _params(dev)
    for n in ("w1", "w2", "w3"):
        p[n].grad = torch.zeros(1, 1, 1, dtype=p[n].dtype, device=dev).expand_as(p[n])
    out = _region(x, p)
    with F_.defer_weight_grads() as queue:
        out.backward(d)
    with pytest.raises(RuntimeError):
        queue.run()


def test_forward_mode_tangents_are_refused(dev):
    """None of the operators has a forward-mode rule: a dual tensor raises, also where no gradient is asked
    for, and its tangent is not dropped."""
    p = {n: t.detach() for n, t in _params(dev).items()}
    x, v = _activations(dev, T)
    calls = {
        "region": lambda t: _region(t, p),
        "region operator": lambda t: torch.ops.piper_amd.expert_region(t, p["w_gate"], p["bias"], p["w1"], p["w2"], p["w3"], K, True, 1.0, None),
        "block": lambda t: _block(t, p),
        "rmsnorm": lambda t: F_.rmsnorm(t, p["norm"]),
        "rmsnorm operator": lambda t: torch.ops.piper_amd.rmsnorm(t, p["norm"], 1e-6),
        "experts": lambda t: _experts(t, p),
        "router": lambda t: F_.router(t, p["w_gate"], p["bias"], top_k=K, route_norm=True),
        "permute": lambda t: F_.permute(t, torch.arange(T, dtype=torch.int32, device=dev), 1),
        "combine": lambda t: F_.combine(t, torch.arange(T, dtype=torch.int32, device=dev), torch.ones(T, 1, device=dev)),
    }
    for name, call in calls.items():
        for grad_mode in (True, False):
            print(f"[case] forward mode, {name}, grad mode {grad_mode}", flush=True)
            call(x)
            with fwAD.dual_level(), torch.set_grad_enabled(grad_mode):
                with pytest.raises(NotImplementedError):
                    call(fwAD.make_dual(x, v))
    # a tangent of a weight counts as much as one of the input
    with fwAD.dual_level(), pytest.raises(NotImplementedError):
        _region(x, dict(p, w2=fwAD.make_dual(p["w2"], torch.ones_like(p["w2"]))))


def test_functorch_transforms(dev):
    """A transform's wrapper tensors have no memory: the kernels refuse them.  (vmap over the operators that
    go through the dispatcher runs them slice by slice.)"""
    p = {n: t.detach() for n, t in _params(dev).items()}
    x, _ = _activations(dev, T)
    perm, one = torch.arange(T, dtype=torch.int32, device=dev), torch.ones(T, 1, device=dev)
    for name, call in {"region": lambda t: _region(t, p), "rmsnorm": lambda t: F_.rmsnorm(t, p["norm"]), "experts": lambda t: _experts(t, p),
                       "permute": lambda t: F_.permute(t, perm, 1), "combine": lambda t: F_.combine(t, perm, one)}.items():
        print(f"[case] functorch grad, {name}", flush=True)
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda t: call(t).float().sum())(x)
    xs = torch.stack([x, 2 * x])
    assert torch.equal(torch.func.vmap(lambda t: F_.rmsnorm(t, p["norm"]))(xs), torch.stack([F_.rmsnorm(t, p["norm"]) for t in xs]))
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: F_.permute(t, perm, 1))(xs)


# (flow, tokens, hidden, experts, top_k, inter, row layout of the copies the weight gradient reads)
HELD = [("region", 4096, 512, 16, 2, 256), ("block", 4096, 512, 16, 2, 256), ("experts", 8192, 512, 16, 1, 256),
        ("region", 4096, 2048, 128, 8, 768), ("block", 4096, 2048, 128, 8, 768)]


@pytest.mark.parametrize("flow,tokens,hidden,experts,top_k,inter", HELD, ids=lambda v: str(v))
def test_a_postponed_weight_pass_keeps_only_what_it_reads(dev, flow, tokens, hidden, experts, top_k, inter):
    """Between the input pass and the weight pass of a microbatch: d_g, d_u and (score *) h, the operands' row
    tables, the gate's d_logits and, with a norm in front, its output; no routed-row gradients and no
    pre-activations."""
    print(f"[case] memory between the passes, {flow} {tokens} x {hidden}", flush=True)
    p = _params(dev, hidden=hidden, experts=experts, inter=inter)
    x, d = _activations(dev, tokens, hidden=hidden)
    x.requires_grad_(True)
    kw = dict(top_k=top_k, route_norm=True)

    def forward():
        if flow == "experts":
            return _experts(x, p)
        if flow == "block":
            return F_.moe_block(x, p["norm"], p["w_gate"], p["bias"], p["w1"], p["w2"], p["w3"], **kw)
        return F_.expert_region(x, p["w_gate"], p["bias"], p["w1"], p["w2"], p["w3"], **kw)

    gc.collect()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = forward()
    with F_.defer_weight_grads() as queue:
        out.backward(d)
    del out
    x.grad = p["norm"].grad = None
    held = torch.cuda.memory_allocated() - before
    rows = tokens * top_k
    padded = max(rows, ops.transposed_ld(rows, hidden, inter, experts, torch.bfloat16)) if flow != "experts" else rows
    reads = 3 * padded * inter * 2
    if flow != "experts":
        reads += rows * 4 + (2 * experts + 1) * 4 + tokens * experts * 4 + (tokens * hidden * 2 if flow == "block" else 0)
    # the caching allocator rounds a block up by as much as 1 MiB
    assert held <= reads + 4 * 2 ** 20, (held, reads)
    queue.run()
    assert p["w1"].grad is not None


def test_backward_of_more_tokens_than_one_launch_has_row_blocks(dev):
    """The gather of the input gradient has 32-token row blocks on a grid dimension of at most 65,535."""
    tokens, hidden, experts, top_k, inter = 65535 * 32 + 77, 32, 4, 2, 32
    print(f"[case] {tokens} tokens", flush=True)
    p = _params(dev, hidden=hidden, experts=experts, inter=inter)
    g = torch.Generator(device=dev).manual_seed(2)
    x0, d = (torch.randn(tokens, hidden, generator=g, device=dev).bfloat16() for _ in range(2))

    def run(rows):
        x = x0[rows].clone().requires_grad_(True)
        out = F_.expert_region(x, p["w_gate"], p["bias"], p["w1"], p["w2"], p["w3"], top_k=top_k, route_norm=True)
        (dx,) = torch.autograd.grad(out, x, d[rows])
        return dx

    whole = run(slice(None))
    # a token's input gradient does not depend on the tokens beside it
    for rows in (slice(0, 4096), slice(65535 * 32 - 64, 65535 * 32), slice(65535 * 32, tokens), slice(65535 * 32 - 33, 65535 * 32 + 33)):
        assert rel_err(whole[rows], run(rows)) <= BF16_TOL, rows


def test_gradients_survive_a_pack_that_is_refused(dev):
    """Nothing is packed and no gradient is dropped where one of them cannot be packed."""
    flat = torch.zeros(64, device=dev)
    good = torch.nn.Parameter(torch.zeros(16, device=dev))
    bad = torch.nn.Parameter(torch.zeros(16, device=dev, dtype=torch.float64))
    for second, specs in ((bad, [(good, 0, 16, (16,)), (bad, 16, 16, (16,))]), (good, [(good, 60, 16, (16,))])):
        good.grad, bad.grad = torch.ones_like(good), torch.ones_like(bad)
        with pytest.raises((TypeError, ValueError)):
            host().pack_param_grads(specs, flat, None)
        assert all(s[0].grad is not None for s in specs)
        assert float(flat.abs().max()) == 0.0


def test_streams_wait_for_each_other(dev):
    """Events between side streams and the default stream, whose handle is null."""
    a, b, main = torch.cuda.Stream(dev), torch.cuda.Stream(dev), torch.cuda.current_stream(dev)
    src = torch.arange(1 << 24, device=dev, dtype=torch.float32)
    wait_stream(a, main)
    with on_stream(a):
        mid = src + 1
    wait_stream(b, a)
    with on_stream(b):
        out = mid * 2
    wait_stream(main, b)
    assert torch.equal(out, (src + 1) * 2)
    torch.cuda.synchronize()


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_operators_and_streams_of_a_device_that_is_not_current(dev):
    one = torch.device("cuda:1")
    with torch.cuda.device(0):
        a, b = torch.cuda.Stream(one), torch.cuda.default_stream(one)
        wait_stream(a, b)
        with on_stream(a):
            idx = torch.randint(0, 16, (9000, 1), device=one, dtype=torch.int32)
        wait_stream(b, a)
        perm = ops.sort_by_expert(idx, 16)[2]
        assert torch.equal(perm.long(), torch.argsort(idx.reshape(-1).long(), stable=True))
        p = torch.nn.Parameter(torch.zeros(16, device=one))
        p.grad = torch.ones_like(p)
        flat = torch.zeros(16, device=one)
        host().pack_param_grads([(p, 0, 16, (16,))], flat, None)
        assert p.grad is None and torch.equal(flat, torch.ones_like(flat))
        assert torch.cuda.current_device() == 0


def _modules(dev):
    torch.manual_seed(0)
    args = MoEArgs(num_experts=E, top_k=K, route_norm=True)
    norm, moe, block = RMSNorm(H).to(dev), AnnotatedMoE(args, H, I).to(dev), MoEFeedForwardBlock(args, H, I).to(dev)
    moe.init_weights()
    block.moe.init_weights()
    return {"norm": norm, "moe": moe, "block": block}


class _Call(torch.nn.Module):
    """One piecewise operator as a module, for torch.jit.trace."""

    def __init__(self, name, dev):
        super().__init__()
        self.name = name
        self.gate = torch.nn.Parameter(_params(dev)["w_gate"].detach())
        self.w = torch.nn.ParameterList([t.detach() for n, t in _params(dev, torch.float32).items() if n in ("w1", "w2", "w3")])
        self.register_buffer("perm", torch.randperm(T, generator=torch.Generator().manual_seed(0)).int().to(dev))
        self.register_buffer("counts", torch.full((E,), T // E, dtype=torch.int32, device=dev))
        self.register_buffer("one", torch.ones(T, 1, device=dev))

    def forward(self, x):
        if self.name == "router":
            return F_.router(x, self.gate, None, top_k=K, route_norm=True)[0]
        if self.name == "permute":
            return F_.permute(x, self.perm, 1)
        if self.name == "combine":
            return F_.combine(x, self.perm, self.one)
        return F_.bmm_experts(*self.w, x, self.counts)


@pytest.mark.parametrize("name", ["norm", "moe", "block", "router", "permute", "combine", "experts"])
def test_jit_trace_records_the_operators(dev, name):
    """A traced module computes its output from its input: the kernels' results are no constants of the trace."""
    print(f"[case] jit.trace, {name}", flush=True)
    g = torch.Generator().manual_seed(3)
    x, other = (torch.randn(T, H, generator=g).to(dev) for _ in range(2))
    mod = _modules(dev)[name] if name in ("norm", "moe", "block") else _Call(name, dev)
    if name in ("norm", "moe", "block"):
        x, other = x.view(2, T // 2, H), other.view(2, T // 2, H)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        traced = torch.jit.trace(mod, x, check_trace=False)
    assert torch.equal(traced(other), mod(other))


class _Names(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen.append(getattr(func, "__name__", ""))
        return func(*args, **(kwargs or {}))


class _Subclass(torch.Tensor):
    pass


@pytest.mark.parametrize("name,operators", [("norm", ["rmsnorm"]), ("moe", ["expert_region"]), ("block", ["rmsnorm", "expert_region"]),
                                            ("experts", ["bmm_experts"])])
def test_torch_function_sees_the_operators(dev, name, operators):
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(3)).to(dev)
    mod = _Call(name, dev) if name == "experts" else _modules(dev)[name]
    x = x if name == "experts" else x.view(2, T // 2, H)
    with _Names() as names:
        out = mod(x)
    assert [n for n in names.seen if n in ("rmsnorm", "expert_region", "bmm_experts")] == operators
    sub = mod(x.as_subclass(_Subclass))
    assert type(sub) is _Subclass and torch.equal(sub.as_subclass(torch.Tensor), out)


@pytest.mark.parametrize("name,operators", [("norm", {"piper_amd::rmsnorm"}), ("moe", {"piper_amd::expert_region"}),
                                            ("block", {"piper_amd::expert_region"}), ("experts", {"piper_artifact::bmm_experts"})])
def test_the_profiler_names_the_operators(dev, name, operators):
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(3)).to(dev)
    mod = _Call(name, dev) if name == "experts" else _modules(dev)[name]
    x = x if name == "experts" else x.view(2, T // 2, H)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        mod(x)
    assert operators <= {e.key for e in prof.key_averages()}


def test_tensors_of_another_device_are_refused(dev):
    """A kernel cannot read host memory: an operand on the CPU, the row counts among them, is an error on the
    host, and so are operands too short for what the kernels read."""
    p = {n: t.detach() for n, t in _params(dev).items()}
    x, _ = _activations(dev, T)
    counts = torch.full((E,), T // E, dtype=torch.int32, device=dev)
    perm, one = torch.arange(T, dtype=torch.int32, device=dev), torch.ones(T, 1, device=dev)
    w = (p["w1"], p["w2"], p["w3"])
    flat, grad = torch.zeros(16, device=dev), torch.nn.Parameter(torch.zeros(16))
    grad.grad = torch.ones(16)
    st = [torch.zeros(16, device=dev) for _ in range(3)]
    calls = {
        "counts": lambda: F_.bmm_experts(*w, x, counts.cpu()),
        "counts, operator": lambda: torch.ops.piper_artifact.bmm_experts(*w, x, counts.cpu()),
        "short counts": lambda: F_.bmm_experts(*w, x, counts[:-1]),
        "other width": lambda: F_.bmm_experts(*w, x[:, :128].contiguous(), counts),
        "expert weight": lambda: F_.bmm_experts(p["w1"].cpu(), p["w2"], p["w3"], x, counts),
        "region weight": lambda: _region(x, dict(p, w2=p["w2"].cpu())),
        "norm weight": lambda: F_.rmsnorm(x, p["norm"].cpu()),
        "gate weight": lambda: F_.router(x, p["w_gate"].cpu(), None, top_k=K, route_norm=True),
        "permutation": lambda: F_.permute(x, perm.cpu(), 1),
        "combine permutation": lambda: F_.combine(x, perm.cpu(), one),
        "short permutation": lambda: F_.combine(x, perm[:-1], one),
        "packed gradient": lambda: host().pack_param_grads([(grad, 0, 16, (16,))], flat, None),
        "AdamW gradient": lambda: ops.adamw_fused_packed(*st, None, [torch.ones(16)], [0], [16], step=1, lr=1e-3, beta1=0.9, beta2=0.95,
                                                         eps=1e-8, weight_decay=0.1),
    }
    for name, call in calls.items():
        print(f"[case] refused operand: {name}", flush=True)
        with pytest.raises((RuntimeError, ValueError)):
            call()
    assert grad.grad is not None
    torch.cuda.synchronize()
