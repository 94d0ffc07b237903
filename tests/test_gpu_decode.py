"""The decode step's three launches against the general path's kernels and the CPU oracle."""
import pytest
import torch

from conftest import BF16_TOL, rel_err
from piper_amd import _lib, ops
from piper_amd._lib import call, current_stream, ptr

pytestmark = pytest.mark.gpu


def _inputs(dev, T, H, E, I, bias, residual, seed):
    g = torch.Generator().manual_seed(seed)
    bf = torch.bfloat16
    t = dict(x=torch.randn(T, H, generator=g).to(bf), norm_w=(1 + 0.1 * torch.randn(H, generator=g)).to(bf),
             w_gate=torch.randn(E, H, generator=g) * 0.05, bias=torch.randn(E, generator=g) if bias else None,
             w1=(torch.randn(E, I, H, generator=g) * 0.05).to(bf), w2=(torch.randn(E, H, I, generator=g) * 0.05).to(bf),
             w3=(torch.randn(E, I, H, generator=g) * 0.05).to(bf), residual=torch.randn(T, H, generator=g).to(bf) if residual else None)
    return {k: None if v is None else v.to(dev) for k, v in t.items()}


@pytest.mark.parametrize("T,H,E,I,K,norm,bias,residual", [
    (1, 2048, 128, 768, 8, True, False, True), (2, 2048, 128, 768, 8, True, True, True), (1, 8, 1, 8, 1, False, False, False),
    (16, 264, 5, 40, 1, True, True, False), (4, 1000, 4, 360, 4, False, False, True), (3, 520, 70, 1024, 5, True, False, True),
    (1, 2056, 300, 776, 16, False, True, False), (2, 72, 1024, 2056, 7, True, False, True)])
def test_decode_step(dev, T, H, E, I, K, norm, bias, residual):
    """Same logits, scores and experts as the general path's router, bit for bit (read back from the workspace), output within bf16
    of float64 on the same experts: tokens that share experts, one expert for all, widths around the 64-deep steps and
    beyond a wave's share in flight."""
    t = _inputs(dev, T, H, E, I, bias, residual, T * H + E)
    need = int(_lib.load().pk_region_decode_workspace_bytes(T, H, E, I, K, _lib.PK_BF16))
    ws, out = torch.empty(need, dtype=torch.uint8, device=dev), torch.empty_like(t["x"])
    call("pk_region_decode", ptr(t["x"]), _lib.PK_BF16, ptr(t["norm_w"] if norm else None), 1e-6, ptr(t["w_gate"]), ptr(t["bias"]), ptr(t["w1"]),
         ptr(t["w2"]), ptr(t["w3"]), 1, 1.5, ptr(t["residual"]), ptr(out), T, H, E, I, K, ptr(ws), need, current_stream(dev))
    x = ops.rmsnorm_fwd(t["x"], t["norm_w"], 1e-6)[0] if norm else t["x"]
    # the workspace: the norm's output, logits, scores, experts and h, each from a multiple of 256 bytes on
    at, took = 0, []
    for n, dtype in ((T * H, torch.bfloat16), (T * E, torch.float32), (T * K, torch.float32), (T * K, torch.int32), (T * K * I, torch.bfloat16)):
        took.append(ws[at:at + n * dtype.itemsize].view(dtype))
        at += (n * dtype.itemsize + 255) // 256 * 256
    assert at == need
    router = ops.gate_logits(x, t["w_gate"], t["bias"])
    scores, experts = ops.route_topk(router, K, True, 1.5)
    if norm:
        assert torch.equal(took[0].view(T, H), x)
    assert torch.equal(took[1].view(T, E), router) and torch.equal(took[2].view(T, K), scores) and torch.equal(took[3].view(T, K), experts)
    d = {k: None if v is None else v.double().cpu() for k, v in t.items()}
    xd = x.double().cpu()
    logits = xd @ d["w_gate"].t() + (d["bias"] if bias else 0.0)
    top, idx = torch.topk(logits, K, dim=1)
    assert E == K or (top[:, -1] - torch.sort(logits, dim=1, descending=True)[0][:, K]).min() > 1e-5      # (no near-tie decides)
    s = torch.gather(torch.softmax(logits, 1), 1, idx)
    s = 1.5 * s / s.sum(1, keepdim=True)
    want = d["residual"].clone() if residual else torch.zeros(T, H, dtype=torch.float64)
    for i in range(T):
        for k in range(K):
            e = int(idx[i, k])
            gate, up = d["w1"][e] @ xd[i], d["w3"][e] @ xd[i]
            want[i] += s[i, k] * (d["w2"][e] @ (gate * torch.sigmoid(gate) * up))
    assert rel_err(out.double().cpu(), want) <= BF16_TOL


def test_decode_step_is_what_the_region_runs(dev):
    """expert_region and moe_block without a backward take the three launches, with one the general path; both agree."""
    from piper_amd import functional as F_
    t = _inputs(dev, 2, 256, 16, 128, False, False, 5)
    args = (t["w_gate"], None, t["w1"], t["w2"], t["w3"])
    for fn in (lambda x: F_.moe_block(x, t["norm_w"], *args, top_k=4, route_norm=True),
               lambda x: F_.expert_region(x, *args, top_k=4, route_norm=True)):
        _lib.timing_enable(True)
        _lib.timing_collect()
        got = fn(t["x"])
        few = len(_lib.timing_collect())
        want = fn(t["x"].clone().requires_grad_(True)).detach()
        many = len(_lib.timing_collect())
        _lib.timing_enable(False)
        assert few == 3 and many > 3 and rel_err(got, want) <= BF16_TOL


@pytest.mark.parametrize("T,H,E,I,K,pays", [
    (1, 2048, 128, 768, 8, True), (2, 2048, 128, 768, 8, True), (14, 2048, 128, 768, 1, False), (12, 2048, 64, 768, 1, True), (16, 1024, 8, 512, 1, False),
    (10, 1024, 8, 512, 1, True), (16, 1000, 24, 360, 1, True), (2, 512, 64, 512, 8, False), (1, 512, 64, 512, 8, True), (5, 1024, 128, 384, 2, True),
    (2, 1024, 128, 384, 8, False), (1, 1024, 8, 4096, 4, False), (1, 1024, 8, 4096, 2, True), (16, 1024, 4, 512, 1, True), (2, 8192, 4, 1024, 4, False)])
def test_decode_step_where_it_pays(dev, T, H, E, I, K, pays):
    """On either side of pk_region_decode_pays the region takes the path that is the faster one there: three launches or the general
    path's.  Where it does not pay the three launches still give the same result when they are called."""
    from piper_amd import functional as F_
    lib = _lib.load()
    assert bool(lib.pk_region_decode_pays(T, H, E, I, K)) == pays
    t = _inputs(dev, T, H, E, I, False, False, T + H + E + I)
    _lib.timing_enable(True)
    _lib.timing_collect()
    got = F_.expert_region(t["x"], t["w_gate"], None, t["w1"], t["w2"], t["w3"], top_k=K, route_norm=True)
    names = [n for n, _ in _lib.timing_collect()]
    _lib.timing_enable(False)
    assert (names == ["gate_logits", "swiglu_gate_up", "swiglu_down"]) == pays, names
    need = int(lib.pk_region_decode_workspace_bytes(T, H, E, I, K, _lib.PK_BF16))
    ws, out = torch.empty(need, dtype=torch.uint8, device=dev), torch.empty_like(t["x"])
    call("pk_region_decode", ptr(t["x"]), _lib.PK_BF16, None, 0.0, ptr(t["w_gate"]), None, ptr(t["w1"]), ptr(t["w2"]), ptr(t["w3"]), 1, 1.0, None,
         ptr(out), T, H, E, I, K, ptr(ws), need, current_stream(dev))
    assert torch.equal(got, out) if pays else rel_err(got, out) <= BF16_TOL


@pytest.mark.parametrize("tokens", [1, 100])
def test_eps_that_the_norm_refuses(dev, tokens):
    """moe_block with an eps below zero raises whichever path its tokens take."""
    from piper_amd import functional as F_
    t = _inputs(dev, tokens, 256, 16, 128, False, False, 6)
    with torch.no_grad(), pytest.raises(RuntimeError, match="invalid argument"):
        F_.moe_block(t["x"], t["norm_w"], t["w_gate"], None, t["w1"], t["w2"], t["w3"], top_k=4, route_norm=True, norm_eps=-1.0)


def test_decode_step_applies_to_few_rows_only():
    """Where it does not apply the workspace query says so (CPU side of the rule; the call itself refuses)."""
    q = _lib.load().pk_region_decode_workspace_bytes
    assert q(2, 2048, 128, 768, 8, _lib.PK_BF16) > 0 and q(16, 64, 4, 64, 1, _lib.PK_BF16) > 0
    for refused in ((3, 2048, 128, 768, 8, _lib.PK_BF16), (1, 2048, 128, 768, 8, _lib.PK_F32), (1, 2044, 128, 768, 8, _lib.PK_BF16),
                    (1, 2048, 128, 764, 8, _lib.PK_BF16), (0, 2048, 128, 768, 8, _lib.PK_BF16)):
        assert q(*refused) == 0
    assert q(1, 2048, 0, 768, 8, _lib.PK_BF16) < 0
