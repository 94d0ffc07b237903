"""GPU parity of the routing kernels against the CPU oracle: indices, permutation and offsets are
compared bit-exactly, scores and gradients to the fp32 tolerance."""
import pytest
import torch

from conftest import F32_TOL, rel_err
from oracle import moe as O
from piper_amd import ops

pytestmark = pytest.mark.gpu


def _note(msg):
    print(f"[case] {msg}", flush=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,H,E,bias", [(256, 256, 8, False), (1000, 2048, 128, True), (3, 40, 5, True)])
def test_gate_logits(dev, dtype, T, H, E, bias):
    _note(f"gate_logits {dtype} T={T} H={H} E={E} bias={bias}")
    g = torch.Generator().manual_seed(0)
    x = torch.randn(T, H, generator=g).to(dtype)
    w = torch.randn(E, H, generator=g) * 0.02
    b = torch.randn(E, generator=g) if bias else None
    got = ops.gate_logits(x.to(dev), w.to(dev), None if b is None else b.to(dev))
    ref = O.gate_logits(x, w, b)
    assert got.dtype == torch.float32
    assert rel_err(got, ref) <= F32_TOL


def _check_topk(dev, logits, K, route_norm, scale=1.0):
    s_ref, i_ref = O.route_topk(logits, K, route_norm, scale)
    s, i = ops.route_topk(logits.to(dev), K, route_norm, scale)
    assert i.dtype == torch.int32
    assert torch.equal(i.cpu().long(), i_ref), "routing indices must be bit-exact"
    assert rel_err(s, s_ref) <= F32_TOL
    return s, i


@pytest.mark.parametrize("T,E,K", [(4096, 128, 8), (1027, 8, 2), (64, 64, 64), (33, 200, 6), (10, 1024, 64), (5, 3, 1), (7, 65, 65 - 1)])
@pytest.mark.parametrize("route_norm", [True, False])
def test_route_topk_random(dev, T, E, K, route_norm):
    _note(f"route_topk random T={T} E={E} K={K} norm={route_norm}")
    g = torch.Generator().manual_seed(T + E + K)
    _check_topk(dev, torch.randn(T, E, generator=g) * 0.9, min(K, 64), route_norm, 1.0 if route_norm else 2.5)


def test_route_topk_ties_to_lower_index(dev):
    _note("route_topk ties")
    g = torch.Generator().manual_seed(5)
    T, E, K = 2048, 128, 8
    # heavy quantisation: many exact ties in every row
    logits = torch.round(torch.randn(T, E, generator=g) * 2.0) / 2.0
    logits[0] = 0.0                       # all equal -> experts 0..7
    logits[1] = 0.0
    logits[1, 5] = -0.0                   # signed zero is still a tie
    logits[2] = torch.arange(E).float()   # strictly increasing -> highest indices, descending
    logits[3, :] = -3.0
    logits[3, 100:] = 7.0                 # 28 equal maxima -> 100..107
    s, i = _check_topk(dev, logits, K, True)
    i = i.cpu()
    assert i[0].tolist() == list(range(8)) and i[1].tolist() == list(range(8))
    assert i[2].tolist() == list(range(127, 119, -1))
    assert i[3].tolist() == list(range(100, 108))


def test_route_topk_argument_errors(dev):
    logits = torch.zeros(4, 8, device=dev)
    with pytest.raises(RuntimeError, match="shape"):
        ops.route_topk(logits, 9, True)          # K > E
    with pytest.raises(RuntimeError, match="shape"):
        ops.route_topk(torch.zeros(2, 2000, device=dev), 2, True)   # E > 1024
    s, i = ops.route_topk(torch.zeros(0, 8, device=dev), 2, True)    # empty input is fine
    assert s.shape == (0, 2)


@pytest.mark.parametrize("T,E,K,empty", [(4096, 128, 8, False), (16384, 128, 8, True), (37, 8, 2, True), (1, 5, 3, False), (700, 1024, 4, True), (64, 8, 8, False)])
def test_sort_by_expert_bit_exact(dev, T, E, K, empty):
    _note(f"sort T={T} E={E} K={K} empty={empty}")
    g = torch.Generator().manual_seed(T * 7 + E)
    logits = torch.randn(T, E, generator=g)
    if empty:
        logits[:, E // 2] = -100.0      # an expert that receives nothing
        logits[:, 0] += 3.0             # and a very popular one
    _, idx = O.route_topk(logits, K, True)
    c_ref, s_ref, p_ref, inv_ref = O.sort_by_expert(idx, E)
    counts, starts, perm, inv = ops.sort_by_expert(idx.int().to(dev), E)
    assert torch.equal(counts.cpu().long(), c_ref)
    assert torch.equal(starts.cpu().long(), s_ref)
    assert torch.equal(perm.cpu().long(), p_ref), "permutation order must be bit-exact"
    assert torch.equal(inv.cpu().long(), inv_ref)
    if empty:
        assert counts[E // 2].item() == 0
    st = ops.counts_to_starts(counts)
    assert torch.equal(st.cpu(), starts.cpu())
    st64 = ops.counts_to_starts(counts.long())
    assert torch.equal(st64.cpu(), starts.cpu())


def test_sort_with_repeated_expert_in_a_row(dev):
    # the sort itself does not require distinct experts per token
    _note("sort duplicates")
    g = torch.Generator().manual_seed(9)
    idx = torch.randint(0, 16, (999, 4), generator=g)
    ref = O.sort_by_expert(idx, 16)
    got = ops.sort_by_expert(idx.int().to(dev), 16)
    for a, b in zip(got, ref):
        assert torch.equal(a.cpu().long(), b)


@pytest.mark.parametrize("route_norm", [True, False])
@pytest.mark.parametrize("T,E,K", [(512, 128, 8), (100, 8, 2), (9, 300, 5)])
def test_route_topk_backward(dev, T, E, K, route_norm):
    _note(f"route_topk_bwd T={T} E={E} K={K} norm={route_norm}")
    g = torch.Generator().manual_seed(11)
    logits = (torch.randn(T, E, generator=g) * 0.9).requires_grad_(True)
    d_scores = torch.randn(T, K, generator=g)
    s_ref, i_ref = O.route_topk(logits, K, route_norm, 1.5)
    (d_ref,) = torch.autograd.grad(s_ref, logits, d_scores)
    got = ops.route_topk_bwd(logits.detach().to(dev), i_ref.int().to(dev), d_scores.to(dev), route_norm, 1.5)
    assert rel_err(got, d_ref) <= F32_TOL


# (the bias gradient of the longer inputs is summed in two steps: row ranges, then the partial rows)
@pytest.mark.parametrize("T,H,E", [(777, 256, 24), (4099, 256, 128), (2500, 128, 20)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gate_logits_backward(dev, dtype, T, H, E):
    _note(f"gate_logits_bwd {dtype} T={T} H={H} E={E}")
    g = torch.Generator().manual_seed(12)
    x = torch.randn(T, H, generator=g).to(dtype)
    w = (torch.randn(E, H, generator=g) * 0.02)
    d_logits = torch.randn(T, E, generator=g)
    xr = x.float().requires_grad_(True)
    wr = w.clone().requires_grad_(True)
    br = torch.zeros(E, requires_grad=True)
    ref = O.gate_logits(xr, wr, br)
    dx_ref, dw_ref, db_ref = torch.autograd.grad(ref, (xr, wr, br), d_logits)
    dw = torch.zeros(E, H, device=dev)
    db = torch.zeros(E, device=dev)
    dx = ops.gate_logits_bwd(d_logits.to(dev), x.to(dev), w.to(dev), True, dw, db, accumulate=False)
    assert rel_err(dx, dx_ref) <= F32_TOL and rel_err(dw, dw_ref) <= F32_TOL and rel_err(db, db_ref) <= F32_TOL
    # accumulate adds on top
    ops.gate_logits_bwd(d_logits.to(dev), x.to(dev), w.to(dev), False, dw, db, accumulate=True)
    assert rel_err(dw, 2 * dw_ref) <= F32_TOL and rel_err(db, 2 * db_ref) <= F32_TOL


@pytest.mark.parametrize("name", ["cfg3", "cfg4"])
def test_end_to_end_routing_from_activations(dev, name):
    """x, W (, bias) -> indices at the full size of both expert-region configurations.  The GPU gate
    sums in a different order than the CPU, so logits differ in the last bits; every token whose
    indices differ from the oracle's must sit on a near-tie (margin below 1e-4 between two of its
    nine largest logits), their number is printed and bounded, and given the GPU's own logits the
    selection is bit-exact."""
    from piper_amd.configs import CFG3, CFG4, make_expert_region_inputs
    cfg = CFG3 if name == "cfg3" else CFG4
    _note(f"routing end to end ({name} shape)")
    inp = make_expert_region_inputs(cfg)
    x, w, b = inp["x"], inp["w_gate"], inp["gate_bias"]
    logits_gpu = ops.gate_logits(x.to(dev), w.to(dev), None if b is None else b.to(dev)).cpu()
    logits_ref = O.gate_logits(x, w, b)
    assert rel_err(logits_gpu, logits_ref) <= F32_TOL
    K = cfg.top_k
    _, i_gpu = ops.route_topk(logits_gpu.to(dev), K, True)
    _, i_from_gpu_logits = O.route_topk(logits_gpu, K, True)
    assert torch.equal(i_gpu.cpu().long(), i_from_gpu_logits)
    _, i_ref = O.route_topk(logits_ref, K, True)
    diff_rows = (i_gpu.cpu().long() != i_ref).any(dim=1).nonzero().flatten()
    srt = torch.sort(logits_ref, dim=1, descending=True).values
    gaps = (srt[:, :K] - srt[:, 1:K + 1])          # margins that decide order and membership
    for r in diff_rows.tolist():
        assert gaps[r].min().item() < 1e-4, f"row {r} differs without a near-tie"
    print(f"[info] {name}: {len(diff_rows)} of {cfg.tokens} tokens routed differently from the CPU evaluation "
          f"(all on margins below 1e-4)", flush=True)
    assert len(diff_rows) <= cfg.tokens // 512


def test_sort_expert_order_hint(dev):
    """order = experts by descending row count, ties to the lower index."""
    g = torch.Generator().manual_seed(3)
    idx = torch.randint(0, 24, (500, 2), generator=g).int()
    idx[idx == 7] = 3          # expert 7 empty, expert 3 popular
    counts, starts, perm, inv, order = ops.sort_by_expert(idx.to(dev), 24, with_order=True)
    c = counts.cpu().tolist()
    expect = sorted(range(24), key=lambda e: (-c[e], e))
    assert order.cpu().tolist() == expect and c[7] == 0 and expect[0] == 3


@pytest.mark.parametrize("A,E", [(1, 1), (63, 512), (1024, 128), (4096, 100), (4096, 513), (4097, 128), (8704, 7), (20000, 1000)])
def test_counting_sort_on_both_sides_of_its_dispatch(dev, A, E):
    """One workgroup (up to 4,096 slots and 512 experts) and histogram + scatter beyond: every table
    bit for bit."""
    print(f"[case] sort A={A} E={E}", flush=True)
    g = torch.Generator().manual_seed(A + E)
    ids = torch.randint(0, E, (A, 1), generator=g, dtype=torch.int32)
    counts, starts, perm, inv, order = ops.sort_by_expert(ids.to(dev), E, with_order=True)
    flat = ids.reshape(-1).long()
    want = torch.argsort(flat, stable=True)
    ref_counts = torch.bincount(flat, minlength=E)
    assert torch.equal(perm.cpu().long(), want)
    assert torch.equal(inv.cpu().long()[want], torch.arange(A))
    assert torch.equal(counts.cpu().long(), ref_counts)
    assert torch.equal(starts.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), ref_counts.cumsum(0)]))
    assert torch.equal(order.cpu().long(), torch.argsort(-ref_counts, stable=True))


@pytest.mark.parametrize("A,E", [(262144, 128), (262145, 17), (524288, 16), (524289, 5), (300001, 1000), (1 << 20, 32)])
def test_counting_sort_of_many_chunks(dev, A, E):
    """512 chunks of slots (1,024 with few experts), whose workgroups add up the chunk histograms themselves,
    and more, where one workgroup does it for all: every table bit for bit, with an expert that gets nothing."""
    print(f"[case] sort A={A} E={E}", flush=True)
    g = torch.Generator().manual_seed(A + E)
    ids = torch.randint(0, E, (A, 1), generator=g, dtype=torch.int32)
    ids[ids == E // 2] = 0
    counts, starts, perm, inv, order = ops.sort_by_expert(ids.to(dev), E, with_order=True)
    flat = ids.reshape(-1).long()
    want = torch.argsort(flat, stable=True)
    ref_counts = torch.bincount(flat, minlength=E)
    assert torch.equal(perm.cpu().long(), want)
    assert torch.equal(inv.cpu().long()[want], torch.arange(A))
    assert torch.equal(counts.cpu().long(), ref_counts)
    assert torch.equal(starts.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), ref_counts.cumsum(0)]))
    assert torch.equal(order.cpu().long(), torch.argsort(-ref_counts, stable=True))


def test_sort_time_grows_with_the_slots(dev):
    """Four times the slots take about four times as long (sixteen where every chunk reads all others)."""
    def us(A, E=1024):
        idx = torch.randint(0, E, (A, 1), device=dev, dtype=torch.int32)
        ops.sort_by_expert(idx, E)
        best = float("inf")
        for _ in range(3):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ops.sort_by_expert(idx, E)
            b.record()
            b.synchronize()
            best = min(best, 1e3 * a.elapsed_time(b))
        return best

    short, long = us(1 << 20), us(1 << 22)
    print(f"[case] sort of 1 M and 4 M slots, 1,024 experts: {short:.0f} and {long:.0f} us", flush=True)
    assert long <= 8 * short


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,E", [(2048, 128), (1000, 120), (1800, 96), (2040, 64)])
def test_gate_with_its_reduction_requested_at_once(dev, dtype, H, E):
    """Up to 256 workgroups the gate requests a workgroup's whole reduction at once (four or eight k-tiles, the last ones
    partly or wholly past the end); one row of tokens more and it goes k-tile by k-tile.  The same products in the same
    order: the tokens of both calls get the same logits bit for bit, and those of the oracle."""
    _note(f"gate ahead {dtype} H={H} E={E}")
    splits = max(1, min(8, H // 128))
    T = 64 * (256 // splits)
    g = torch.Generator().manual_seed(9)
    x = torch.randn(T + 1, H, generator=g).to(dtype)
    w = torch.randn(E, H, generator=g) * 0.05
    few, more = ops.gate_logits(x[:T].to(dev), w.to(dev)), ops.gate_logits(x.to(dev), w.to(dev))
    assert torch.equal(few, more[:T])
    assert rel_err(few, O.gate_logits(x[:T], w, None)) <= F32_TOL


def _launches(fn):
    """what fn returns, and the names of the kernels it launched"""
    from piper_amd import _lib
    _lib.timing_enable(True)
    _lib.timing_collect()
    out = fn()
    names = [n for n, _ in _lib.timing_collect()]
    _lib.timing_enable(False)
    return out, names


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("dtype,T,H,E", [
    (torch.bfloat16, 65, 1024, 32), (torch.bfloat16, 200, 264, 17), (torch.bfloat16, 3000, 1000, 33), (torch.bfloat16, 2500, 488, 65),
    (torch.bfloat16, 4096, 512, 128), (torch.bfloat16, 4096, 256, 100), (torch.bfloat16, 2000, 1992, 24), (torch.float32, 65, 512, 20),
    (torch.float32, 130, 260, 31), (torch.float32, 1030, 1000, 24), (torch.float32, 4096, 300, 97), (torch.float32, 4095, 1020, 32)])
def test_gate_in_the_front_kernel_gives_the_bits_of_the_gate_gemm(dev, dtype, T, H, E, bias):
    """gate_front_kernel against pk_x3mm::kernel: the same tokens and experts with more experts behind them than the front
    kernel takes (129), which leaves the reduction's splits as they are.  Every pair of logits is equal bit for bit, with
    two to eight splits, one to four tiles of experts, widths that end inside a step and operands of three planes."""
    _note(f"front against gemm {dtype} T={T} H={H} E={E}")
    g = torch.Generator().manual_seed(T + H + E)
    x = torch.randn(T, H, generator=g).to(dtype).to(dev)
    w = (torch.randn(129, H, generator=g) * 0.05).to(dev)
    b = torch.randn(129, generator=g).to(dev) if bias else None
    front, few = _launches(lambda: ops.gate_logits(x, w[:E].contiguous(), b[:E].contiguous() if bias else None))
    gemm, many = _launches(lambda: ops.gate_logits(x, w, b))
    assert len(few) == 1 and len(many) == 2      # (the GEMM's partial results are added up by a second launch)
    assert torch.equal(front, gemm[:, :E])
    assert rel_err(gemm.double().cpu(), x.double().cpu() @ w.double().cpu().t() + (b.double().cpu() if bias else 0.0)) <= F32_TOL


@pytest.mark.parametrize("dtype,T,H,E,alone,with_norm", [
    (torch.bfloat16, 65, 768, 32, True, True), (torch.bfloat16, 4096, 768, 32, True, True), (torch.bfloat16, 4097, 256, 32, True, True),
    (torch.bfloat16, 2048, 512, 64, True, True), (torch.bfloat16, 4096, 768, 96, True, True), (torch.float32, 1024, 512, 16, True, True),
    # more weight than the launches it stands for are worth, a few tokens
    (torch.bfloat16, 65, 1024, 96, False, False), (torch.bfloat16, 500, 768, 128, False, False), (torch.float32, 100, 1000, 96, False, False),
    (torch.float32, 1030, 1000, 48, False, False), (torch.bfloat16, 300, 1024, 64, False, True), (torch.bfloat16, 2048, 768, 128, False, True),
    # one token more than the CUs take at once
    (torch.bfloat16, 4097, 768, 128, False, False), (torch.bfloat16, 4097, 2048, 48, False, False), (torch.float32, 4097, 1000, 96, False, False),
    (torch.bfloat16, 4097, 768, 32, False, True), (torch.bfloat16, 8192, 1536, 64, False, False)])
def test_the_front_kernel_is_taken_where_it_pays(dev, dtype, T, H, E, alone, with_norm):
    """gate_front_kernel on either side of front_pays, for the gate alone and with norm, top-k and sort: where it was taken and
    took up to twice as long as the launches it stands for, those are back.  The same bits from every one of them."""
    from piper_amd import _lib
    from piper_amd._lib import call, current_stream, dtype_code, ptr
    _note(f"front kernel {dtype} T={T} H={H} E={E}")
    K = min(E, 4)
    g = torch.Generator().manual_seed(T + H + E)
    x, norm_w = torch.randn(T, H, generator=g).to(dtype).to(dev), torch.ones(H, dtype=dtype, device=dev)
    w = (torch.randn(E, H, generator=g) * 0.02).to(dev)
    xn = ops.rmsnorm_fwd(x, norm_w, 1e-6)[0]
    gate, names = _launches(lambda: ops.gate_logits(xn, w, None))
    assert len(names) == (1 if alone else 2), names
    ws = torch.empty(int(_lib.load().pk_gate_route_sort_workspace_bytes(T, H, E, K)), dtype=torch.uint8, device=dev)
    got = [torch.empty_like(x), torch.empty(T, device=dev), torch.empty_like(gate), torch.empty(T, K, device=dev)]
    ints = [torch.empty(n, dtype=torch.int32, device=dev) for n in (T * K, E + 1, T * K)]
    _, names = _launches(lambda: call("pk_norm_gate_route_sort", ptr(x), dtype_code(dtype), ptr(norm_w), 1e-6, ptr(got[0]), ptr(got[1]), ptr(w), None,
                                      T, H, E, K, 1, 1.0, ptr(got[2]), ptr(got[3]), ptr(ints[0]), None, ptr(ints[1]), ptr(ints[2]), None, None,
                                      ptr(ws), ws.numel(), current_stream(dev)))
    assert ("rmsnorm_fwd" not in names) == with_norm, names
    scores, idx = ops.route_topk(gate, K, True)
    assert torch.equal(got[0], xn) and torch.equal(got[2], gate) and torch.equal(got[3], scores) and torch.equal(ints[0].view(T, K), idx)
    assert torch.equal(ints[2], ops.sort_by_expert(idx, E)[2])


@pytest.mark.parametrize("T,H,E,K,bias", [(1, 256, 8, 2, True), (65, 2048, 128, 8, False), (70, 520, 130, 5, True), (5000, 2048, 128, 8, True)])
def test_gate_and_topk_in_one_call_match_the_two_calls(dev, T, H, E, K, bias):
    """pk_gate_route sums the gate GEMM's split-K partial results inside the top-k kernel: logits,
    scores and indices bit for bit those of pk_gate_logits followed by pk_route_topk."""
    from piper_amd._lib import host
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H, generator=g).bfloat16().to(dev)
    w = (torch.randn(E, H, generator=g) * 0.02).to(dev)
    b = torch.randn(E, generator=g).to(dev) if bias else None
    want_s, want_i = ops.route_topk(ops.gate_logits(x, w, b), K, True, 1.5)
    got_s, got_i = host().router(x, w, b, K, True, 1.5, None)
    assert torch.equal(got_i, want_i) and torch.equal(got_s, want_s)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,H,E,K", [(1, 8, 4, 2), (33, 136, 8, 3), (300, 2048, 128, 8), (65, 72, 6, 2), (40, 70, 12, 9)])
def test_router_backward_in_one_call_matches_the_three_calls(dev, dtype, T, H, E, K):
    """pk_region_router_bwd adds the gate's share of d_x where the routed rows are gathered: d_logits, d_x
    and the gate's gradients bit for bit those of route_topk_bwd, gate_logits_bwd and permute_bwd, with
    the score gradients given directly and as partial sums; widths that cannot be read in 16-byte
    pieces take the separate kernels inside."""
    from piper_amd import _lib
    from piper_amd._lib import call, current_stream, dtype_code, ptr
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g).to(dtype).to(dev)
    w = (torch.randn(E, H, generator=g) * 0.02).to(dev)
    logits = torch.randn(T, E, generator=g).to(dev)
    rows = torch.randn(T * K, H, generator=g).to(dtype).to(dev)
    part = torch.randn(3, T * K, generator=g).to(dev)
    _, idx = ops.route_topk(logits, K, True)
    _, _, perm, inv = ops.sort_by_expert(idx, E)
    d_s = ((part[0] + part[1]) + part[2])[inv.long()].reshape(T, K)
    d_logits = ops.route_topk_bwd(logits, idx, d_s, True, 1.5)
    want_w, want_b = torch.empty_like(w), torch.empty(E, device=dev)
    d_x32 = ops.gate_logits_bwd(d_logits, x, w, d_w_gate=want_w, d_gate_bias=want_b)
    want_x = ops.permute_bwd(rows, inv, K, addend_f32=d_x32)
    ws = torch.empty(int(_lib.load().pk_region_router_bwd_workspace_bytes(T, H, E, dtype_code(dtype))), dtype=torch.uint8, device=dev)
    for partial in (False, True):
        got_l, got_x, got_w, got_b = torch.empty_like(logits), torch.empty_like(x), torch.empty_like(w), torch.empty(E, device=dev)
        call("pk_region_router_bwd", ptr(logits), ptr(idx), None if partial else ptr(d_s), ptr(part), 3, ptr(inv), 1, 1.5, ptr(x),
             dtype_code(dtype), ptr(w), ptr(rows), ptr(got_x), ptr(got_w), ptr(got_b), 0, ptr(got_l), T, H, E, K, ptr(ws), ws.numel(),
             current_stream(dev))
        assert torch.equal(got_l, d_logits) and torch.equal(got_x, want_x) and torch.equal(got_w, want_w) and torch.equal(got_b, want_b)


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("dtype,T,H,E,K", [(torch.bfloat16, 1, 8, 4, 2), (torch.float32, 33, 136, 8, 3), (torch.bfloat16, 2100, 256, 132, 4),
                                           (torch.float32, 2048, 2052, 4, 1), (torch.bfloat16, 300, 70, 12, 9), (torch.bfloat16, 40, 8200, 8, 2)])
def test_router_and_norm_backward_share_launches(dev, dtype, T, H, E, K, accumulate):
    """pk_region_router_norm_bwd: everything that pk_region_router_bwd and pk_rmsnorm_bwd give one after the other, bit for
    bit, with the gate's gradients split or not, the bias in one or two steps, and rows that fit a wave or do not."""
    from piper_amd import _lib
    from piper_amd._lib import call, current_stream, dtype_code, ptr
    g = torch.Generator().manual_seed(T + H)
    x, rows, addend = (torch.randn(n, H, generator=g).to(dtype).to(dev) for n in (T, T * K, T))
    w = (torch.randn(E, H, generator=g) * 0.02).to(dev)
    norm_w = torch.randn(H, generator=g).to(dtype).to(dev)
    xn, rstd = ops.rmsnorm_fwd(x, norm_w, 1e-6)
    logits, d_s = torch.randn(T, E, generator=g).to(dev), torch.randn(T, K, generator=g).to(dev)
    _, idx = ops.route_topk(logits, K, True)
    inv = ops.sort_by_expert(idx, E)[3]
    old_w, old_b, old_n = torch.randn(E, H, generator=g).to(dev), torch.randn(E, generator=g).to(dev), torch.randn(H, generator=g).to(dtype).to(dev)
    lib, code, stream = _lib.load(), dtype_code(dtype), current_stream(dev)

    def run(entry, ws_bytes, middle, norm):
        out = [torch.empty_like(logits), torch.empty_like(x), old_w.clone(), old_b.clone(), torch.empty_like(x), old_n.clone()]
        d_l, d_xn, d_w, d_b, d_x, d_n = out
        ws = torch.empty(int(ws_bytes), dtype=torch.uint8, device=dev)
        call(entry, ptr(logits), ptr(idx), ptr(d_s), None, 0, ptr(inv), 1, 1.5, ptr(xn), code, ptr(w), ptr(rows), ptr(d_xn), ptr(d_w),
             ptr(d_b), int(accumulate), ptr(d_l), *([ptr(t) for t in (x, norm_w, rstd, addend, d_x, d_n)] if middle else []), T, H, E, K,
             ptr(ws), ws.numel(), stream)
        if norm:
            nws = torch.empty(int(lib.pk_rmsnorm_bwd_workspace_bytes(T, H)), dtype=torch.uint8, device=dev)
            call("pk_rmsnorm_bwd", ptr(d_xn), ptr(x), code, ptr(norm_w), ptr(rstd), ptr(addend), ptr(d_x), ptr(d_n), int(accumulate), T, H,
                 ptr(nws), nws.numel(), stream)
        return out

    want = run("pk_region_router_bwd", lib.pk_region_router_bwd_workspace_bytes(T, H, E, code), False, True)
    got = run("pk_region_router_norm_bwd", lib.pk_region_router_norm_bwd_workspace_bytes(T, H, E, code), True, False)
    for name, a, b in zip(("d_logits", "d_xn", "d_w_gate", "d_gate_bias", "d_x", "d_norm_weight"), got, want):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("dtype,T,H,E,K,bias", [
    (torch.bfloat16, 1, 8, 1, 1, False), (torch.float32, 15, 36, 5, 5, True), (torch.bfloat16, 16, 1000, 24, 4, False),
    (torch.float32, 17, 2048, 16, 2, True), (torch.bfloat16, 33, 392, 17, 17, True), (torch.bfloat16, 1030, 1000, 64, 64, False),
    (torch.bfloat16, 65, 768, 128, 8, True), (torch.float32, 500, 1028, 65, 3, False), (torch.bfloat16, 8192, 256, 32, 6, False),
    (torch.bfloat16, 100, 2048, 24, 3, True), (torch.float32, 40, 1024, 16, 2, False), (torch.bfloat16, 4100, 256, 72, 2, False),
    (torch.bfloat16, 70, 1032, 40, 2, True), (torch.bfloat16, 24, 2048, 128, 8, True), (torch.float32, 64, 8188, 20, 3, False),
    (torch.bfloat16, 33, 8200, 130, 2, False), (torch.float32, 65, 36, 5, 5, True), (torch.bfloat16, 81, 8, 1, 1, False),
    (torch.bfloat16, 66, 1000, 33, 33, True),
    (torch.bfloat16, 64, 1032, 32, 8, True), (torch.bfloat16, 8193, 64, 8, 2, False), (torch.bfloat16, 40, 4104, 8, 2, False)])
def test_norm_gate_topk_and_sort_in_one_call(dev, dtype, T, H, E, K, bias):
    """pk_norm_gate_route_sort on either side of every limit of its one-launch path: bit for bit what the norm, the gate,
    the top-k and the sort give one by one, the logits within 1e-5 of float64 on the norm's output."""
    from piper_amd import _lib
    from piper_amd._lib import call, current_stream, dtype_code, ptr
    g = torch.Generator().manual_seed(T + H + E)
    x, norm_w = torch.randn(T, H, generator=g).to(dtype).to(dev), torch.randn(H, generator=g).to(dtype).to(dev)
    w = (torch.randn(E, H, generator=g) * 0.02).to(dev)
    b = torch.randn(E, generator=g).to(dev) if bias else None
    want_xn, want_rstd = ops.rmsnorm_fwd(x, norm_w, 1e-6)
    want_l = ops.gate_logits(want_xn, w, b)
    want_s, want_i = ops.route_topk(want_l, K, True, 1.5)
    want_sort = ops.sort_by_expert(want_i, E, with_order=True)
    ws = torch.empty(int(_lib.load().pk_gate_route_sort_workspace_bytes(T, H, E, K)), dtype=torch.uint8, device=dev)
    i32 = dict(dtype=torch.int32, device=dev)
    for norm in (True, False):
        xn, rstd, logits, scores = torch.empty_like(x), torch.empty_like(want_rstd), torch.empty_like(want_l), torch.empty_like(want_s)
        idx, got_sort = torch.empty_like(want_i), [torch.empty(n, **i32) for n in (E, E + 1, T * K, T * K, E)]
        tail = [ptr(w), ptr(b), T, H, E, K, 1, 1.5, ptr(logits), ptr(scores), ptr(idx), *[ptr(t) for t in got_sort], ptr(ws), ws.numel(),
                current_stream(dev)]
        if norm:
            call("pk_norm_gate_route_sort", ptr(x), dtype_code(dtype), ptr(norm_w), 1e-6, ptr(xn), ptr(rstd), *tail)
            assert torch.equal(xn, want_xn) and torch.equal(rstd, want_rstd)
        else:
            call("pk_gate_route_sort", ptr(want_xn), dtype_code(dtype), *tail)
        assert torch.equal(logits, want_l) and torch.equal(scores, want_s) and torch.equal(idx, want_i)
        for name, a, c in zip(("counts", "starts", "perm", "inv_perm", "order"), got_sort, want_sort):
            assert torch.equal(a, c), name
    exact = want_xn.double().cpu() @ w.double().cpu().t() + (b.double().cpu() if bias else 0.0)
    assert rel_err(want_l.double().cpu(), exact) <= F32_TOL


@pytest.mark.parametrize("T,H,E,K,bias", [(129, 2048, 128, 8, True), (1033, 1600, 61, 1, False), (2048, 1024, 128, 3, True), (2049, 1024, 128, 1, True),
                                          (205, 1024, 97, 5, False)])
def test_topk_with_the_sorts_histogram(dev, T, H, E, K, bias):
    """Above the gates that gate_front_kernel takes and up to 16 K chunk counts (2,048 tokens of 128 experts, 2,049 are too
    many): the top-k writes the histograms of 16 tokens each that the sort places the slots by.  Partly filled last
    chunks, one and two experts a lane, more than 1,024 slots: bit for bit the separate calls."""
    test_norm_gate_topk_and_sort_in_one_call(dev, torch.bfloat16, T, H, E, K, bias)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("product", ["forward", "d_x", "weight gradient"])
def test_router_products_at_every_end_of_their_k_loops(dev, dtype, product):
    """No, one to seven whole k-tiles of 32 with and without a part of one behind them, two in flight at most; rows and
    columns past the ends are read from the last ones.  A sum of n fp32-accurate products is within (n + 8) 2^-24 of the sum
    of their magnitudes (every plane product left out is below 2^-24 of its product)."""
    g = torch.Generator().manual_seed(31)
    for n in (4, 28, 32, 36, 64, 68, 96, 100, 128, 132, 160, 164, 192, 196, 224, 228):
        if product == "forward":             # more workgroups than are requested at once, one split
            T, H, E = 64 * 260 + 1, n, 12
        elif product == "d_x":
            T, H, E = 129, 196, n
        else:                                # 512 tiles: one split
            T, H, E = n - n % 3, 2044, 1020
        _note(f"{product} {dtype} T={T} H={H} E={E}")
        x = torch.randn(T, H, generator=g).to(dtype)
        w, d = torch.randn(E, H, generator=g) * 0.05, torch.randn(T, E, generator=g)
        if product == "forward":
            got, a, b = ops.gate_logits(x.to(dev), w.to(dev)), x.double(), w.double().t()
        elif product == "d_x":
            got, a, b = ops.gate_logits_bwd(d.to(dev), x.to(dev), w.to(dev)), d.double(), w.double()
        else:
            got = torch.empty(E, H, device=dev)
            ops.gate_logits_bwd(d.to(dev), x.to(dev), w.to(dev), False, got)
            a, b = d.double().t(), x.double()
        bound = (a.shape[1] + 8) * 2.0**-24 * (a.abs() @ b.abs())
        assert bool(((got.double().cpu() - a @ b).abs() <= bound).all()), (n, float(((got.double().cpu() - a @ b).abs() / bound).max()))
