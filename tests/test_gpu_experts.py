"""GPU parity of the grouped SwiGLU expert kernels (forward, input gradient, weight gradient)
against the CPU oracle.  bf16 results are judged against the oracle evaluated in fp32 on the
same bf16 inputs (tolerance 2e-2 of the output's maximum), fp32 results to 1e-5."""
import pytest
import torch

from conftest import BF16_TOL, F32_TOL, rel_err, rel_err_by_expert
from oracle import moe as O
from piper_amd import functional as F_
from piper_amd import ops

pytestmark = pytest.mark.gpu


def _make(seed, counts, H, I, dtype):
    g = torch.Generator().manual_seed(seed)
    E = len(counts)
    A = int(sum(counts))
    x = torch.randn(A, H, generator=g).to(dtype)
    w1 = (torch.randn(E, I, H, generator=g) * 0.05).to(dtype)
    w3 = (torch.randn(E, I, H, generator=g) * 0.05).to(dtype)
    w2 = (torch.randn(E, H, I, generator=g) * 0.05).to(dtype)
    dy = torch.randn(A, H, generator=g).to(dtype)
    return x, w1, w2, w3, dy, torch.tensor(counts, dtype=torch.long)


def _oracle(x, w1, w2, w3, dy, counts):
    """fp32 evaluation with autograd; also returns the SwiGLU intermediates' gradients."""
    xr, w1r, w2r, w3r = (t.float().requires_grad_(True) for t in (x, w1, w2, w3))
    y = O.grouped_swiglu(w1r, w2r, w3r, xr, counts)
    dx, dw1, dw2, dw3 = torch.autograd.grad(y, (xr, w1r, w2r, w3r), dy.float())
    return y.detach(), dx, dw1, dw2, dw3


CASES = [
    # (counts, H, I)   -- ragged, empty experts, single rows, more than one 128-row tile
    ([128, 128, 128, 128], 256, 256),
    ([0, 5, 300, 0, 129, 1, 127, 0], 256, 128),
    ([37] * 16, 128, 384),
    ([0, 0, 0, 700], 384, 256),
    # enough 256-row units per workgroup for the 256x256 tiles, with a reduction of only four k-tiles
    ([8192, 8192], 128, 1536),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,H,I", CASES)
def test_grouped_swiglu_fwd_dgrad_wgrad(dev, dtype, counts, H, I):
    print(f"[case] grouped_swiglu {dtype} counts={counts[:8]} H={H} I={I}", flush=True)
    x, w1, w2, w3, dy, cnt = _make(3, counts, H, I, dtype)
    y_ref, dx_ref, dw1_ref, dw2_ref, dw3_ref = _oracle(x, w1, w2, w3, dy, cnt)
    tol = BF16_TOL if dtype == torch.bfloat16 else F32_TOL
    E = len(counts)
    X, W1, W2, W3, DY = (t.to(dev) for t in (x, w1, w2, w3, dy))
    starts = ops.counts_to_starts(cnt.to(dev))
    y, g, u, h = ops.grouped_swiglu_fwd(X, W1, W2, W3, starts)
    assert y.dtype == dtype and rel_err(y, y_ref) <= tol
    # saved pre-activations are what they claim to be
    if sum(counts) > 0:
        e0 = next(e for e, c in enumerate(counts) if c > 0)
        s0 = int(sum(counts[:e0]))
        g_ref = x[s0:s0 + counts[e0]].float() @ w1[e0].float().t()
        assert rel_err(g[s0:s0 + counts[e0]], g_ref) <= tol
    dx, dg, du = ops.grouped_swiglu_dgrad(DY, W1, W2, W3, g, u, starts)
    assert rel_err(dx, dx_ref) <= tol
    dw1, dw2, dw3 = ops.grouped_swiglu_wgrad(DY, h, dg, du, X, starts, E)
    assert rel_err(dw1, dw1_ref) <= tol and rel_err(dw2, dw2_ref) <= tol and rel_err(dw3, dw3_ref) <= tol
    # every expert on its own scale: its rows of y and d_x, its weight gradients
    for name, got, ref, by_rows in (("y", y, y_ref, True), ("d_x", dx, dx_ref, True), ("d_w1", dw1, dw1_ref, False),
                                    ("d_w2", dw2, dw2_ref, False), ("d_w3", dw3, dw3_ref, False)):
        worst, e = rel_err_by_expert(got, ref, counts, rows=by_rows)
        assert worst <= tol, (name, "expert", e, counts[e], worst)
    for e, c in enumerate(counts):
        if c == 0:  # an expert without rows gets exact zeros, not garbage
            assert float(dw1[e].abs().max()) == 0.0 and float(dw2[e].abs().max()) == 0.0 and float(dw3[e].abs().max()) == 0.0
    # accumulate=True adds a second microbatch on top
    ops.grouped_swiglu_wgrad(DY, h, dg, du, X, starts, E, d_w1=dw1, d_w2=dw2, d_w3=dw3, accumulate=True)
    assert rel_err(dw2, 2 * dw2_ref) <= tol and rel_err(dw1, 2 * dw1_ref) <= tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,H,I", CASES + [([10, 0, 70, 3, 1], 192, 64)])
def test_scaled_backward_matches_combine_bwd_then_dgrad(dev, dtype, counts, H, I):
    """The backward with the weighted combine folded into the d_h GEMM (d_out rows gathered, score
    applied in the epilogue, score gradient from the same accumulator) against the unfused chain
    combine_bwd -> dgrad_dh -> wgrad, and against fp32 autograd through the oracle."""
    print(f"[case] scaled backward {dtype} counts={counts[:8]} H={H} I={I}", flush=True)
    K = 2
    A = int(sum(counts))
    assert A % K == 0
    T, E = A // K, len(counts)
    gen = torch.Generator().manual_seed(11)
    _, w1, w2, w3, _, cnt = _make(5, counts, H, I, dtype)
    perm = torch.randperm(A, generator=gen).to(torch.int32)          # sorted row -> flat (token, k) slot
    tok = perm.long() // K
    x_tok = torch.randn(T, H, generator=gen).to(dtype)
    x_sorted = x_tok[tok]
    scores = torch.rand(T, K, generator=gen) + 0.1
    d_out = torch.randn(T, H, generator=gen).to(dtype)
    tol = BF16_TOL if dtype == torch.bfloat16 else F32_TOL

    XT, XS, W1, W2, W3, PERM, SC, DO = (t.to(dev) for t in (x_tok, x_sorted, w1, w2, w3, perm, scores, d_out))
    starts = ops.counts_to_starts(cnt.to(dev))
    y, g, u, h = ops.grouped_swiglu_fwd(XT, W1, W2, W3, starts, row_map=PERM, row_map_div=K)

    # fp32 reference: out[t] = sum_k s[t,k] * y[row(t,k)]
    xr, w1r, w2r, w3r = (t.float().requires_grad_(True) for t in (x_sorted, w1, w2, w3))
    sr = scores.clone().requires_grad_(True)
    y_ref = O.grouped_swiglu(w1r, w2r, w3r, xr, cnt)
    out_ref = torch.zeros(T, H).index_add(0, tok, y_ref * sr.reshape(-1)[perm.long()].unsqueeze(1))
    dx_ref, dw1_ref, dw2_ref, dw3_ref, ds_ref = torch.autograd.grad(out_ref, (xr, w1r, w2r, w3r, sr), d_out.float())

    d_g, d_u, hs, d_s = ops.grouped_swiglu_dgrad_dh_scaled(DO, PERM, SC, W2, g, u, starts)
    assert d_s.shape == (T, K) and rel_err(d_s, ds_ref) <= tol
    d_xs = ops.grouped_swiglu_dgrad_dx(d_g, d_u, W1, W3, starts)
    assert rel_err(d_xs, dx_ref) <= tol
    dw1, dw2, dw3 = ops.grouped_swiglu_wgrad(DO, hs, d_g, d_u, XT, starts, E, row_map=PERM, row_map_div=K, scaled=True)
    assert rel_err(dw1, dw1_ref) <= tol and rel_err(dw2, dw2_ref) <= tol and rel_err(dw3, dw3_ref) <= tol
    for name, got, ref, by_rows in (("d_x", d_xs, dx_ref, True), ("d_w1", dw1, dw1_ref, False),
                                    ("d_w2", dw2, dw2_ref, False), ("d_w3", dw3, dw3_ref, False)):
        worst, e = rel_err_by_expert(got, ref, counts, rows=by_rows)
        assert worst <= tol, (name, "expert", e, counts[e], worst)

    # the unfused chain on the same inputs
    d_y, d_s2 = ops.combine_bwd(DO, y, PERM, SC)
    d_g2, d_u2 = ops.grouped_swiglu_dgrad_dh(d_y, W2, g, u, starts)
    loose = 2 * tol          # both sides round at different places
    assert rel_err(d_s, d_s2) <= loose and rel_err(d_g, d_g2) <= loose and rel_err(d_u, d_u2) <= loose
    _, dw2_b, _ = ops.grouped_swiglu_wgrad(d_y, h, d_g2, d_u2, XS, starts, E)
    assert rel_err(dw2, dw2_b) <= loose
    for e, c in enumerate(counts):
        if c == 0:
            assert float(dw2[e].abs().max()) == 0.0


def _row_tile_boundary_counts(E):
    """Row counts around the 256- and 128-row block tiles: exact multiples, one above, a few tens
    above, short and empty experts."""
    edge = [256, 257, 287, 288, 289, 255, 1, 0, 544, 545, 320, 33, 32, 31, 512, 513, 543, 800, 300, 270,
            264, 250, 129, 128, 127, 1056, 1057, 16, 272, 260]
    counts = [edge[i % len(edge)] for i in range(E)]
    return counts


def test_row_tiles_at_block_tile_boundaries(dev):
    """Forward and input gradient on a launch with 128 experts whose row counts sit on every side
    of the block tile boundaries, every expert against fp32 matmuls of the same bf16 inputs on the
    device; the rows of an expert's last, partly filled row tile are also compared on their own."""
    E, H, I = 128, 1024, 512
    counts = _row_tile_boundary_counts(E)
    A = sum(counts)
    print(f"[case] row tile boundaries E={E} A={A} H={H} I={I}", flush=True)
    g_ = torch.Generator().manual_seed(21)
    x = torch.randn(A, H, generator=g_).to(torch.bfloat16).to(dev)
    dy = torch.randn(A, H, generator=g_).to(torch.bfloat16).to(dev)
    w1 = (torch.randn(E, I, H, generator=g_) * 0.05).to(torch.bfloat16).to(dev)
    w3 = (torch.randn(E, I, H, generator=g_) * 0.05).to(torch.bfloat16).to(dev)
    w2 = (torch.randn(E, H, I, generator=g_) * 0.05).to(torch.bfloat16).to(dev)
    starts = ops.counts_to_starts(torch.tensor(counts, dtype=torch.long, device=dev))
    y, g, u, h = ops.grouped_swiglu_fwd(x, w1, w2, w3, starts)
    dx, dg, du = ops.grouped_swiglu_dgrad(dy, w1, w2, w3, g, u, starts)
    torch.cuda.synchronize()
    s = 0
    for e, c in enumerate(counts):
        if c == 0:
            continue
        xe = x[s:s + c].float().requires_grad_(True)
        ge = xe @ w1[e].float().t()
        ue = xe @ w3[e].float().t()
        he = torch.nn.functional.silu(ge) * ue
        ye = he @ w2[e].float().t()
        (dxe,) = torch.autograd.grad(ye, xe, dy[s:s + c].float())
        for name, got, ref in (("g", g, ge), ("u", u, ue), ("h", h, he), ("y", y, ye), ("dx", dx, dxe)):
            assert rel_err(got[s:s + c], ref) <= BF16_TOL, (name, e, c, rel_err(got[s:s + c], ref))
            t0 = (c - 1) // 256 * 256      # first row of the expert's last 256-row group
            if t0 > 0:
                assert rel_err(got[s + t0:s + c], ref[t0:]) <= BF16_TOL, (name, "last row tile", e, c)
        s += c


T_CASES = [
    # ragged around the 8-row padding and the 32-row k-tile, empty experts, one long expert
    ([0, 1, 7, 8, 9, 31, 32, 33, 0, 300, 64, 255], 256, 256),
    ([700, 0, 0, 2], 512, 256),
    ([256] * 6, 256, 512),
    ([4096, 3000, 1000, 96], 256, 1536),
    # more weight-gradient tiles than workgroups, so a workgroup walks several units: units handed
    # out from the counters (long experts) with experts of 0, 1 and 33 rows between long ones ...
    ([3000, 0, 1, 2500, 33, 0, 700, 600, 500, 400, 300, 64, 32, 70, 100, 96], 1024, 768),
    # ... and the static hand-out with many short experts (reductions of 0 to 3 k-tiles back to back)
    ([0, 1, 33, 64, 5, 96, 31, 70, 0, 0, 65, 2] * 24, 256, 256),
    # enough 256-row units per workgroup for the 256x256x32 tiles (the d_x GEMM then reads 32-deep
    # k-tiles of the transposed copies), with ragged last row tiles
    ([8192, 8000, 8300, 7777, 8192, 8448, 8193, 8190], 1024, 256),
]


@pytest.mark.parametrize("counts,H,I", T_CASES)
def test_transposed_backward_pair_matches_the_plain_pair(dev, counts, H, I):
    """pk_grouped_swiglu_dgrad_dh_scaled_t / pk_grouped_swiglu_wgrad_scaled_t (one operand of every
    weight-gradient GEMM K-contiguous, persistent workgroups) against
    pk_grouped_swiglu_dgrad_dh_scaled / pk_grouped_swiglu_wgrad_scaled on the same inputs, against
    fp32 autograd through the oracle, and the layout of the transposed copies."""
    print(f"[case] transposed backward counts={counts} H={H} I={I}", flush=True)
    K = 2
    A = int(sum(counts))
    if A % K:
        counts = list(counts); counts[-1] += 1; A += 1
    T, E = A // K, len(counts)
    dtype = torch.bfloat16
    gen = torch.Generator().manual_seed(21)
    _, w1, w2, w3, _, cnt = _make(6, counts, H, I, dtype)
    perm = torch.randperm(A, generator=gen).to(torch.int32)
    tok = perm.long() // K
    x_tok = torch.randn(T, H, generator=gen).to(dtype)
    scores = torch.rand(T, K, generator=gen) + 0.1
    d_out = torch.randn(T, H, generator=gen).to(dtype)
    XT, W1, W2, W3, PERM, SC, DO = (t.to(dev) for t in (x_tok, w1, w2, w3, perm, scores, d_out))
    starts = ops.counts_to_starts(cnt.to(dev))
    ldt = ops.transposed_ld(A, H, I, E, dtype)
    assert ldt >= ((A + 63) // 64 + E) * 64 and ldt % 256 == 128
    assert ops.transposed_ld(A, H + 128, I, E, dtype) == 0 and ops.transposed_ld(A, H, I, E, torch.float32) == 0
    _, g, u, _ = ops.grouped_swiglu_fwd(XT, W1, W2, W3, starts, row_map=PERM, row_map_div=K)

    d_g, d_u, hs, d_s = ops.grouped_swiglu_dgrad_dh_scaled(DO, PERM, SC, W2, g, u, starts)
    # poison what the transposed call allocates next, so untouched pad columns would show as NaN
    junk = torch.full((3 * I * ldt + 16,), float("nan"), dtype=dtype, device=dev)
    del junk
    d_g2, d_u2, d_gT, d_uT, hsT, d_s2 = ops.grouped_swiglu_dgrad_dh_scaled_t(DO, PERM, SC, W2, g, u, starts)
    assert torch.equal(d_g, d_g2) and torch.equal(d_u, d_u2) and torch.equal(d_s, d_s2)
    st = starts.cpu().tolist()
    for e, c in enumerate(counts):
        p0 = (st[e] // 64) * 64 + 64 * e
        c32 = (c + 31) // 32 * 32      # zeros up to the end of the expert's last block of 32 rows
        for full, tr in ((d_g, d_gT), (d_u, d_uT), (hs, hsT)):
            # [ldt/32, I, 32] -> [I, ldt]: column i, padded row r
            blk = tr.permute(1, 0, 2).reshape(I, ldt)[:, p0:p0 + c32]
            assert torch.equal(blk[:, :c], full[st[e]:st[e] + c].t()), f"expert {e}"
            assert torch.count_nonzero(blk[:, c:]).item() == 0, f"pad columns of expert {e}"

    # without the row-major outputs: the same transposed copies, and the d_x GEMM that reads its A
    # operand from them gives the d_x of the row-major pair bit for bit (same products, same order)
    none_g, none_u, d_gT3, d_uT3, hsT3, d_s3 = ops.grouped_swiglu_dgrad_dh_scaled_t(DO, PERM, SC, W2, g, u, starts, row_major=False)
    assert none_g is None and none_u is None and torch.equal(d_s3, d_s)
    for e, c in enumerate(counts):
        p0 = (st[e] // 64) * 64 + 64 * e
        c32 = (c + 31) // 32 * 32
        for a, b in ((d_gT, d_gT3), (d_uT, d_uT3), (hsT, hsT3)):
            assert torch.equal(a.permute(1, 0, 2).reshape(I, ldt)[:, p0:p0 + c32], b.permute(1, 0, 2).reshape(I, ldt)[:, p0:p0 + c32])
    d_x_rows = ops.grouped_swiglu_dgrad_dx(d_g, d_u, W1, W3, starts)
    d_x_blocks = ops.grouped_swiglu_dgrad_dx_t(d_gT3, d_uT3, W1, W3, starts, A)
    assert torch.equal(d_x_rows, d_x_blocks)

    ref = ops.grouped_swiglu_wgrad(DO, hs, d_g, d_u, XT, starts, E, row_map=PERM, row_map_div=K, scaled=True)
    order = torch.argsort(cnt, descending=True, stable=True).to(torch.int32).to(dev)
    for eo in (None, order):
        got = ops.grouped_swiglu_wgrad_scaled_t(DO, hsT, d_gT, d_uT, XT, starts, E, row_map=PERM, row_map_div=K, expert_order=eo)
        for a, b, name in zip(got, ref, ("d_w1", "d_w2", "d_w3")):
            # same products, same fp32 summation order over the rows: equal up to the last bf16 bit
            assert rel_err(a, b) <= 2.0 ** -7, name
            for e, c in enumerate(counts):
                if c == 0:
                    assert float(a[e].abs().max()) == 0.0
    # fp32 reference through the oracle
    x_sorted = x_tok[tok]
    xr, w1r, w2r, w3r = (t.float().requires_grad_(True) for t in (x_sorted, w1, w2, w3))
    y_ref = O.grouped_swiglu(w1r, w2r, w3r, xr, cnt)
    out_ref = torch.zeros(T, H).index_add(0, tok, y_ref * scores.reshape(-1)[perm.long()].unsqueeze(1))
    dw_ref = torch.autograd.grad(out_ref, (w1r, w2r, w3r), d_out.float())
    for a, b, name in zip(got, (dw_ref[0], dw_ref[1], dw_ref[2]), ("d_w1", "d_w2", "d_w3")):
        assert rel_err(a, b) <= BF16_TOL
        # every expert on its own scale: a one-row expert's gradient is a few per cent of the
        # largest one and would hide behind the whole-tensor maximum
        worst, e = rel_err_by_expert(a, b, counts, rows=False)
        assert worst <= BF16_TOL, (name, "expert", e, counts[e], worst)
    # accumulate: adds to what is there, twice gives 2x (+ one rounding)
    acc = [t.clone() for t in got]
    ops.grouped_swiglu_wgrad_scaled_t(DO, hsT, d_gT, d_uT, XT, starts, E, row_map=PERM, row_map_div=K,
                                      d_w1=acc[0], d_w2=acc[1], d_w3=acc[2], accumulate=True, expert_order=order)
    for a, b in zip(acc, got):
        assert rel_err(a, 2 * b.float()) <= 2.0 ** -7
    # argument checks: a row length below the query's, and a shape without the path
    with pytest.raises(RuntimeError):
        _lib_call_short_ld(DO, hsT, d_gT, d_uT, XT, PERM, starts, E, H, I, A, K, ldt - 64)


def _lib_call_short_ld(DO, hsT, d_gT, d_uT, XT, PERM, starts, E, H, I, A, K, ldt):
    from piper_amd._lib import call, current_stream, dtype_code, ptr
    w = torch.empty((E, I, H), dtype=DO.dtype, device=DO.device)
    call("pk_grouped_swiglu_wgrad_scaled_t", ptr(DO), ptr(hsT), ptr(d_gT), ptr(d_uT), ldt, ptr(XT), ptr(PERM), K, ptr(starts),
         ptr(None), ptr(w), ptr(None), ptr(None), 0, A, H, I, E, dtype_code(DO.dtype), current_stream(DO.device))


def test_mfma_path_agrees_with_fma_path(dev):
    """bf16 shapes outside the MFMA tiling (H or I not a multiple of 128) run on the FMA kernel."""
    print("[case] bf16 fallback shapes", flush=True)
    counts = [10, 0, 70, 3]
    x, w1, w2, w3, dy, cnt = _make(4, counts, 192, 64, torch.bfloat16)
    y_ref, dx_ref, dw1_ref, dw2_ref, dw3_ref = _oracle(x, w1, w2, w3, dy, cnt)
    X, W1, W2, W3, DY = (t.to(dev) for t in (x, w1, w2, w3, dy))
    starts = ops.counts_to_starts(cnt.to(dev))
    y, g, u, h = ops.grouped_swiglu_fwd(X, W1, W2, W3, starts)
    dx, dg, du = ops.grouped_swiglu_dgrad(DY, W1, W2, W3, g, u, starts)
    dw1, dw2, dw3 = ops.grouped_swiglu_wgrad(DY, h, dg, du, X, starts, 4)
    for a, b in ((y, y_ref), (dx, dx_ref), (dw1, dw1_ref), (dw2, dw2_ref), (dw3, dw3_ref)):
        assert rel_err(a, b) <= BF16_TOL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_fused_permute_operand_load(dev, dtype):
    """row_map = perm, div = K: reading x[perm[p] // K] inside the GEMM equals permute then GEMM."""
    print(f"[case] fused permute {dtype}", flush=True)
    T, H, I, E, K = 300, 256, 128, 8, 2
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(T, E, generator=g)
    logits[:, 3] = -50.0
    _, idx = O.route_topk(logits, K, True)
    counts, starts_ref, perm, inv = O.sort_by_expert(idx, E)
    x = torch.randn(T, H, generator=g).to(dtype)
    _, w1, w2, w3, _, _ = _make(6, [1] * E, H, I, dtype)
    X, W1, W2, W3 = (t.to(dev) for t in (x, w1, w2, w3))
    starts = starts_ref.int().to(dev)
    P = perm.int().to(dev)
    routed = ops.permute_fwd(X, P, K)
    y_a, g_a, u_a, h_a = ops.grouped_swiglu_fwd(routed, W1, W2, W3, starts)
    y_b, g_b, u_b, h_b = ops.grouped_swiglu_fwd(X, W1, W2, W3, starts, row_map=P, row_map_div=K)
    assert torch.equal(y_a, y_b) and torch.equal(g_a, g_b) and torch.equal(h_a, h_b)
    dy = torch.randn(T * K, H, generator=g).to(dtype).to(dev)
    dx, dg, du = ops.grouped_swiglu_dgrad(dy, W1, W2, W3, g_a, u_a, starts)
    wa = ops.grouped_swiglu_wgrad(dy, h_a, dg, du, routed, starts, E)
    wb = ops.grouped_swiglu_wgrad(dy, h_a, dg, du, X, starts, E, row_map=P, row_map_div=K)
    for a, b in zip(wa, wb):
        assert torch.equal(a, b)


@pytest.mark.parametrize("counts_dtype", [torch.int64, torch.int32])
def test_reference_operator_bmm_experts(dev, counts_dtype):
    """torch.ops.piper_artifact.bmm_experts(w1, w2, w3, x, num_tokens_per_expert) with autograd:
    the reference's operator boundary (qwen3_bmm_experts_patch.py:63-87)."""
    print("[case] piper_artifact::bmm_experts", flush=True)
    counts = [60, 0, 200, 4]
    x, w1, w2, w3, dy, cnt = _make(8, counts, 256, 128, torch.bfloat16)
    y_ref, dx_ref, dw1_ref, dw2_ref, dw3_ref = _oracle(x, w1, w2, w3, dy, cnt)
    F_.register_reference_op()
    X, W1, W2, W3 = (t.to(dev).requires_grad_(True) for t in (x, w1, w2, w3))
    y = torch.ops.piper_artifact.bmm_experts(W1, W2, W3, X, cnt.to(counts_dtype).to(dev))
    assert y.shape == x.shape and rel_err(y, y_ref) <= BF16_TOL
    y.backward(dy.to(dev))
    assert rel_err(X.grad, dx_ref) <= BF16_TOL
    assert rel_err(W1.grad, dw1_ref) <= BF16_TOL and rel_err(W2.grad, dw2_ref) <= BF16_TOL and rel_err(W3.grad, dw3_ref) <= BF16_TOL
    with torch.no_grad():
        y2 = torch.ops.piper_artifact.bmm_experts(W1, W2, W3, X, cnt.to(counts_dtype).to(dev))
    assert torch.equal(y2, y.detach())
    meta = torch.ops.piper_artifact.bmm_experts(*(t.detach().to("meta") for t in (W1, W2, W3, X)), cnt.to("meta"))
    assert meta.shape == x.shape and meta.is_meta


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_bmm_experts_rows_past_the_last_expert_are_zero(dev, dtype):
    """x has more rows than sum(num_tokens_per_expert): the reference returns zeros there
    (`out = x.new_zeros`, qwen3_bmm_experts_patch.py:43) and no gradient flows into them.  Checked
    against the oracle's restatement of the padded-bmm algorithm."""
    print(f"[case] bmm_experts with unowned rows {dtype}", flush=True)
    counts = [40, 0, 130, 5]
    extra = 37
    x, w1, w2, w3, dy, cnt = _make(11, counts, 256, 128, dtype)
    g = torch.Generator().manual_seed(12)
    x = torch.cat([x, torch.randn(extra, x.shape[1], generator=g).to(dtype)])
    dy = torch.cat([dy, torch.randn(extra, dy.shape[1], generator=g).to(dtype)])
    leaves = [t.detach().clone().float().requires_grad_(True) for t in (w1, w2, w3, x)]
    y_ref = O.padded_bmm_experts(*leaves, cnt)
    y_ref.backward(dy.float())
    assert torch.count_nonzero(y_ref[sum(counts):]) == 0 and torch.count_nonzero(leaves[3].grad[sum(counts):]) == 0
    F_.register_reference_op()
    W1, W2, W3, X = (t.to(dev).requires_grad_(True) for t in (w1, w2, w3, x))
    # poison the allocator's free blocks so that rows the kernels skip would show
    junk = torch.full((x.shape[0] * 4, x.shape[1]), float("nan"), device=dev, dtype=dtype)
    del junk
    y = torch.ops.piper_artifact.bmm_experts(W1, W2, W3, X, cnt.to(dev))
    tol = BF16_TOL if dtype == torch.bfloat16 else F32_TOL
    assert torch.count_nonzero(y[sum(counts):]).item() == 0
    assert rel_err(y, y_ref) <= tol
    y.backward(dy.to(dev))
    assert torch.count_nonzero(X.grad[sum(counts):]).item() == 0
    assert rel_err(X.grad, leaves[3].grad) <= tol
    for got, ref in zip((W1, W2, W3), leaves[:3]):
        assert rel_err(got.grad, ref.grad) <= tol
    with torch.no_grad():
        assert torch.count_nonzero(torch.ops.piper_artifact.bmm_experts(W1, W2, W3, X, cnt.to(dev))[sum(counts):]).item() == 0


def test_argument_errors(dev):
    z = torch.zeros(4, 8, device=dev, dtype=torch.bfloat16)
    w = torch.zeros(2, 16, 8, device=dev, dtype=torch.bfloat16)
    w2 = torch.zeros(2, 8, 16, device=dev, dtype=torch.bfloat16)
    starts = torch.tensor([0, 2, 4], dtype=torch.int32, device=dev)
    with pytest.raises(ValueError):
        ops.grouped_swiglu_fwd(z, w, w, w, starts)             # w2 has the wrong shape
    with pytest.raises(ValueError):
        ops.grouped_swiglu_fwd(z.float(), w, w2, w, starts)    # dtype mismatch


def test_reference_operator_under_dynamo_fullgraph(dev):
    """The op traced by Dynamo with fullgraph=True (src/compile.py:273) and run by the eager
    backend gives the same forward and gradients as the direct call."""
    counts = [5, 0, 130, 61]
    x, w1, w2, w3, dy, cnt = _make(9, counts, 256, 128, torch.bfloat16)
    X, W1, W2, W3, DY, CNT = (t.to(dev) for t in (x, w1, w2, w3, dy, cnt))

    def region(w1, w2, w3, x, c):
        return F_.bmm_experts(w1, w2, w3, x, c)

    def run(fn):
        leaves = [t.clone().requires_grad_(True) for t in (W1, W2, W3, X)]
        out = fn(*leaves, CNT)
        grads = torch.autograd.grad(out, leaves, DY)
        return out, grads

    torch._dynamo.reset()
    o1, g1 = run(region)
    o2, g2 = run(torch.compile(region, backend="eager", fullgraph=True))
    assert torch.equal(o1, o2)
    for a, b in zip(g1, g2):
        assert torch.equal(a, b)


def test_scaled_backward_argument_errors_and_empty_input(dev):
    """Status codes of the C entry point itself: nothing is launched for a bad call."""
    from piper_amd import _lib
    from piper_amd._lib import PK_BF16, current_stream, ptr
    lib = _lib.load()
    E, H, I, T, K = 2, 256, 128, 16, 2
    A = T * K
    bf = dict(device=dev, dtype=torch.bfloat16)
    d_out, w2 = torch.zeros(T, H, **bf), torch.zeros(E, H, I, **bf)
    g, u, dg, du, hs = (torch.zeros(A, I, **bf) for _ in range(5))
    perm = torch.arange(A, dtype=torch.int32, device=dev)
    sc = torch.ones(T, K, device=dev)
    ds = torch.zeros(T, K, device=dev)
    starts = torch.tensor([0, A // 2, A], dtype=torch.int32, device=dev)
    need = int(lib.pk_grouped_swiglu_dgrad_dh_scaled_workspace_bytes(A, I))
    assert need == (I // 64) * A * 4
    ws = torch.zeros(need // 4, device=dev)
    s = current_stream(dev)

    def call(ws_ptr, ws_bytes, rows=A, row_map=ptr(perm), div=K):
        return lib.pk_grouped_swiglu_dgrad_dh_scaled(ptr(d_out), row_map, div, ptr(sc), ptr(w2), ptr(g), ptr(u), ptr(starts),
                                                     ptr(dg), ptr(du), ptr(hs), ptr(ds), ws_ptr, ws_bytes, rows, H, I, E,
                                                     PK_BF16, s)
    assert call(ptr(ws), need) == 0
    assert call(ptr(ws), need - 4) == -4          # PK_ERR_WORKSPACE
    assert call(None, 0) == -4
    assert call(ptr(ws), need, row_map=None) == -1     # PK_ERR_ARG: the gather map is not optional here
    assert call(ptr(ws), need, div=0) == -1
    assert call(None, 0, rows=0) == 0                  # no rows: nothing to do, nothing required
    assert lib.pk_grouped_swiglu_dgrad_dh_scaled_workspace_bytes(-1, I) == -1
    torch.cuda.synchronize()


def test_grouped_gemms_replay_in_a_hip_graph(dev):
    """The persistent kernels take their work units from counters that the last workgroup of a
    launch resets: a captured graph must give the eager result on every replay, also with new
    input values and with eager launches in between."""
    counts = [300, 0, 513, 77, 128, 1, 260, 5]
    H, I = 256, 256
    x, w1, w2, w3, dy, cnt = _make(7, counts, H, I, torch.bfloat16)
    X, W1, W2, W3, DY = (t.to(dev) for t in (x, w1, w2, w3, dy))
    starts = ops.counts_to_starts(cnt.to(dev))
    E = len(counts)

    def run(xin, dyin):
        y, g, u, h = ops.grouped_swiglu_fwd(xin, W1, W2, W3, starts)
        dx, dg, du = ops.grouped_swiglu_dgrad(dyin, W1, W2, W3, g, u, starts)
        dw1, dw2, dw3 = ops.grouped_swiglu_wgrad(dyin, h, dg, du, xin, starts, E)
        return y, dx, dw1, dw2, dw3

    xs, dys = X.clone(), DY.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run(xs, dys)                       # warm-up outside the capture
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = run(xs, dys)
    for rep in range(4):
        scale = 1.0 + 0.25 * rep
        xs.copy_(X * scale)
        dys.copy_(DY * (2.0 - 0.25 * rep))
        graph.replay()
        torch.cuda.synchronize()
        want = run(xs.clone(), dys.clone())            # eager, between the replays
        torch.cuda.synchronize()
        for got, ref, name in zip(outs, want, ("y", "dx", "dw1", "dw2", "dw3")):
            assert torch.equal(got, ref), f"replay {rep}: {name}"


TILE_CASES = [
    # (counts, H, I): rows on both sides of the 64-row tiles, empty experts, widths that leave a remainder in
    # the 64-wide tiles and in the k-tiles (32 fp32 / 64 bf16), down to a single 16-byte piece
    ([0, 1, 63, 64, 65, 127, 128, 129, 0], 72, 40),
    ([3, 2], 8, 8),
    ([70, 0, 33], 200, 1000),
    # enough rows for the 128 x 128 tiles in every product
    ([3000, 1, 4000, 200, 0, 2500], 1032, 520),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,H,I", TILE_CASES)
def test_widths_without_a_multiple_of_the_wide_tiles(dev, dtype, counts, H, I):
    """tile_gemm.h (fp32, and bf16 widths that are no multiple of 128) against float64 matmuls of the same
    inputs: x gathered through a row map, accumulation into existing gradients, exact zeros for an
    expert without rows.  fp32 sums of n products are within n * 2^-24 of the sum of magnitudes, far
    below F32_TOL of the largest result; bf16 as everywhere (BF16_TOL)."""
    print(f"[case] tile gemm {dtype} E={len(counts)} A={sum(counts)} H={H} I={I}", flush=True)
    x, w1, w2, w3, dy, cnt = (t.to(dev) for t in _make(31, counts, H, I, dtype))
    E, A = len(counts), x.shape[0]
    tol = BF16_TOL if dtype == torch.bfloat16 else F32_TOL
    order = torch.randperm(A, generator=torch.Generator().manual_seed(1)).to(dev)
    x_at = torch.empty_like(x)
    x_at[order] = x                      # row p of the sorted operand is x_at[order[p]]
    rows = order.to(torch.int32)
    starts = ops.counts_to_starts(cnt)
    y, g, u, h = ops.grouped_swiglu_fwd(x_at, w1, w2, w3, starts, row_map=rows, row_map_div=1)
    dx, dg, du = ops.grouped_swiglu_dgrad(dy, w1, w2, w3, g, u, starts)
    dw1, dw2, dw3 = ops.grouped_swiglu_wgrad(dy, h, dg, du, x_at, starts, E, row_map=rows, row_map_div=1)
    acc = [t.clone() for t in (dw1, dw2, dw3)]
    ops.grouped_swiglu_wgrad(dy, h, dg, du, x_at, starts, E, row_map=rows, row_map_div=1, d_w1=acc[0], d_w2=acc[1], d_w3=acc[2],
                             accumulate=True)
    torch.cuda.synchronize()
    s = 0
    for e, c in enumerate(counts):
        if c == 0:
            assert all(float(t[e].abs().max()) == 0.0 for t in (dw1, dw2, dw3, *acc))
            continue
        leaves = [t.double().requires_grad_(True) for t in (x[s:s + c], w1[e], w2[e], w3[e])]
        xe, a1, a2, a3 = leaves
        ge, ue = xe @ a1.t(), xe @ a3.t()
        he = torch.nn.functional.silu(ge) * ue
        ye = he @ a2.t()
        dxe, d1, d2, d3 = torch.autograd.grad(ye, leaves, dy[s:s + c].double())
        for name, got, ref in (("g", g[s:s + c], ge), ("u", u[s:s + c], ue), ("h", h[s:s + c], he), ("y", y[s:s + c], ye),
                               ("dx", dx[s:s + c], dxe), ("dw1", dw1[e], d1), ("dw2", dw2[e], d2), ("dw3", dw3[e], d3),
                               ("dw1 added", acc[0][e], 2 * d1), ("dw2 added", acc[1][e], 2 * d2), ("dw3 added", acc[2][e], 2 * d3)):
            assert rel_err(got, ref) <= tol, (name, e, c, rel_err(got, ref))
        s += c


FP32_TILE_CASES = [
    # (counts, H, I), with the 64 x 64 tiles that gate/up and d_h | down and d_x would have:
    # 84 | 96: 32 x 32 tiles
    ([0, 1, 31, 32, 33, 63, 64, 65, 100, 131], 456, 424),
    # 112 | 128: 64 x 32
    ([0, 1, 31, 32, 33, 63, 64, 65, 101, 200], 504, 424),
    # few rows an expert: 290 | 348, 32 x 64 tiles, experts with more than one of them
    ([0, 1, 16, 15, 3, 7, 8, 9] * 5 + [0, 1, 2, 33, 3, 7, 60, 1], 712, 584),
    # 31 rows: 527, 32 x 64 in d_h only
    ([31] * 32, 392, 1032),
    # 343, 64 x 32 with a split reduction in all but gate/up
    ([100, 99, 101, 64, 136, 100] * 4, 392, 392),
]


@pytest.mark.parametrize("K", [1, 2])
@pytest.mark.parametrize("counts,H,I", FP32_TILE_CASES)
def test_fp32_tiles_by_their_number(dev, counts, H, I, K):
    """The tiles that launch_ragged_m picks in fp32 by their number and the rows an expert, forward and region backward, for
    calls that keep the order of their sums (one expert per token) and others, against float64 matmuls: sums of
    n products are within n * 2^-24 of the sum of magnitudes in any order, far below F32_TOL."""
    from piper_amd._lib import call, current_stream, dtype_code, ptr
    from piper_amd import _lib
    import ctypes
    counts = list(counts)
    counts[-1] += sum(counts) % 2
    print(f"[case] fp32 tiles A={sum(counts)} E={len(counts)} H={H} I={I} K={K}", flush=True)
    A, E = sum(counts), len(counts)
    x, w1, w2, w3, d_out, cnt = (t.to(dev) for t in _make(47, counts, H, I, torch.float32))
    x, d_out = x[:A // K], d_out[:A // K]
    gen = torch.Generator().manual_seed(6)
    perm = torch.randperm(A, generator=gen).to(torch.int32).to(dev)
    scores = (torch.rand(A, generator=gen) + 0.1).to(dev)
    starts = ops.counts_to_starts(cnt)
    y, g, u, h = ops.grouped_swiglu_fwd(x, w1, w2, w3, starts, row_map=perm, row_map_div=K)
    dg, du, hs = (torch.full_like(g, float("nan")) for _ in range(3))
    ds = torch.zeros(A, device=dev)
    ws = torch.full((int(_lib.load().pk_region_dgrad_dh_workspace_bytes(A, I)) // 4,), float("nan"), device=dev)
    n_part = ctypes.c_int64(-1)
    call("pk_region_dgrad_dh", ptr(d_out), ptr(perm), K, ptr(scores), ptr(w2), ptr(g), ptr(u), ptr(starts), ptr(dg), ptr(du), ptr(hs), ptr(ds),
         ctypes.addressof(n_part), ptr(ws), ws.numel() * 4, A, H, I, E, dtype_code(torch.float32), current_stream(dev))
    ds = ws[:n_part.value * A].view(n_part.value, A).double().sum(0)
    dx = torch.full((A, H), float("nan"), device=dev)
    call("pk_region_dgrad_dx_any_order" if K > 1 else "pk_region_dgrad_dx", ptr(dg), ptr(du), ptr(w1), ptr(w3), ptr(starts), ptr(dx), A, H, I, E,
         dtype_code(torch.float32), current_stream(dev))
    rows = (perm.long() // K)
    s = 0
    for e, c in enumerate(counts):
        if c == 0:
            continue
        r = slice(s, s + c)
        s += c
        xe, de, sc = x[rows[r]].double(), d_out[rows[r]].double(), scores[perm.long()[r]].double()[:, None]
        ge, ue = xe @ w1[e].double().t(), xe @ w3[e].double().t()
        sg = torch.sigmoid(ge)
        he, dh = ge * sg * ue, de @ w2[e].double()
        dge, due = sc * dh * ue * (sg * (1 + ge * (1 - sg))), sc * dh * (ge * sg)
        for name, got, ref in (("g", g[r], ge), ("u", u[r], ue), ("h", h[r], he), ("y", y[r], he @ w2[e].double().t()), ("dg", dg[r], dge),
                               ("du", du[r], due), ("hs", hs[r], sc * he),
                               ("dx", dx[r], dge @ w1[e].double() + due @ w3[e].double())):
            assert rel_err(got, ref) <= F32_TOL, (name, e, c, rel_err(got, ref))
        # a sum of I products that cancel: judged, as the bound is, by the sum of their magnitudes
        assert ((ds[r] - (dh * he).sum(1)).abs() <= F32_TOL * (dh * he).abs().sum(1)).all(), ("ds", e, c)


SKINNY_CASES = [
    # (counts, H, I): below, at and above the 16- and 32-row units, reductions of less than one step (64)
    # per wave and with a remainder, widths with a partly filled column tile, empty experts
    ([1], 64, 16),
    ([0, 1, 0, 2, 15, 16, 17, 0, 3], 200, 72),
    ([33, 1, 31, 32, 40, 0], 520, 264),
    ([9] * 12, 2048, 768),
]


@pytest.mark.parametrize("counts,H,I", SKINNY_CASES)
def test_experts_with_few_rows(dev, counts, H, I):
    """The weight-streaming forward (skinny_gemm.h) against float64 matmuls of the same bf16 inputs, with
    and without a row map and with g and u left out: the same bits every time."""
    from piper_amd import _lib
    print(f"[case] skinny counts={counts[:9]} H={H} I={I}", flush=True)
    x, w1, w2, w3, _, cnt = (t.to(dev) for t in _make(37, counts, H, I, torch.bfloat16))
    A = x.shape[0]
    starts = ops.counts_to_starts(cnt)
    y, g, u, h = ops.grouped_swiglu_fwd(x, w1, w2, w3, starts)
    order = torch.randperm(A, generator=torch.Generator().manual_seed(2)).to(dev)
    x_at = torch.empty_like(x)
    x_at[order] = x
    y2, g2, u2, h2 = ops.grouped_swiglu_fwd(x_at, w1, w2, w3, starts, row_map=order.to(torch.int32), row_map_div=1)
    assert torch.equal(y, y2) and torch.equal(g, g2) and torch.equal(u, u2) and torch.equal(h, h2)
    h3, y3 = torch.empty_like(h), torch.empty_like(y)
    rc = _lib.load().pk_grouped_swiglu_fwd(x.data_ptr(), None, 1, w1.data_ptr(), w2.data_ptr(), w3.data_ptr(), starts.data_ptr(), None, None,
                                           h3.data_ptr(), y3.data_ptr(), A, H, I, len(counts), _lib.PK_BF16, _lib.current_stream(dev))
    assert rc == 0 and torch.equal(h, h3) and torch.equal(y, y3)
    s = 0
    for e, c in enumerate(counts):
        if c == 0:
            continue
        xe = x[s:s + c].double()
        ge, ue = xe @ w1[e].double().t(), xe @ w3[e].double().t()
        he = torch.nn.functional.silu(ge) * ue
        for name, got, ref in (("g", g, ge), ("u", u, ue), ("h", h, he), ("y", y, he @ w2[e].double().t())):
            assert rel_err(got[s:s + c], ref) <= BF16_TOL, (name, e, c)
        s += c


@pytest.mark.parametrize("experts,A", [(128, 512), (128, 513), (64, 512), (64, 513)])
def test_experts_with_few_rows_and_popular_experts(dev, experts, A):
    """Both sides of the lines between the weight-streaming forward and the wide tiles (4 rows an expert at
    three wide units per CU, 8 below), with counts that fall as 1 / rank down to none."""
    weights = 1.0 / torch.arange(1, experts + 1).double()
    counts = (weights / weights.sum() * A).long()
    counts[0] += A - int(counts.sum())
    counts[experts // 2] += int(counts[-1])
    counts[-1] = 0
    test_experts_with_few_rows(dev, counts.tolist(), 256, 768)


@pytest.mark.parametrize("H,I,E,A", [(512, 768, 128, 9599), (512, 768, 128, 14336), (512, 768, 128, 24703), (2048, 128, 128, 5247),
                                     (1024, 512, 64, 28799), (1024, 640, 64, 1663)])
def test_one_more_row_takes_other_kernels_to_the_same_bits(dev, H, I, E, A):
    """128 experts of 512 x 768: from these sizes on one more row takes gate/up (9,600 rows), d_x (14,337) and down (24,704)
    from the tiles to the persistent kernels, with 2048 x 128 d_x (5,248), with 64 of 1024 x 512 down (28,800); with 64 of
    1024 x 640 d_x goes from 128 x 128 to 64 x 64 tiles (1,664).  Tiles that do not
    split the reduction add a product's terms in the persistent kernels' order and, from a quarter above one round of gate/up
    units on, form h with their sigmoid, so at these crossings what the other rows get does not change; values against
    float64 for a few experts."""
    print(f"[case] one more row after {A}", flush=True)
    x, w1, w2, w3, dy, cnt = (t.to(dev) for t in _make(43, [A // E] * (E - 1) + [A + 1 - A // E * (E - 1)], H, I, torch.bfloat16))
    got = []
    for n in (A, A + 1):
        c = cnt.clone()
        c[-1] -= A + 1 - n
        starts = ops.counts_to_starts(c)
        y, g, u, h = ops.grouped_swiglu_fwd(x[:n], w1, w2, w3, starts)
        got.append((y, g, u, h) + tuple(ops.grouped_swiglu_dgrad(dy[:n], w1, w2, w3, g, u, starts)))
    for few, more in zip(*got):
        assert torch.equal(few, more[:A])
    y, g, u, h = got[0][:4]
    s = 0
    for e in range(3):
        r = slice(s, s + A // E)
        ge, ue = x[r].double() @ w1[e].double().t(), x[r].double() @ w3[e].double().t()
        he = torch.nn.functional.silu(ge) * ue
        for name, out, ref in (("g", g, ge), ("u", u, ue), ("h", h, he), ("y", y, he @ w2[e].double().t())):
            assert rel_err(out[r], ref) <= BF16_TOL, (name, e)
        s += A // E


@pytest.mark.parametrize("H,I,E,K,T", [(256, 768, 128, 8, 512), (2048, 1024, 4, 2, 80)])
def test_few_rows_an_expert_leave_out_the_transposed_copies(dev, H, I, E, K, T):
    """Up to 32 rows an expert (128 experts, more units of d_h than CUs) or 40 (4 experts) the region's backward runs without the
    transposed copies, with one more token through them: the weight-gradient kernels that were launched say so.  Every
    gradient against float64 on the same experts, on both sides."""
    from piper_amd import _lib
    gen = torch.Generator(device=dev).manual_seed(H + E)
    rand = lambda *shape, scale=1.0: torch.randn(shape, generator=gen, device=dev) * scale
    w1, w3 = (rand(E, I, H, scale=0.05).bfloat16().requires_grad_(True) for _ in range(2))
    w2, w_gate = rand(E, H, I, scale=0.05).bfloat16().requires_grad_(True), rand(E, H, scale=0.05).requires_grad_(True)
    x_all, d_all = rand(T + 1, H).bfloat16(), rand(T + 1, H).bfloat16()
    for tokens in (T, T + 1):
        print(f"[case] {tokens} tokens, {E} experts {H} x {I}", flush=True)
        x, d_out = x_all[:tokens].clone().requires_grad_(True), d_all[:tokens]
        out = F_.expert_region(x, w_gate, None, w1, w2, w3, top_k=K, route_norm=True)
        _lib.timing_enable(True)
        _lib.timing_collect()
        got = torch.autograd.grad(out, (x, w_gate, w1, w2, w3), d_out)
        names = [n for n, _ in _lib.timing_collect()]
        _lib.timing_enable(False)
        assert ("swiglu_wgrad" in names) == (tokens == T) and ("swiglu_wgrad_w13" in names) == (tokens > T), names
        idx = ops.route_topk(ops.gate_logits(x.detach(), w_gate.detach()), K, True)[1].long()
        ref = [t.detach().double().requires_grad_(True) for t in (x, w_gate, w1, w2, w3)]
        xd, gd, w1d, w2d, w3d = ref
        scores = torch.gather(torch.softmax(xd @ gd.t(), 1), 1, idx)
        scores = scores / scores.sum(1, keepdim=True)
        y = torch.zeros_like(xd)
        for e in range(E):
            t, k = (idx == e).nonzero(as_tuple=True)
            h = torch.nn.functional.silu(xd[t] @ w1d[e].t()) * (xd[t] @ w3d[e].t())
            y = y.index_add(0, t, (h @ w2d[e].t()) * scores[t, k][:, None])
        want = torch.autograd.grad(y, ref, d_out.double())
        for name, a, b in zip(("x", "w_gate", "w1", "w2", "w3"), got, want):
            assert rel_err(a, b) <= BF16_TOL, name


def _dx_of_random_gradients(dev, seed, counts, H, I):
    """d_g, d_u, w1, w3 and d_x(n): pk_region_dgrad_dx of the first n rows"""
    from piper_amd import _lib
    gen = torch.Generator(device=dev).manual_seed(seed)
    E, A = len(counts), sum(counts)
    d_g, d_u = (torch.randn((A, I), generator=gen, device=dev).bfloat16() for _ in range(2))
    w1, w3 = ((torch.randn((E, I, H), generator=gen, device=dev) * 0.05).bfloat16() for _ in range(2))
    cnt = torch.tensor(counts, dtype=torch.long, device=dev)

    def d_x(n):
        c = cnt.clone()
        c[-1] -= A - n
        starts = ops.counts_to_starts(c)
        out = torch.empty((n, H), dtype=torch.bfloat16, device=dev)
        _lib.call("pk_region_dgrad_dx", d_g.data_ptr(), d_u.data_ptr(), w1.data_ptr(), w3.data_ptr(), starts.data_ptr(), out.data_ptr(), n, H, I, E,
                  _lib.PK_BF16, _lib.current_stream(dev))
        return out
    return d_g, d_u, w1, w3, d_x


def test_input_gradient_of_every_last_unit(dev):
    """d_x in 256-row units (1,000 rows an expert and more, 8 column tiles: over 512 units) whose last unit holds one to eight
    32-row chunks, full or with a single row: a wave has none to four of them with rows.  Against float64."""
    H, I = 2048, 256
    last = [129, 160, 161, 192, 193, 224, 225, 255, 1, 32, 33, 64, 65, 96, 97, 128]
    counts = [1024 + n for n in last]
    print(f"[case] d_x last units {last}", flush=True)
    d_g, d_u, w1, w3, d_x = _dx_of_random_gradients(dev, 51, counts, H, I)
    got, s = d_x(sum(counts)), 0
    for e, c in enumerate(counts):
        want = d_g[s:s + c].double() @ w1[e].double() + d_u[s:s + c].double() @ w3[e].double()
        assert rel_err(got[s:s + c], want) <= BF16_TOL, (e, c)
        assert rel_err(got[s + 1024:s + c], want[1024:]) <= BF16_TOL, (e, c)      # the last unit by itself
        s += c


def test_input_gradient_on_both_sides_of_the_taller_units(dev):
    """320 rows an expert (64 experts, 2048 x 256) take d_x to 256-row units, one row fewer to 128-row ones: the same sums in the
    same order, so the rows that both calls have get the same bits; values against float64."""
    H, I, E = 2048, 256, 64
    counts = [320 + (-1) ** e * (37 * (e // 2) % 150) for e in range(E)]
    A = sum(counts)
    assert A == 320 * E
    print("[case] d_x at 320 rows an expert", flush=True)
    d_g, d_u, w1, w3, d_x = _dx_of_random_gradients(dev, 53, counts, H, I)
    tall = d_x(A)
    assert torch.equal(d_x(A - 1), tall[:A - 1])
    s = 0
    for e in range(E):
        c = counts[e]
        want = d_g[s:s + c].double() @ w1[e].double() + d_u[s:s + c].double() @ w3[e].double()
        assert rel_err(tall[s:s + c], want) <= BF16_TOL, (e, c)
        s += c


REGION_BACKWARD_CASES = [
    # (counts, H, I): split reductions with every row and column remainder, unsplit 64-row tiles, 128-row
    # tiles, the persistent kernels at widths of 256 and 128 columns, a single row
    ([0, 1, 63, 64, 65, 200, 0, 33], 72, 40),
    ([1], 256, 256),
    ([130, 0, 64, 300] * 8, 256, 512),
    ([1000, 999, 0, 1025, 800, 1100, 900, 1300, 1000], 72, 1000),
    ([2900, 2800, 3000], 128, 1024),
    ([5000, 6000, 5003], 128, 384),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,H,I", REGION_BACKWARD_CASES)
def test_region_input_gradient_by_size(dev, dtype, counts, H, I):
    """pk_region_dgrad_dh (whichever tiles it picks, the score gradient in parts or whole) and
    pk_region_dgrad_dx against float64 matmuls of the same inputs."""
    from piper_amd import _lib
    from piper_amd._lib import call, current_stream, dtype_code, ptr
    import ctypes
    print(f"[case] region input gradient {dtype} counts={counts[:9]} H={H} I={I}", flush=True)
    tol = BF16_TOL if dtype == torch.bfloat16 else F32_TOL
    counts = list(counts) + ([1] if sum(counts) % 2 else [])
    A, E, K = sum(counts), len(counts), 2
    _, w1, w2, w3, _, cnt = (t.to(dev) for t in _make(41, counts, H, I, dtype))
    gen = torch.Generator().manual_seed(5)
    perm = torch.randperm(A, generator=gen).to(torch.int32).to(dev)
    scores = (torch.rand(A // K, K, generator=gen) + 0.1).to(dev)
    d_out = torch.randn(A // K, H, generator=gen).to(dtype).to(dev)
    g, u = (torch.randn(A, I, generator=gen).to(dtype).to(dev) for _ in range(2))
    starts = ops.counts_to_starts(cnt)
    dg, du, hs = (torch.full_like(g, float("nan")) for _ in range(3))
    ds = torch.zeros(A, device=dev)
    ws = torch.full((int(_lib.load().pk_region_dgrad_dh_workspace_bytes(A, I)) // 4,), float("nan"), device=dev)
    n_part = ctypes.c_int64(-1)
    call("pk_region_dgrad_dh", ptr(d_out), ptr(perm), K, ptr(scores), ptr(w2), ptr(g), ptr(u), ptr(starts), ptr(dg), ptr(du), ptr(hs), ptr(ds),
         ctypes.addressof(n_part), ptr(ws), ws.numel() * 4, A, H, I, E, dtype_code(dtype), current_stream(dev))
    n = n_part.value
    assert n in (0, (I + 31) // 32, (I + 63) // 64, (I + 127) // 128)
    if n > 0:
        ds = torch.zeros_like(ds).index_copy(0, perm.long(), ws[:n * A].view(n, A).sum(0))
    dx = torch.full((A, H), float("nan"), dtype=dtype, device=dev)
    call("pk_region_dgrad_dx", ptr(dg), ptr(du), ptr(w1), ptr(w3), ptr(starts), ptr(dx), A, H, I, E, dtype_code(dtype), current_stream(dev))
    dg0, du0 = ops.grouped_swiglu_dgrad_dh(d_out[perm.long() // K].contiguous(), w2, g, u, starts)      # without the scores
    sc = scores.reshape(-1)[perm.long()].double().unsqueeze(1)
    go = g.double().requires_grad_(True)
    uo = u.double().requires_grad_(True)
    h = torch.nn.functional.silu(go) * uo
    dh, dx_ref, s = torch.empty(A, I, dtype=torch.float64, device=dev), torch.empty(A, H, dtype=torch.float64, device=dev), 0
    for e, c in enumerate(counts):
        dh[s:s + c] = d_out[perm[s:s + c].long() // K].double() @ w2[e].double()
        dx_ref[s:s + c] = dg[s:s + c].double() @ w1[e].double() + du[s:s + c].double() @ w3[e].double()
        s += c
    dg_ref, du_ref = torch.autograd.grad(h, (go, uo), dh)
    ds_ref = torch.zeros(A, dtype=torch.float64, device=dev).index_copy(0, perm.long(), (dh * h).sum(1).detach())
    for name, got, ref in (("d_g", dg, dg_ref * sc), ("d_u", du, du_ref * sc), ("score * h", hs, h.detach() * sc), ("d_score", ds, ds_ref),
                           ("d_x", dx, dx_ref), ("d_g unscaled", dg0, dg_ref), ("d_u unscaled", du0, du_ref)):
        assert rel_err(got, ref) <= tol, (name, rel_err(got, ref))


# widths and row counts that leave a remainder in the last k-tile of every product
REMAINDER_CASES = [
    ([3, 70, 0, 129], 200, 104),        # 64-wide tiles, reductions split over groups of waves
    ([65] * 64, 328, 136),              # 64-wide tiles, one group
    ([190] * 24, 1000, 360),            # 128-wide tiles
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,H,I", REMAINDER_CASES)
def test_infinities_stay_in_the_rows_and_columns_that_hold_them(dev, dtype, counts, H, I):
    """The tile kernels read an expert's first row, and a row's first elements, where a tile's remainder has none of its own, and mask
    both operands: an infinity in these places is neither multiplied by zero nor seen by anybody else (bit for bit)."""
    print(f"[case] infinities {dtype} counts={counts[:4]}x{len(counts)} H={H} I={I}", flush=True)
    x, w1, w2, w3, dy, cnt = _make(23, counts, H, I, dtype)
    X, W1, W2, W3, DY = (t.to(dev) for t in (x, w1, w2, w3, dy))
    starts = ops.counts_to_starts(cnt.to(dev))
    E, e = len(counts), 1
    row = counts[0]                      # first row of expert 1
    y, g, u, h = ops.grouped_swiglu_fwd(X, W1, W2, W3, starts)
    dw1, dw2, dw3 = ops.grouped_swiglu_wgrad(DY, h, g, u, X, starts, E)      # g and u stand for any d_g and d_u

    X2, DY2 = X.clone(), DY.clone()
    X2[row, 0] = float("inf")
    DY2[row, 5] = float("inf")
    y2, g2, u2, h2 = ops.grouped_swiglu_fwd(X2, W1, W2, W3, starts)
    assert torch.isinf(g2[row]).all() and torch.isinf(u2[row]).all()
    others = torch.arange(sum(counts), device=dev) != row
    for got, want in ((y2, y), (g2, g), (u2, u), (h2, h)):
        assert torch.equal(got[others], want[others])
    e1, e2, e3 = ops.grouped_swiglu_wgrad(DY2, h, g, u, X2, starts, E)
    assert torch.isinf(e2[e, 5]).all() and torch.isinf(e1[e, :, 0]).all() and torch.isinf(e3[e, :, 0]).all()
    keep = torch.ones(E, H, dtype=torch.bool, device=dev)
    keep[e, 5] = False
    assert torch.equal(e2[keep], dw2[keep])
    keep = torch.ones(E, H, dtype=torch.bool, device=dev)
    keep[e, 0] = False
    keep = keep[:, None, :].expand(E, I, H)
    assert torch.equal(e1[keep], dw1[keep]) and torch.equal(e3[keep], dw3[keep])


# Weight gradients of 256-wide tiles: rows of one expert around the k-tile's 32, and shapes whose workgroups form one tile, two
# neighbouring ones or four; with 512 rows an expert the 64-deep k-tiles.  Experts come in chunks that are dealt to the XCDs:
# fewer experts than XCDs do not get here, nine leave chunks over.
RUN_CASES = [
    ([0, 1, 31, 32, 33, 64, 65, 100, 300], 512, 768),                # one tile at a time
    ([31, 0, 65, 32] * 8, 1024, 512),                                # two
    ([0, 33, 64, 1, 97, 32, 45, 90] * 16, 1024, 1024),               # four
    ([900, 0, 31, 2, 1500, 65, 1000, 700], 1024, 512),               # 64-deep k-tiles
    ([300, 0, 31, 2, 500, 65, 900, 97], 1024, 512),                  # 32-deep ones in a ring of four stages
    ([224, 240, 0, 33, 500, 64, 700, 300] * 2, 1024, 768),           # (from two tiles for every CU on)
    ([0, 70, 33, 1, 130, 20, 64, 9] * 2, 768, 768),                  # an odd number of tiles an expert, dealt out in chunks of 3
    ([40, 0, 90, 32] * 3, 1280, 1280),                               # of 7, which cross from one expert to the next
    ([600, 0, 900, 1, 40, 1200, 700, 800], 1280, 768),               # of 2, which 45 is no multiple of
    ([40, 0, 65, 33], 1024, 1024),                                   # fewer experts than XCDs
    ([300, 500, 1, 0, 460], 2048, 768),
    ([1000, 700, 0, 900], 2048, 2048),
]


@pytest.mark.parametrize("counts,H,I", RUN_CASES)
@pytest.mark.parametrize("mapped", [True, False])
def test_weight_gradients_in_runs_of_tiles(dev, counts, H, I, mapped):
    """Every gradient against float64, stored over NaNs and added to old values, with gathered rows and without."""
    print(f"[case] runs of tiles counts={counts[:8]}x{len(counts)} H={H} I={I} mapped={mapped}", flush=True)
    E, A, K = len(counts), sum(counts), 2 if mapped else 1
    gen = torch.Generator(device=dev).manual_seed(H + I + E)
    rand = lambda *shape: torch.randn(shape, generator=gen, device=dev).bfloat16()
    T = -(-A // K)
    perm = torch.randperm(T * K, generator=gen, device=dev)[:A].int()
    x, dy, hs, dg, du = rand(T, H), rand(T, H), rand(A, I), rand(A, I), rand(A, I)
    starts = ops.counts_to_starts(torch.tensor(counts, dtype=torch.int32, device=dev))
    order = torch.argsort(torch.tensor(counts, device=dev), descending=True, stable=True).int()
    old = [rand(*s) for s in ((E, I, H), (E, H, I), (E, I, H))]
    kw = dict(row_map=perm, row_map_div=K, scaled=True) if mapped else {}
    fresh = [torch.full_like(o, float("nan")) for o in old]
    ops.grouped_swiglu_wgrad(dy, hs, dg, du, x, starts, E, d_w1=fresh[0], d_w2=fresh[1], d_w3=fresh[2], expert_order=order, **kw)
    added = [o.clone() for o in old]
    ops.grouped_swiglu_wgrad(dy, hs, dg, du, x, starts, E, d_w1=added[0], d_w2=added[1], d_w3=added[2], accumulate=True, **kw)
    rows = (perm // K).long() if mapped else torch.arange(A, device=dev)
    first = 0
    for e, n in enumerate(counts):
        r = slice(first, first + n)
        first += n
        if e >= 16 and e + 8 < E:          # the pattern repeats
            continue
        xe, dye = x[rows[r]].double(), dy[rows[r]].double()
        for got, acc, o, a, b in zip(fresh, added, old, (dg[r].double(), dye, du[r].double()), (xe, hs[r].double(), xe)):
            want, size = a.T @ b, a.abs().T @ b.abs()
            # fp32 sums of n products, then one rounding to bf16 (and one more of the sum with the old value)
            bound = want.abs() * 2**-8 + size * (n + 1) * 2**-23
            assert ((got[e].double() - want).abs() <= bound).all(), (e, n)
            total = want + o[e].double()
            bound = total.abs() * 2**-8 + bound + (size + total.abs()) * (n + 2) * 2**-23
            assert ((acc[e].double() - total).abs() <= bound).all(), (e, n)


@pytest.mark.parametrize("mapped", [True, False])
@pytest.mark.parametrize("skew", [True, False])
def test_units_of_160_rows(dev, mapped, skew):
    """Sizes that the persistent products take in units of 160 rows (gate/up, down and d_x alike): experts around one and two units, with
    one row, a chunk and one, and none.  Every result against float64 of what the product read."""
    H, I, E, A = 768, 1024, 8, 21504
    counts = [0, 1, 159, 160, 161, 321, 33] if skew else [2560, 2720, 2687, 2689, 2700, 2721, 2710]
    counts.append(A - sum(counts))
    print(f"[case] units of 160 rows counts={counts} mapped={mapped}", flush=True)
    gen = torch.Generator(device=dev).manual_seed(160 + skew)
    rand = lambda *shape, scale=1.0: (torch.randn(shape, generator=gen, device=dev) * scale).bfloat16()
    K = 2 if mapped else 1
    x = rand(A // K, H)
    w1, w3, w2 = rand(E, I, H, scale=0.05), rand(E, I, H, scale=0.05), rand(E, H, I, scale=0.05)
    perm = torch.randperm(A, generator=gen, device=dev).int()
    starts = ops.counts_to_starts(torch.tensor(counts, dtype=torch.int32, device=dev))
    kw = dict(row_map=perm, row_map_div=K, num_rows=A) if mapped else {}
    y, g, u, h = ops.grouped_swiglu_fwd(x, w1, w2, w3, starts, **kw)
    dx = ops.grouped_swiglu_dgrad_dx(g, u, w1, w3, starts)                 # g and u stand for any d_g and d_u
    rows = (perm // K).long() if mapped else torch.arange(A, device=dev)

    def check(got, pairs, what):
        """got: the sum of the products of `pairs`, in fp32 and rounded once"""
        want = sum(a @ b for a, b in pairs)
        size, k = sum(a.abs() @ b.abs() for a, b in pairs), sum(a.shape[1] for a, _ in pairs)
        assert ((got.double() - want).abs() <= want.abs() * 2**-8 + size * (k + 1) * 2**-23).all(), what

    first = 0
    for e, n in enumerate(counts):
        r = slice(first, first + n)
        first += n
        xe, ge, ue, he = x[rows[r]].double(), g[r].double(), u[r].double(), h[r].double()
        check(g[r], [(xe, w1[e].double().T)], ("g", e, n))
        check(u[r], [(xe, w3[e].double().T)], ("u", e, n))
        # silu with the hardware's exponential and reciprocal, one rounding to bf16
        want = torch.nn.functional.silu(ge) * ue
        assert ((he - want).abs() <= want.abs() * (2**-8 + 2**-18) + 1e-30).all(), ("h", e, n)
        check(y[r], [(he, w2[e].double().T)], ("y", e, n))
        check(dx[r], [(ge, w1[e].double()), (ue, w3[e].double())], ("d_x", e, n))


# Tile kernels request the k-tiles that are there and no others: reductions of none, one to nine k-tiles for a group of waves, a part of
# one at their ends.  Widths whose tiles are 64 wide with four, two and one such groups, and 128 wide.
K_LOOP_CASES = [(104, 72, 4), (200, 104, 2), (584, 264, 1), (1000, 512, 1)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,I,groups", K_LOOP_CASES)
@pytest.mark.parametrize("mapped", [True, False])
def test_weight_gradients_at_every_end_of_their_k_loops(dev, dtype, H, I, groups, mapped):
    print(f"[case] k-loop ends, weight gradients {dtype} H={H} I={I} groups={groups} mapped={mapped}", flush=True)
    bk = (64 if dtype == torch.bfloat16 else 32) * groups
    counts = [max(0, n * bk + off) for n, off in zip([0, 1, 1, 2, 2, 3, 4, 5, 6, 7, 8, 9, 9], [0, -bk + 1, 0, 0, -3, 0, 5, -1, 0, 1, 0, -7, 0])]
    E, A, K = len(counts), sum(counts), 2 if mapped else 1
    gen = torch.Generator(device=dev).manual_seed(H + I + bk)
    rand = lambda *shape: torch.randn(shape, generator=gen, device=dev).to(dtype)
    T = -(-A // K)
    perm = torch.randperm(T * K, generator=gen, device=dev)[:A].int()
    x, dy, hs, dg, du = rand(T, H), rand(T, H), rand(A, I), rand(A, I), rand(A, I)
    starts = ops.counts_to_starts(torch.tensor(counts, dtype=torch.int32, device=dev))
    kw = dict(row_map=perm, row_map_div=K, scaled=True) if mapped else {}
    got = [torch.full(s, float("nan"), dtype=dtype, device=dev) for s in ((E, I, H), (E, H, I), (E, I, H))]
    ops.grouped_swiglu_wgrad(dy, hs, dg, du, x, starts, E, d_w1=got[0], d_w2=got[1], d_w3=got[2], **kw)
    rows = (perm // K).long() if mapped else torch.arange(A, device=dev)
    ulp = 2**-8 if dtype == torch.bfloat16 else 2**-24
    first = 0
    for e, n in enumerate(counts):
        r = slice(first, first + n)
        first += n
        xe, dye = x[rows[r]].double(), dy[rows[r]].double()
        for g, a, b in zip(got, (dg[r].double(), dye, du[r].double()), (xe, hs[r].double(), xe)):
            want, size = a.T @ b, a.abs().T @ b.abs()
            assert ((g[e].double() - want).abs() <= want.abs() * ulp + size * (n + 1) * 2**-23).all(), (e, n)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("many", [True, False])
def test_tile_products_at_every_end_of_their_k_loops(dev, dtype, many):
    """Gate/up over H, down and d_x over I (d_x twice as long).  many: enough tiles that nobody shares a reduction."""
    bk = 64 if dtype == torch.bfloat16 else 32
    counts = [0, 1, 63, 64, 65, 130] * (10 if many else 1)
    E, A = len(counts), sum(counts)
    gen = torch.Generator(device=dev).manual_seed(bk + many)
    rand = lambda *shape, scale=1.0: (torch.randn(shape, generator=gen, device=dev) * scale).to(dtype)
    starts = ops.counts_to_starts(torch.tensor(counts, dtype=torch.int32, device=dev))
    ulp = 2**-8 if dtype == torch.bfloat16 else 2**-24

    def check(got, pairs, what):
        want = sum(a @ b for a, b in pairs)
        size, k = sum(a.abs() @ b.abs() for a, b in pairs), sum(a.shape[1] for a, _ in pairs)
        assert ((got.double() - want).abs() <= want.abs() * ulp + size * (k + 1) * 2**-23).all(), what

    for n in range(1, 10):
        for k in (n * bk - 24, n * bk):
            for H, I in ((k, 392), (392, k)):
                print(f"[case] k-loop ends {dtype} H={H} I={I} E={E}", flush=True)
                x, w1, w3, w2 = rand(A, H), rand(E, I, H, scale=0.05), rand(E, I, H, scale=0.05), rand(E, H, I, scale=0.05)
                y, g, u, h = ops.grouped_swiglu_fwd(x, w1, w2, w3, starts)
                dx = ops.grouped_swiglu_dgrad_dx(g, u, w1, w3, starts)
                first = 0
                for e in range(E):
                    r = slice(first, first + counts[e])
                    first += counts[e]
                    if e >= 6 and e + 6 < E:           # the pattern repeats
                        continue
                    xe, ge, ue = x[r].double(), g[r].double(), u[r].double()
                    check(g[r], [(xe, w1[e].double().T)], ("g", e))
                    check(u[r], [(xe, w3[e].double().T)], ("u", e))
                    check(y[r], [(h[r].double(), w2[e].double().T)], ("y", e))
                    check(dx[r], [(ge, w1[e].double()), (ue, w3[e].double())], ("d_x", e))


# fp32 products whose tiles are mostly padding: their loads leave out the rows that are not there.  From one row an expert to half a
# tile on average with some tiles full, in the tiles that few and many of them are cut into.
SPARSE_CASES = [
    ([1, 2, 0, 5], 456, 392),                        # 32 x 32, four groups
    ([8] * 24, 1000, 392),                           # 64 x 32
    ([16] * 16, 512, 400),                           # 32 x 64
    ([0, 130, 1, 31, 2, 20, 33, 5] * 4, 1000, 520),  # 64 x 64
    ([32, 64, 1, 7] * 16, 904, 424),
]


@pytest.mark.parametrize("counts,H,I", SPARSE_CASES)
def test_fp32_products_with_mostly_empty_tiles(dev, counts, H, I):
    print(f"[case] mostly empty tiles counts={counts[:8]}x{len(counts)} H={H} I={I}", flush=True)
    E, A, K = len(counts), sum(counts) - sum(counts) % 2, 2
    counts = counts[:-1] + [counts[-1] - (sum(counts) - A)]
    gen = torch.Generator(device=dev).manual_seed(E + H)
    rand = lambda *shape, scale=1.0: torch.randn(shape, generator=gen, device=dev) * scale
    x, dy, w1, w3, w2 = rand(A // K, H), rand(A // K, H), rand(E, I, H, scale=0.05), rand(E, I, H, scale=0.05), rand(E, H, I, scale=0.05)
    perm = torch.randperm(A, generator=gen, device=dev).int()
    scores = torch.rand((A // K, K), generator=gen, device=dev) + 0.1
    starts = ops.counts_to_starts(torch.tensor(counts, dtype=torch.int32, device=dev))
    y, g, u, h = ops.grouped_swiglu_fwd(x, w1, w2, w3, starts, row_map=perm, row_map_div=K, num_rows=A)
    dg, du, hs, ds = ops.grouped_swiglu_dgrad_dh_scaled(dy, perm, scores, w2, g, u, starts)
    dx = ops.grouped_swiglu_dgrad_dx(g, u, w1, w3, starts)
    rows = (perm // K).long()

    def check(got, pairs, what):
        want = sum(a @ b for a, b in pairs)
        size, k = sum(a.abs() @ b.abs() for a, b in pairs), sum(a.shape[1] for a, _ in pairs)
        assert ((got.double() - want).abs() <= size * (k + 2) * 2**-23).all(), what

    first = 0
    for e, n in enumerate(counts):
        r = slice(first, first + n)
        first += n
        xe, ge, ue, dye = x[rows[r]].double(), g[r].double(), u[r].double(), dy[rows[r]].double()
        sc = scores.flatten()[perm[r].long()].double()
        check(g[r], [(xe, w1[e].double().T)], ("g", e))
        check(u[r], [(xe, w3[e].double().T)], ("u", e))
        check(y[r], [(h[r].double(), w2[e].double().T)], ("y", e))
        check(dx[r], [(ge, w1[e].double()), (ue, w3[e].double())], ("d_x", e))
        # d_u = score * d_h * silu(g): the product's bound times the factor, and a few roundings of the factor itself
        dh, size = dye @ w2[e].double(), dye.abs() @ w2[e].double().abs()
        f = sc[:, None] * torch.nn.functional.silu(ge)
        assert ((du[r].double() - dh * f).abs() <= (size * (H + 2) * 2**-23 + dh.abs() * 2**-20) * f.abs() + 1e-30).all(), ("d_u", e)
        sg = torch.sigmoid(ge)
        f = sc[:, None] * ue * (sg * (1 + ge * (1 - sg)))
        # (1 + g (1 - sigmoid)) can cancel: its own rounding is relative to its terms
        terms = sc[:, None] * ue.abs() * sg * (1 + ge.abs())
        assert ((dg[r].double() - dh * f).abs() <= size * (H + 2) * 2**-23 * f.abs() + dh.abs() * terms * 2**-20 + 1e-30).all(), ("d_g", e)
        hv = torch.nn.functional.silu(ge) * ue
        assert ((hs[r].double() - sc[:, None] * hv).abs() <= sc[:, None] * hv.abs() * 2**-20 + 1e-30).all(), ("score * h", e)
        bound = (size * hv.abs()).sum(1) * (H + I) * 2**-22
        assert ((ds.flatten()[perm[r].long()].double() - (dh * hv).sum(1)).abs() <= bound + 1e-30).all(), ("d_score", e)


@pytest.mark.parametrize("H", [128, 256])
def test_units_of_160_rows_with_short_reductions(dev, H):
    """Gate/up with two or four k-tiles and gathered rows: the loader enters the next unit in the epilogue, not in the k-loop."""
    I, E, K = 1280, 64, 2
    counts = [159, 160, 161, 319, 320, 321, 1, 639] * 8
    A = sum(counts)
    print(f"[case] units of 160 rows, H={H}", flush=True)
    gen = torch.Generator(device=dev).manual_seed(H)
    rand = lambda *shape, scale=1.0: (torch.randn(shape, generator=gen, device=dev) * scale).bfloat16()
    x = rand(A // K, H)
    w1, w3, w2 = rand(E, I, H, scale=0.1), rand(E, I, H, scale=0.1), rand(E, H, I, scale=0.05)
    perm = torch.randperm(A, generator=gen, device=dev).int()
    starts = ops.counts_to_starts(torch.tensor(counts, dtype=torch.int32, device=dev))
    y, g, u, h = ops.grouped_swiglu_fwd(x, w1, w2, w3, starts, row_map=perm, row_map_div=K, num_rows=A)
    rows = (perm // K).long()
    first = 0
    for e, n in enumerate(counts):
        r = slice(first, first + n)
        first += n
        xe, ge, ue = x[rows[r]].double(), g[r].double(), u[r].double()
        for got, w in ((g, w1), (u, w3)):
            want, size = xe @ w[e].double().T, xe.abs() @ w[e].double().abs().T
            assert ((got[r].double() - want).abs() <= want.abs() * 2**-8 + size * (H + 1) * 2**-23).all(), e
        want = torch.nn.functional.silu(ge) * ue
        assert ((h[r].double() - want).abs() <= want.abs() * (2**-8 + 2**-18) + 1e-30).all(), e


def test_gate_and_up_do_not_depend_on_the_units_height(dev):
    """The first 16 of 64 experts by themselves are on 128-row units, all of them on 160-row ones: the same sums in the same order."""
    H, I, K = 2048, 1280, 2
    counts = [159, 160, 161, 319, 320, 321, 1, 639] * 8
    A, few = sum(counts), sum(counts[:16])
    print("[case] 160- against 128-row units", flush=True)
    gen = torch.Generator(device=dev).manual_seed(160)
    rand = lambda *shape, scale=1.0: (torch.randn(shape, generator=gen, device=dev) * scale).bfloat16()
    x = rand(A // K, H)
    w1, w3, w2 = rand(64, I, H, scale=0.05), rand(64, I, H, scale=0.05), rand(64, H, I, scale=0.05)
    perm = torch.randperm(A, generator=gen, device=dev).int()
    starts = ops.counts_to_starts(torch.tensor(counts, dtype=torch.int32, device=dev))
    _, g, u, h = ops.grouped_swiglu_fwd(x, w1, w2, w3, starts, row_map=perm, row_map_div=K, num_rows=A)
    _, g2, u2, h2 = ops.grouped_swiglu_fwd(x, w1[:16], w2[:16], w3[:16], starts[:17].contiguous(), row_map=perm[:few].contiguous(),
                                           row_map_div=K, num_rows=few)
    assert torch.equal(g[:few], g2) and torch.equal(u[:few], u2) and torch.equal(h[:few], h2)
