"""The work that a user of piper_amd has it do, as cases that can be timed and compared.

Four kinds of work, each through the public entry points, as a training or inference program calls them:

* ``infer``: ``MoEFeedForwardBlock`` (norm, router, experts, residual) without autograd, from one decoded
  token to a prefill of several thousand tokens;
* ``train``: forward and backward of the same block with the gradients of every parameter
  (``flow="fused"``), or of ``AnnotatedMoE(fused=False)``, the reference's op-by-op data flow with the
  ``piper_artifact::bmm_experts`` operator in it (``flow="ops"``);
* ``bucket``: the ZeRO bucket path of an iteration: zero, a gradient pack per microbatch, one AdamW step
  (``hold``: the last pack is folded into the step, as ``StageExecutor(fuse_last_pack=True)`` does);
* ``stage``: ``StageExecutor.run``: microbatches in 1F1B order over the MoE blocks of a stage whose
  parameters live in ZeRO buckets, packs on a second stream, one update.

Widths are those of the benchmark configurations (``piper_amd.configs``), of the tests, or generic.
"""
from __future__ import annotations

import math

import torch

from piper_amd.bucket import BucketState, ParamStorage, StageStore, flatten_params
from piper_amd.configs import ADAMW, bucket_manifest_cfg2, zipf_logit_bias
from piper_amd.executor import StageExecutor, one_f_one_b
from piper_amd.functional import moe_block
from piper_amd.moe import AnnotatedMoE, MoEArgs, MoEFeedForwardBlock
from piper_amd.optim import FusedAdamW
from piper_amd.stage import StageNode, load_stage

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
WIDE = dict(hidden=2048, experts=128, top_k=8, inter=768)      # the benchmark's expert region
TINY = dict(hidden=256, experts=8, top_k=2, inter=512)         # the small fp32 configuration

# what the largest listed case costs; no drawn case costs more
_MAX_FLOPS = 18 * 8 * 2048 * 768 * 16384
_MAX_BYTES = 7e9


def listed() -> list[dict]:
    return [
        # one sequence being decoded: launches and the weights of eight experts
        dict(name="decode_1", kind="infer", tokens=1, dtype="bf16", skew=0.0, **WIDE),
        # a decode batch: every expert has a row or two, so the weights are the traffic
        dict(name="decode_24", kind="infer", tokens=24, dtype="bf16", skew=0.0, **WIDE),
        # the prompt of one request, of no particular length
        dict(name="prefill_1777", kind="infer", tokens=1777, dtype="bf16", skew=0.0, **WIDE),
        # a short, odd microbatch (fine-tuning, the tail of a packed batch)
        dict(name="train_509", kind="train", flow="fused", tokens=509, dtype="bf16", skew=0.0, **WIDE),
        # the benchmark's microbatch, evenly routed
        dict(name="train_4096", kind="train", flow="fused", tokens=4096, dtype="bf16", skew=0.0, **WIDE),
        # the benchmark's long microbatch with Zipf-distributed expert popularity
        dict(name="train_16384_skewed", kind="train", flow="fused", tokens=16384, dtype="bf16", skew=0.45, **WIDE),
        # a small fp32 model
        dict(name="train_f32_1000", kind="train", flow="fused", tokens=1000, dtype="f32", skew=0.0, hidden=512, experts=16,
             top_k=4, inter=256),
        # widths that are no multiple of a tile
        dict(name="train_ragged_widths", kind="train", flow="fused", tokens=1030, dtype="bf16", skew=0.0, hidden=1000, experts=24,
             top_k=4, inter=360),
        # reference model code: router, reorderer, gather, experts operator, scatter one by one
        dict(name="ops_1024", kind="train", flow="ops", tokens=1024, dtype="bf16", skew=0.0, hidden=1024, experts=32, top_k=4,
             inter=512),
        # the parameters of two decoder layers in one bucket, one microbatch
        dict(name="bucket_96", kind="bucket", tensors=0, scale=0, dtype="bf16", microbatches=1, hold=False),
        # a bucket of norm vectors, biases and small matrices
        dict(name="bucket_small", kind="bucket", tensors=40, scale=3000, dtype="bf16", microbatches=2, hold=True),
        # the small fp32 configuration as it is run: four microbatches of 2 x 128 tokens, one bucket, one step
        dict(name="stage_f32", kind="stage", layers=1, microbatches=4, tokens=256, dtype="f32", hold=False, **TINY),
    ]


# ------------------------------------------------------------------------------------- draws
def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _widths(rng, dtype: str) -> dict:
    """Half of the draws have widths in multiples of 128, the rest in multiples of 8."""
    experts = rng.choice([4, 8, 16, 24, 32, 64, 128])
    top_k = min(experts, rng.choice([1, 2, 4, 6, 8]))
    step = rng.choice([128, 128, 8])
    top = 2048 if dtype == "bf16" else 1024
    hidden = max(1, _log_int(rng, 256, top) // step) * step
    inter = max(1, _log_int(rng, 128, top // 2) // step) * step
    return dict(hidden=hidden, experts=experts, top_k=top_k, inter=inter)


def _drawn(rng) -> dict:
    kind = rng.choice(["infer", "infer", "infer", "train", "train", "train", "train", "bucket", "bucket", "stage"])
    if kind == "infer":
        w = dict(WIDE) if rng.random() < 0.5 else _widths(rng, "bf16")
        return dict(kind=kind, tokens=_log_int(rng, 1, 8192), dtype="bf16", skew=rng.choice([0.0, 0.45]), **w)
    if kind == "train":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        w = dict(WIDE) if dtype == "bf16" and rng.random() < 0.4 else _widths(rng, dtype)
        return dict(kind=kind, flow=rng.choice(["fused", "fused", "fused", "ops"]),
                    tokens=_log_int(rng, 64, 16384 if dtype == "bf16" else 4096), dtype=dtype, skew=rng.choice([0.0, 0.45]), **w)
    if kind == "bucket":
        return dict(kind=kind, tensors=_log_int(rng, 4, 256), scale=_log_int(rng, 1000, 2_000_000), dtype=rng.choice(["bf16", "bf16", "f32"]),
                    microbatches=rng.choice([1, 2, 4]), hold=rng.random() < 0.5)
    dtype = rng.choice(["bf16", "f32"])
    return dict(kind=kind, layers=rng.choice([1, 2, 3]), microbatches=rng.choice([2, 4, 8]), tokens=_log_int(rng, 64, 2048), dtype=dtype,
                hold=rng.random() < 0.5, **_widths(rng, dtype))


def draw(rng) -> dict:
    while True:
        case = _drawn(rng)
        w = work(case)
        if w["flops"] <= _MAX_FLOPS * (1.0 if case.get("dtype") == "bf16" else 0.03) and w["bytes"] <= _MAX_BYTES:
            return case


# ------------------------------------------------------------------------------------- inputs
def _moe_args(case: dict) -> MoEArgs:
    return MoEArgs(num_experts=case["experts"], top_k=case["top_k"], route_norm=True, gate_bias=bool(case.get("skew")))


def _fill_moe(moe: AnnotatedMoE, case: dict, gen: torch.Generator) -> None:
    moe.init_weights(std=0.02, generator=gen)
    if case.get("skew"):
        with torch.no_grad():
            moe.router.gate.bias.copy_(zipf_logit_bias(case["experts"], 1.2, case["skew"]))


def _bucket_shapes(case: dict) -> list[tuple[int, ...]]:
    if case["tensors"] == 0:
        return [s for _, s in bucket_manifest_cfg2()]
    # vectors next to matrices, none of a round size, from a sixteenth of `scale` elements to twice `scale`
    shapes = []
    for i in range(case["tensors"]):
        n = int(case["scale"] * (0.0625, 1.0, 0.3, 2.0)[i % 4]) + 7 * i + 1
        shapes.append((n,) if i % 4 == 0 else (max(1, n // 96), 96))
    return shapes


def prepare(case: dict, seed: int):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    if case["kind"] in ("infer", "train"):
        with torch.device(dev):
            if case.get("flow", "fused") == "fused":
                module = MoEFeedForwardBlock(_moe_args(case), case["hidden"], case["inter"], dtype=dtype)
                moe = module.moe
            else:
                module = moe = AnnotatedMoE(_moe_args(case), case["hidden"], case["inter"], dtype=dtype, fused=False)
        _fill_moe(moe, case, gen)
        x = torch.randn((1, case["tokens"], case["hidden"]), generator=gen, device=dev).to(dtype)
        if case["kind"] == "infer":
            return dict(case=case, module=module.requires_grad_(False), x=x)
        d_out = torch.randn((1, case["tokens"], case["hidden"]), generator=gen, device=dev).to(dtype)
        return dict(case=case, module=module, x=x.requires_grad_(True), d_out=d_out, params=list(module.parameters()))

    if case["kind"] == "bucket":
        shapes = _bucket_shapes(case)
        params = [torch.nn.Parameter((torch.randn(s, generator=gen, device=dev) * 0.02).to(dtype)) for s in shapes]
        grads = [[(torch.randn(s, generator=gen, device=dev) * 1e-3).to(dtype) for s in shapes] for _ in range(case["microbatches"])]
        bucket = flatten_params(BucketState(), params, optim_class=lambda ps: FusedAdamW(ps, **ADAMW))
        store = StageStore(buckets={0: bucket}, zero_managed_ubids={0})
        return dict(case=case, bucket=bucket, params=params, grads=grads, storage=ParamStorage(store))

    # stage
    top_k = case["top_k"]

    def layer(x, p):
        return moe_block(x, p["ffn_norm"], p["w_gate"], None, p["w1"], p["w2"], p["w3"], top_k=top_k, route_norm=True)

    H, I, E = case["hidden"], case["inter"], case["experts"]
    nodes = []
    for _ in range(case["layers"]):
        p = dict(ffn_norm=torch.ones(H, device=dev, dtype=dtype))
        for name, shape in (("w1", (E, I, H)), ("w2", (E, H, I)), ("w3", (E, I, H))):
            p[name] = (torch.randn(shape, generator=gen, device=dev) * 0.02).to(dtype)
        p["w_gate"] = torch.randn((E, H), generator=gen, device=dev) * 0.02
        nodes.append(StageNode(layer, {k: torch.nn.Parameter(v) for k, v in p.items()}))
    store = load_stage(nodes, [[i] for i in range(case["layers"])], optim_class=lambda ps: FusedAdamW(ps, **ADAMW))
    xs = [torch.randn((case["tokens"], H), generator=gen, device=dev).to(dtype) for _ in range(case["microbatches"])]
    targets = [torch.randn((case["tokens"], H), generator=gen, device=dev) for _ in range(case["microbatches"])]
    executor = StageExecutor(store, compute_stream=torch.cuda.Stream(), pack_stream=torch.cuda.Stream(), fuse_last_pack=case["hold"],
                             loss_fn=lambda out, target: torch.nn.functional.mse_loss(out.float(), target, reduction="sum") / out.shape[0])
    tasks = one_f_one_b(case["microbatches"], list(store.buckets))
    return dict(case=case, executor=executor, tasks=tasks, xs=xs, targets=targets, store=store)


# ------------------------------------------------------------------------------------- one pass
def _optimizer_state(bucket: BucketState) -> list[torch.Tensor]:
    st = bucket.shard_optimizer.state[bucket.shard_param]
    return [bucket.flat_params.detach(), bucket.flat_grads, st["master"].detach(), st["exp_avg"], st["exp_avg_sq"]]


def run(state):
    case = state["case"]
    if case["kind"] == "infer":
        with torch.no_grad():
            return state["module"](state["x"])
    if case["kind"] == "train":
        module, x = state["module"], state["x"]
        x.grad = None
        for p in state["params"]:
            p.grad = None
        out = module(x)
        out.backward(state["d_out"])
        return [out.detach(), x.grad] + [p.grad for p in state["params"]]
    if case["kind"] == "bucket":
        storage, params = state["storage"], state["params"]
        storage.zero_grad_buffers()
        for mb, grads in enumerate(state["grads"]):
            for p, g in zip(params, grads):
                p.grad = g
            if case["hold"] and mb == len(state["grads"]) - 1:
                storage.hold_param_grads(0)
            else:
                storage.accumulate_zero_param_grads_to_flat(0)
        storage.step_zero_shard_optimizers()
        return _optimizer_state(state["bucket"])
    result = state["executor"].run(state["tasks"], state["xs"], state["targets"])
    out = [torch.stack(result["losses"])]
    for bucket in state["store"].buckets.values():
        for b in bucket.with_companions():
            out += _optimizer_state(b)
    return out


# ------------------------------------------------------------------------------------- work
def _experts_touched(case: dict) -> float:
    """Expected number of experts with at least one row, routing evenly."""
    return case["experts"] * (1.0 - (1.0 - case["top_k"] / case["experts"]) ** case["tokens"])


def work(case: dict) -> dict:
    """Each input read once, each output written once; the products of the experts and the router."""
    es = 2 if case["dtype"] == "bf16" else 4
    if case["kind"] == "bucket":
        n = sum(math.prod(s) for s in _bucket_shapes(case))
        packs = case["microbatches"] - (1 if case["hold"] else 0)
        # gradients read, bucket written where something is packed, master and moments both ways, parameters written
        per = es * case["microbatches"] + (4 if packs or not case["hold"] else 0) + 24 + (2 if es == 2 else 0)
        return {"bytes": n * per, "flops": 0}
    T, H, I, E, K = (case[k] for k in ("tokens", "hidden", "inter", "experts", "top_k"))
    expert = 3 * H * I                              # one expert's weights
    forward = 6 * T * K * H * I + 2 * T * H * E
    if case["kind"] == "infer":
        return {"bytes": es * (_experts_touched(case) * expert + 2 * T * H) + 4 * E * H, "flops": forward}
    if case["kind"] == "train":
        # weights in, weight gradients out (all experts), x and d_out in, out and d_x out
        return {"bytes": es * ((_experts_touched(case) + E) * expert + 4 * T * H) + 8 * E * H, "flops": 3 * forward}
    n = case["layers"] * (E * expert + H)
    mb = case["microbatches"]
    traffic = n * (2 * es + 24 + 4 + (2 if es == 2 else 0)) + mb * T * H * (es + 4)
    return {"bytes": traffic, "flops": 3 * mb * case["layers"] * forward}


def tolerance(case: dict):
    """bf16: products of bf16 operands summed in fp32 and rounded to bf16 between the operators, so 1e-2; a
    router logit that moves by one fp32 rounding can swap two experts whose logits are a near-tie, which
    changes that token's row (and its row's share of a weight gradient) by a fraction of its size: `max`.
    fp32: sums of a few thousand fp32 products.  After AdamW, whose first steps divide a gradient by its
    own magnitude, a gradient near zero carries its relative error into the parameter."""
    if case["kind"] == "bucket":
        return {"rel": 1e-5, "max": 1e-2} if case["dtype"] == "f32" else {"rel": 1e-3, "max": 1e-2}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 1e-4, "max": 0.2} if case["kind"] == "stage" else {"rel": 1e-5, "max": 1e-3}
