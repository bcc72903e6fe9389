"""The work that users have this framework do: fused attention with a forward-mode tangent, and its gradients.

A case is one attention layer of one step, called through the public surface (``JVPAttn.fwd_dual`` on dual tensors,
``attention`` without tangents).  ``grads`` says what the step then asks of it:

* ``none``     the forward alone (sampling, evaluation, the tangent as a quantity of its own)
* ``o``        gradients of q, k, v from O; the tangent is a target that no gradient flows through (consistency and
               flow-map training, and every first-order step)
* ``tangent``  gradients of q, k, v from O' alone (Hessian-vector products)
* ``both``     gradients of q, k, v from O and O'
* ``all``      the same for the tangent inputs as well (a layer inside a network whose tangents are trained through)
"""
import math

import torch
import torch.autograd.forward_ad as fwAD

from jvp_flash_attention_amd import JVPAttn, attention

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
DOCUMENTS = 4  # documents packed into one row of a "packed" batch, on average


def _case(name, dtype, batch, heads, q_len, head_dim, mask="none", grads="none", kv_heads=None, kv_len=None, tangents=True,
          tangent_std=1.0, dropout=0.0):
    return {"name": name, "dtype": dtype, "batch": batch, "heads": heads, "kv_heads": kv_heads or heads, "q_len": q_len,
            "kv_len": kv_len or q_len, "head_dim": head_dim, "mask": mask, "grads": grads, "tangents": tangents,
            "tangent_std": tangent_std, "dropout": dropout}


def listed():
    return [
        # a short sequence, forward only: launches and host time are what counts
        _case("dual_l128_d64", "bf16", 2, 12, 128, 64),
        # image patches (14 x 14 and one more) with the tangent as a target
        _case("target_l197_d64", "bf16", 8, 6, 197, 64, grads="o"),
        # second-order step on a short causal sequence
        _case("hvp_l1024_d128", "bf16", 1, 16, 1024, 128, mask="causal", grads="tangent"),
        # fp32, keys padded per batch entry
        _case("fp32_padding_l1024_d64", "fp32", 4, 8, 1024, 64, mask="padding", grads="both"),
        # fp32, a learned bias per head
        _case("fp32_bias_l1024_d64", "fp32", 4, 8, 1024, 64, mask="bias", grads="both"),
        # plain first-order training of a causal language model: grouped heads, dropout, a length of no tile
        _case("lm_dropout_l1500_d64", "bf16", 4, 16, 1500, 64, mask="causal", grads="o", kv_heads=4, tangents=False, dropout=0.1),
        # ordinary dense step at the head dim of the smaller models
        _case("both_l2048_d64", "bf16", 4, 16, 2048, 64, grads="both", tangent_std=0.1),
        # documents packed into one row, tangents trained through, an odd length
        _case("packed_all_l2077_d128", "bf16", 2, 16, 2077, 128, mask="packed", grads="all"),
        # queries over a padded context of another length, wide heads, the tangent as a target
        _case("cross_target_l1000_d256", "fp16", 4, 8, 1000, 256, mask="padding", grads="o", kv_len=1500),
        # the dense forward at full size
        _case("dual_l4096_d128", "bf16", 4, 16, 4096, 128),
        # causal step at full size in fp16
        _case("causal_fp16_l4096_d128", "fp16", 2, 32, 4096, 128, mask="causal", grads="both"),
        # second-order step on the longest sequence
        _case("hvp_l32768_d128", "bf16", 1, 16, 32768, 128, mask="causal", grads="tangent"),
    ]


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        head_dim = rng.choice([32, 64, 64, 64, 128, 128, 128, 256])
        heads = rng.choice([2, 3, 4, 6, 8, 12, 16, 16, 24, 32])
        q_len = int(math.exp(rng.uniform(math.log(32), math.log(16384))))
        mask = rng.choice(["none", "none", "none", "causal", "causal", "causal", "padding", "padding", "packed", "bias", "dense"])
        tangents = rng.random() < 0.8
        kv_len = q_len
        if mask in ("none", "padding", "bias") and rng.random() < 0.25:
            kv_len = max(32, int(q_len * math.exp(rng.uniform(-1.0, 1.0))))
        kv_heads = rng.choice([k for k in range(1, heads + 1) if heads % k == 0]) if rng.random() < 0.2 else heads
        grads = rng.choice(["none", "o", "o", "tangent", "both", "both", "all"]) if tangents else rng.choice(["none", "o", "o"])
        case = _case(None, dtype, rng.choice([1, 1, 2, 2, 3, 4, 8]), heads, q_len, head_dim, mask, grads, kv_heads, kv_len, tangents,
                     rng.choice([0.1, 1.0]), rng.choice([0.1, 0.2]) if rng.random() < 0.1 else 0.0)
        del case["name"]
        elements = case["batch"] * heads * max(q_len, kv_len) * head_dim
        if _cost(case) <= most and elements <= 1 << 28 and _mask_bytes(case) <= 1 << 30:
            return case


def _mask_bytes(case):
    planes = {"none": 0, "causal": 0, "padding": case["batch"], "packed": case["batch"] * case["q_len"],
              "bias": case["batch"] * case["heads"] * case["q_len"] * BYTES[case["dtype"]],
              "dense": case["batch"] * case["heads"] * case["q_len"]}[case["mask"]]
    return planes * case["kv_len"]


def _attended(case):
    """Share of the score matrix that the mask leaves to compute (its expectation, where the mask comes from the seed)."""
    if case["mask"] == "causal":
        return 0.5 * (1 + 1 / case["q_len"])
    if case["mask"] == "padding":
        return 0.75
    if case["mask"] == "packed":  # two points of a row with no boundary between them
        return 2 / DOCUMENTS - 2 / DOCUMENTS**2 * (1 - math.exp(-DOCUMENTS))
    return 1.0


def _products(case):
    """Matrix products over the score matrix that one pass cannot do without."""
    forward = 6 if case["tangents"] else 2
    backward = {"none": 0, "o": 5, "tangent": 10, "both": 12, "all": 15}[case["grads"]]
    return forward + backward


def _cost(case):
    n = case["batch"] * case["heads"] * case["q_len"] * case["kv_len"] * case["head_dim"]
    return 2.0 * n * _products(case) * _attended(case) * (16 if case["dtype"] == "fp32" else 1)


def work(case):
    q = case["batch"] * case["heads"] * case["q_len"] * case["head_dim"]
    kv = case["batch"] * case["kv_heads"] * case["kv_len"] * case["head_dim"]
    qs = 4 if case["tangents"] else 2  # q, O and their tangents
    kvs = 4 if case["tangents"] else 2
    if case["grads"] != "none":
        qs += 1 + {"o": 1, "tangent": 1, "both": 2, "all": 2}[case["grads"]]  # dq, and the gradients that arrive
        kvs += 2
    if case["grads"] == "all":
        qs, kvs = qs + 1, kvs + 2
    n = case["batch"] * case["heads"] * case["q_len"] * case["kv_len"] * case["head_dim"]
    return {"bytes": (qs * q + kvs * kv) * BYTES[case["dtype"]] + _mask_bytes(case), "flops": 2.0 * n * _products(case) * _attended(case)}


def prepare(case, seed):
    device = torch.device("cuda")
    gen = torch.Generator(device=device).manual_seed(seed)
    dtype, B, H = DTYPES[case["dtype"]], case["batch"], case["heads"]
    Lq, Lk = case["q_len"], case["kv_len"]
    q_shape, kv_shape = (B, H, Lq, case["head_dim"]), (B, case["kv_heads"], Lk, case["head_dim"])

    def normal(shape, std=1.0):
        return torch.randn(shape, generator=gen, device=device, dtype=torch.float32).mul_(std).to(dtype)

    state = {"causal": case["mask"] == "causal", "dropout": case["dropout"], "grads": case["grads"], "mask": None, "seed": seed}
    state["primals"] = [normal(s) for s in (q_shape, kv_shape, kv_shape)]
    state["tangents"] = [normal(s, case["tangent_std"]) for s in (q_shape, kv_shape, kv_shape)] if case["tangents"] else None
    if case["grads"] in ("o", "both", "all"):
        state["go"] = normal(q_shape)
    if case["grads"] in ("tangent", "both", "all"):
        state["gt"] = normal(q_shape)
    if case["grads"] != "none":
        state["primals"] = [t.requires_grad_(True) for t in state["primals"]]
    if case["grads"] == "all":
        state["tangents"] = [t.requires_grad_(True) for t in state["tangents"]]
    if case["mask"] == "padding":
        lengths = torch.randint((Lk + 1) // 2, Lk + 1, (B, 1, 1, 1), generator=gen, device=device)
        state["mask"] = torch.arange(Lk, device=device) < lengths
    elif case["mask"] == "packed":
        document = (torch.rand(B, Lq, generator=gen, device=device) < DOCUMENTS / Lq).cumsum(1)
        state["mask"] = document[:, None, :, None] == document[:, None, None, :]
    elif case["mask"] == "bias":
        state["mask"] = torch.randn(B, H, Lq, Lk, generator=gen, device=device, dtype=dtype)
    elif case["mask"] == "dense":
        state["mask"] = torch.rand(B, H, Lq, Lk, generator=gen, device=device) < 0.9
    return state


def run(state):
    mask, causal, dropout, grads = state["mask"], state["causal"], state["dropout"], state["grads"]
    q, k, v = state["primals"]
    if dropout:  # a run that can be repeated
        torch.random.default_generator.manual_seed(state["seed"])
    if state["tangents"] is None:
        o = attention(q, k, v, attn_mask=mask, dropout_p=dropout, causal=causal)
        if grads == "none":
            return {"o": o}
        return {"o": o.detach(), "grads": torch.autograd.grad(o, (q, k, v), state["go"])}
    qt, kt, vt = state["tangents"]
    with fwAD.dual_level():
        out = JVPAttn.fwd_dual(fwAD.make_dual(q, qt), fwAD.make_dual(k, kt), fwAD.make_dual(v, vt), attn_mask=mask,
                               dropout_p=dropout, causal=causal)
        o, ot = fwAD.unpack_dual(out)
        if grads == "none":
            return {"o": o, "ot": ot}
        if grads == "o":
            g = torch.autograd.grad(o, (q, k, v), state["go"])
        elif grads == "tangent":
            g = torch.autograd.grad(ot, (q, k, v), state["gt"])
        elif grads == "both":
            g = torch.autograd.grad((o, ot), (q, k, v), (state["go"], state["gt"]))
        else:
            g = torch.autograd.grad((o, ot), (q, k, v, qt, kt, vt), (state["go"], state["gt"]))
        return {"o": o.detach(), "ot": ot.detach(), "grads": g}


def tolerance(case):
    # four times the largest error of any output against the same attention in fp64, over the listed sizes and forty
    # drawn ones: 2.6e-3 in bf16, 3.2e-4 in fp16, 2.1e-6 in fp32 (the longest sums)
    return {"rel": {"bf16": 1e-2, "fp16": 1.3e-3, "fp32": 1e-5}[case["dtype"]]}
