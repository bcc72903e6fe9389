"""Backwards whose dk/dv and dq workgroups share one launch against those that take two: a few heads on their own fill a
fraction of the GPU and go in one; the same heads among many others go in two."""
import pytest
import torch

from jvp_flash_attention_amd import _lib

pytestmark = pytest.mark.gpu

FORMS = [(t, D) for t in (torch.bfloat16, torch.float16, torch.float32) for D in (32, 64, 128, 256) if (t, D) != (torch.float32, 256)]


@pytest.mark.parametrize("dtype,D", FORMS)
@pytest.mark.parametrize("kind", ["none", "causal", "packed mask", "padding", "bias", "grouped", "dropout"])
def test_alone_and_among_others(dtype, D, kind):
    print("case", dtype, D, kind, flush=True)
    L = 520  # 5 blocks of 128 rows a head, the last of 8 rows
    # 20 blocks of either role; 200, which is more than a block of some role to a compute unit and what the capped kernel at D = 64
    # is for; and blocks past every limit on one launch: 2048 in 16 bits at D <= 64 and in fp32 at D = 32; elsewhere a multiple of 256
    # units (then two launches round up to nothing) past 2.5 of them (five heads of 256 columns make 45 blocks of 64 rows)
    few, some, many = 4, 40, 424 if D == 32 or (D == 64 and dtype != torch.float32) else 256
    share = 4 if kind == "grouped" else 1
    g = torch.Generator(device="cuda").manual_seed(D)
    q, qt, go, gt = (torch.randn(1, many, L, D, generator=g, device="cuda").to(dtype) for _ in range(4))
    k, v, kt, vt = (torch.randn(1, many // share, L, D, generator=g, device="cuda").to(dtype) for _ in range(4))
    mask, mk = None, _lib.MASK_NONE
    if kind == "packed mask":
        doc = (torch.rand(1, L, generator=g, device="cuda") < 6 / L).cumsum(1)
        mask, mk = doc[:, None, :, None] == doc[:, None, None, :], _lib.MASK_BOOL
    elif kind == "padding":
        mask, mk = (torch.arange(L, device="cuda") < 411)[None, None, None], _lib.MASK_BOOL
    elif kind == "bias":
        mask, mk = torch.randn(1, 1, L, L, generator=g, device="cuda").to(dtype), _lib.MASK_ADD
    drop = (0.2, 11) if kind == "dropout" else (0.0, 0)
    be, causal, scale = _lib.backend(), kind == "causal", D**-0.5

    def step(n, grads):
        m = n // share
        a = [q[:, :n], k[:, :m], v[:, :m], qt[:, :n], kt[:, :m], vt[:, :m], go[:, :n], gt[:, :n]]
        a = [x.contiguous() for x in a]
        if grads == "plain":
            a[3:6] = [None] * 3
            a[7] = None
        if grads == "tangent":
            a[6] = None
        o, ot, M, mu = be.fwd(*a[:6], mask, mk, causal, scale, *drop)
        return be.bwd(*a[:6], o, ot, M, mu, a[6], a[7], mask, mk, causal, scale, grads == "six", *drop)

    # the same products in the same type, row statistics added in another order at most, O and O' possibly from kernels
    # that split the keys: a rounding of the element type of a term of the row's size here and there
    ulp = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}[dtype]
    for grads in ("plain", "o and tangent", "tangent", "six"):
        print("gradients", grads, flush=True)
        among = step(many, grads)
        _lib.set_split(kind == "grouped")  # (blocks dealt to several workgroups are another kernel's; groups of heads are not)
        try:
            alone = [step(few, grads), step(some, grads)]
        finally:
            _lib.set_split(True)
        for one in alone:
            for name, a, b in zip(("dq", "dk", "dv", "dqt", "dkt", "dvt"), one, among):
                if a is None:
                    continue
                a, b = a.float(), b[:, : a.shape[1]].float()
                assert torch.isfinite(a).all() and ((a - b).norm() <= 2 * ulp * b.norm()).item(), (grads, a.shape[1], name)
