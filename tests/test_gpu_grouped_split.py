"""Grouped heads in the backward: a group's query heads dealt to several dk/dv workgroups (fp32 shares, then a merge)
against one workgroup visiting them all."""
import pytest
import torch

from jvp_flash_attention_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 32), (torch.bfloat16, 64), (torch.float16, 128), (torch.bfloat16, 256),
                                     (torch.float32, 64), (torch.float32, 256)])
@pytest.mark.parametrize("H,Hk,L,Lk", [(6, 2, 65, 65), (4, 1, 200, 129), (12, 2, 33, 300)])
@pytest.mark.parametrize("mode", ["plain", "dual", "six", "padding", "dropout"])
def test_split_groups_agree_with_whole_ones(dtype, D, H, Hk, L, Lk, mode):
    print("case", dtype, D, H, Hk, L, Lk, mode, flush=True)
    g = torch.Generator(device="cuda").manual_seed(D + H + L)
    rand = lambda h, n: torch.randn(2, h, n, D, generator=g, device="cuda").to(dtype)  # noqa: E731
    q, k, v, qt, kt, vt = rand(H, L), rand(Hk, Lk), rand(Hk, Lk), rand(H, L), rand(Hk, Lk), rand(Hk, Lk)
    go, gt = rand(H, L), rand(H, L)
    mask, kind = None, _lib.MASK_NONE
    if mode == "padding":
        kind = _lib.MASK_BOOL
        mask = torch.arange(Lk, device="cuda") < torch.tensor([Lk, Lk // 2], device="cuda").view(2, 1, 1, 1)
    drop = dict(dropout_p=0.25, dropout_seed=5) if mode == "dropout" else {}
    dual = mode != "plain"
    be = _lib.backend()
    tangents = (qt, kt, vt) if dual else (None,) * 3
    o, ot, M, mu = be.fwd(q, k, v, *tangents, mask, kind, False, D**-0.5, **drop)

    def grads():
        return be.bwd(q, k, v, *tangents, o, ot, M, mu, go, gt if dual else None, mask, kind, False, D**-0.5,
                      want_tangent_grads=mode in ("six", "dropout"), **drop)

    _lib.set_split(False)
    try:
        want = grads()
    finally:
        _lib.set_split(True)
    got = grads()
    # both add the same fp32 products in another order and round once, so an entry may round to the neighbouring value:
    # a spacing of at most 2^-7 of the entry in bf16 and 2^-10 in fp16 (7 and 10 fraction bits).  In fp32 the order itself
    # is what is left: up to n = 2 x 4 heads x 200 queries additions round partial sums of the result's size, an error of
    # sqrt(n) 2^-24 = 2.4e-6 on either side, 3.4e-6 for the difference; three times that is allowed.
    bar = {torch.bfloat16: 2**-7, torch.float16: 2**-10, torch.float32: 1e-5}[dtype]
    for name, a, b in zip(("dq", "dk", "dv", "dqt", "dkt", "dvt"), got, want):
        if b is None:
            continue
        a, b = a.double(), b.double()
        assert torch.isfinite(a).all() and (a - b).abs().max() <= bar * b.abs().max(), name
