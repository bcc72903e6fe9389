"""Grouped heads in the backward: a group's query heads dealt to several dk/dv workgroups (fp32 shares, then a merge)
against one workgroup visiting them all."""
import ctypes as C

import pytest
import torch

from jvp_flash_attention_amd import _lib

pytestmark = pytest.mark.gpu

KERNELS = [(torch.bfloat16, 32), (torch.bfloat16, 64), (torch.float16, 128), (torch.bfloat16, 256), (torch.float32, 64), (torch.float32, 256)]


def _share_bytes(H, Hk, L, Lk, D, dtype, Z=2, six=False):
    prob = _lib.make_problem(torch.empty(Z, H, L, D, dtype=dtype, device="meta"), None, _lib.MASK_NONE, False, 1.0)
    return _lib.load().jvpfa_bwd_split_workspace_bytes(C.byref(prob), Lk, Hk, int(six))


@pytest.mark.parametrize("dtype,D", KERNELS)
@pytest.mark.parametrize("H", [5, 7])
@pytest.mark.parametrize("mode", ["plain", "six", "padding"])
def test_uneven_shares_agree_with_whole_groups(dtype, D, H, mode):
    """A prime group in shares that differ by a head: 64 key blocks, of which three (four) times as many fill the GPU once."""
    shares = {5: 3, 7: 4}[H]
    assert _share_bytes(H, 1, 70, 4096, D, dtype) == shares * 2 * (2 * 4096 * D) * 4
    test_split_groups_agree_with_whole_ones(dtype, D, H, 1, 70, 4096, mode)


@pytest.mark.parametrize("dtype,D", KERNELS)
def test_shares_are_bounded(dtype, D):
    """Whatever the group: dk and dv of at most 10 workgroups of 128 keys per compute unit, and none where the blocks alone
    fill it."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for H, Hk, Lk, Z in [(71, 1, 2048, 8), (71, 1, 2048, 31), (28, 4, 4096, 2), (64, 1, 128, 1), (13, 1, 100000, 1), (12, 4, 1111, 3)]:
        got = _share_bytes(H, Hk, 1024, Lk, D, dtype, Z)
        assert got <= 10 * cus * 128 * D * 8 and got % (2 * Z * Hk * Lk * D * 4) == 0, (H, Hk, Lk, Z, got)
    assert _share_bytes(28, 4, 1024, 128 * cus, D, dtype) == 0


@pytest.mark.parametrize("dtype,D", KERNELS)
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
