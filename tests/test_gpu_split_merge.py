"""Forwards whose blocks' keys are dealt to several workgroups: what is not a number comes out where whole blocks have it."""
import ctypes as C

import pytest
import torch

from jvp_flash_attention_amd import _lib

pytestmark = pytest.mark.gpu


def _step(dev, gs, mask, kind, causal, scale):
    be = _lib.backend()
    o, ot, M, mu = be.fwd(*dev, mask, kind, causal, scale)
    return [o, ot, M, mu, *be.bwd(*dev, o, ot, M, mu, *gs, mask, kind, causal, scale)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("where", ["row", "queries", "keys of a share", "tangent keys", "last value", "infinite key", "everything"])
@pytest.mark.parametrize("causal", [False, True])
def test_what_is_not_a_number_stays_where_it_is(dtype, D, dual, where, causal):
    """A share whose scores are all NaN has no reference point to be weighed by; its row is NaN all the same."""
    print("case", dtype, D, dual, where, causal, flush=True)
    H, L = 2, 2048
    g = torch.Generator().manual_seed(11)
    dev = [torch.randn(1, H, L, D, generator=g).to(dtype).cuda() for _ in range(8)]
    nan = float("nan")
    if where == "row":
        dev[0][0, 1, 1500] = nan
    elif where == "queries":
        dev[0][0, 0] = nan
    elif where == "keys of a share":  # in eight shares or fewer: at least one whole share
        dev[1][0, 0, 512:1536] = nan
    elif where == "tangent keys":
        dev[4][0, 0, 512:1536] = nan
    elif where == "last value":  # rows before it weigh it by an exact zero
        dev[2][0, 0, L - 1] = nan
    elif where == "infinite key":
        dev[1][0, 0, 700, 3] = float("inf")
    else:
        for x in dev[:6]:
            x.fill_(nan)
    if not dual:
        dev[3:6], dev[7] = [None] * 3, None
    kind, scale = _lib.MASK_NONE, D**-0.5
    p = _lib.make_problem(dev[0], None, kind, causal, scale)
    assert _lib.load().jvpfa_fwd_split_workspace_bytes(C.byref(p), L) > 0
    args = (dev[:6], dev[6:], None, kind, causal, scale)
    got = _step(*args)
    _lib.set_split(False)
    try:
        whole = _step(*args)
    finally:
        _lib.set_split(True)
    # P of 16 bits is rounded against another reference point in each share
    near = 1e-5 if dtype == torch.float32 else 2.0**-7 if dtype == torch.bfloat16 else 2.0**-10
    for i, (a, b) in enumerate(zip(got, whole)):
        if a is None:
            continue
        alive = torch.isfinite(b)
        assert torch.equal(alive, torch.isfinite(a)), i
        assert torch.equal(torch.isnan(a), torch.isnan(b)), i
        assert (a[alive].float() - b[alive].float()).norm() <= near * b[alive].float().norm(), i


@pytest.mark.parametrize("D", [64, 128])
def test_masked_shares_of_values_that_are_not_numbers(D):
    """fp32 under a boolean mask: shares that visit nothing hold no values, and shares whose visited keys are all masked hold 0 * NaN."""
    Z, H, L = 2, 2, 1024
    g = torch.Generator().manual_seed(12)
    dev = [torch.randn(Z, H, L, D, generator=g).cuda() for _ in range(8)]
    mask = torch.zeros(Z, 1, L, L, dtype=torch.bool)
    mask[0, :, :, :200] = True  # the last shares visit nothing
    mask[1] = (torch.arange(L) // 300)[:, None] == (torch.arange(L) // 300)[None, :]
    dev[2][0, 0, 250] = float("nan")  # in a tile that is visited, masked in all rows
    dev[2][1, 1, 600] = float("nan")
    dev[1][0, 1, 900] = float("nan")  # in a tile that no row visits
    args = (dev[:6], dev[6:], mask.cuda(), _lib.MASK_BOOL, False, D**-0.5)
    p = _lib.make_problem(dev[0], args[2], _lib.MASK_BOOL, False, D**-0.5)
    assert _lib.load().jvpfa_fwd_split_workspace_bytes(C.byref(p), L) > 0
    got = _step(*args)
    _lib.set_split(False)
    try:
        whole = _step(*args)
    finally:
        _lib.set_split(True)
    for i, (a, b) in enumerate(zip(got, whole)):
        if a is None:
            continue
        alive = torch.isfinite(b)
        assert torch.equal(alive, torch.isfinite(a)) and torch.equal(torch.isnan(a), torch.isnan(b)), i
        assert (a[alive] - b[alive]).norm() <= 1e-5 * b[alive].norm(), i
