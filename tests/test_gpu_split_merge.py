"""Calls whose blocks' tiles are dealt to several workgroups: what is not a number comes out where whole blocks have it, and the workspace is the one in use."""
import ctypes as C

import pytest
import torch

from jvp_flash_attention_amd import _lib

pytestmark = pytest.mark.gpu


def dealt_parts(dev, gs, mask, kind, causal, scale, six=False):
    """Whether the forward and the backward of exactly this call go over blocks that several workgroups share."""
    lib, (q, k, _, qt, _, _) = _lib.load(), dev
    f, b = _lib.FwdArgs(), _lib.BwdArgs()
    for a in (f, b):
        a.struct_size, a.p = C.sizeof(type(a)), _lib.make_problem(q, mask, kind, causal, scale)
        a.Hk, a.Lk = k.shape[1], k.shape[2]
    f.qt = None if qt is None else qt.data_ptr()
    b.gt = None if gs[1] is None else gs[1].data_ptr()
    b.dqt = q.data_ptr() if six else None
    return lib.jvpfa_fwd_split_needed(C.byref(f)) > 0, lib.jvpfa_bwd_split_needed(C.byref(b)) > 0


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
    args = (dev[:6], dev[6:], None, kind, causal, scale)
    assert dealt_parts(*args)[0]
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
    assert dealt_parts(*args)[0]
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


def _fwd_args(dev, o, ot, M, mu, causal, scale):
    a = _lib.FwdArgs()
    a.struct_size = C.sizeof(_lib.FwdArgs)
    a.p = _lib.make_problem(dev[0], None, _lib.MASK_NONE, causal, scale)
    for name, x in zip(("q", "k", "v", "qt", "kt", "vt", "o", "ot", "M", "mu"), (*dev, o, ot, M, mu)):
        setattr(a, name, None if x is None else x.data_ptr())
    a.Hk, a.Lk = dev[1].shape[1], dev[1].shape[2]
    return a


@pytest.mark.parametrize("dtype,D,H,Hk,L,causal", [(torch.float32, 128, 8, 8, 512, False), (torch.float32, 64, 2, 2, 2048, True), (torch.float32, 128, 16, 4, 1024, True),
                                                   (torch.bfloat16, 128, 2, 2, 2048, False), (torch.float16, 64, 3, 3, 3000, True), (torch.bfloat16, 128, 8, 2, 1500, True)])
@pytest.mark.parametrize("dual", [False, True])
def test_a_call_takes_the_workspace_that_it_uses(dtype, D, H, Hk, L, causal, dual):
    """What is asked for is what is written and allocated: nothing behind it, nothing for a call that stays whole, no half for tangents that are not there."""
    print("case", dtype, D, H, Hk, L, causal, dual, flush=True)
    g = torch.Generator().manual_seed(L)
    dev = [torch.randn(1, h, L, D, generator=g).to(dtype).cuda() for h in (H, Hk, Hk, H, Hk, Hk)]
    if not dual:
        dev[3:] = [None] * 3
    be, lib, scale, rows = _lib.backend(), _lib.load(), D**-0.5, H * L
    want = be.fwd(*dev, None, _lib.MASK_NONE, causal, scale)
    outputs = sum(x.numel() * x.element_size() for x in want if x is not None)
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    again = be.fwd(*dev, None, _lib.MASK_NONE, causal, scale)
    taken = torch.cuda.max_memory_allocated() - base - outputs
    slack = 5 << 20  # blocks of the allocator that were not worth splitting, at most 1 MiB each
    if dtype == torch.float32 and Hk != H:
        assert taken <= slack
    a = _fwd_args(dev, *again, causal, scale)
    needed = lib.jvpfa_fwd_split_needed(C.byref(a))
    assert needed % (rows * ((2 if dual else 1) * D + 4) * 4) == 0 and taken <= needed + slack
    assert (needed == 0) == (dtype == torch.float32 and Hk != H)
    assert needed <= lib.jvpfa_fwd_split_workspace_bytes(C.byref(a.p), L)
    if not needed:
        return
    assert needed // (rows * ((2 if dual else 1) * D + 4) * 4) in range(2, 9)
    space = torch.full((needed + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    for x in again:
        if x is not None:
            x.fill_(float("nan"))
    a.split_workspace, a.split_workspace_bytes = space.data_ptr(), needed
    _lib.check(lib.jvpfa_fwd(C.byref(a), torch.cuda.current_stream().cuda_stream))
    assert all(torch.equal(x, y) for x, y in zip(again, want) if y is not None)
    assert (space[needed:] == 0x5A).all() and not (space[:needed] == 0x5A).all()
    a.split_workspace_bytes = needed - 1  # too little: whole blocks
    space.fill_(0x5A)
    _lib.check(lib.jvpfa_fwd(C.byref(a), torch.cuda.current_stream().cuda_stream))
    assert (space == 0x5A).all() and torch.isfinite(again[0]).all()


@pytest.mark.parametrize("dtype,D,H,Hk,L", [(torch.float32, 64, 8, 8, 700), (torch.float32, 128, 8, 2, 512), (torch.bfloat16, 128, 4, 4, 1024), (torch.bfloat16, 64, 3, 3, 3000)])
@pytest.mark.parametrize("grads", ["plain", "both", "six"])
def test_a_backward_takes_the_workspace_that_it_uses(dtype, D, H, Hk, L, grads):
    print("case", dtype, D, H, Hk, L, grads, flush=True)
    g = torch.Generator().manual_seed(L)
    dev = [torch.randn(1, h, L, D, generator=g).to(dtype).cuda() for h in (H, Hk, Hk, H, Hk, Hk, H, H)]
    if grads == "plain":
        dev[3:6], dev[7] = [None] * 3, None
    be, lib, scale = _lib.backend(), _lib.load(), D**-0.5
    o, ot, M, mu = be.fwd(*dev[:6], None, _lib.MASK_NONE, True, scale)
    want = be.bwd(*dev[:6], o, ot, M, mu, *dev[6:], None, _lib.MASK_NONE, True, scale, grads == "six")
    got = [None if x is None else torch.full_like(x, float("nan")) for x in want]
    rows = torch.empty(lib.jvpfa_bwd_workspace_bytes(1, H, L), dtype=torch.uint8, device="cuda")
    a = _lib.BwdArgs()
    a.struct_size = C.sizeof(_lib.BwdArgs)
    a.p = _lib.make_problem(dev[0], None, _lib.MASK_NONE, True, scale)
    names = ("q", "k", "v", "qt", "kt", "vt", "o", "ot", "M", "mu", "go", "gt", "dq", "dk", "dv", "dqt", "dkt", "dvt", "workspace")
    for name, x in zip(names, (*dev[:6], o, ot, M, mu, *dev[6:], *got, rows)):
        setattr(a, name, None if x is None else x.data_ptr())
    a.Hk, a.Lk = Hk, L
    needed = lib.jvpfa_bwd_split_needed(C.byref(a))
    assert needed <= lib.jvpfa_bwd_split_workspace_bytes(C.byref(a.p), L, Hk, int(grads == "six"))
    space = torch.full((needed + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    a.split_workspace, a.split_workspace_bytes = space.data_ptr(), needed
    _lib.check(lib.jvpfa_bwd(C.byref(a), torch.cuda.current_stream().cuda_stream))
    assert all(torch.equal(x, y) for x, y in zip(got, want) if y is not None)
    assert (space[needed:] == 0x5A).all() and (needed == 0 or not (space[:needed] == 0x5A).all())
