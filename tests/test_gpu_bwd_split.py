"""Backwards of small grids, whose blocks are dealt to several workgroups: against the same call unsplit and the dense oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

from jvp_flash_attention_amd import _lib
from oracle import dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("grads", ["plain", "both", "tangent"])
@pytest.mark.parametrize("H,L,Lk,causal", [(1, 1.0, 1.0, False), (2, 1.02, 1.3, False), (1, 0.1, 1.5, False), (1, 1.5, 0.1, False), (2, 1.4, 1.4, True),
                                           (1, 1.05, 1.7, True), (1, 1.7, 0.6, True)])
def test_split_blocks(dtype, D, grads, H, L, Lk, causal):
    # lengths in units of one that is split: 12 tiles into shares of no fewer than 3, 4 or 6
    unit = 64 * 12
    split_or_not(dtype, D, grads, H, max(1, int(unit * L)), max(1, int(unit * Lk)), causal)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("grads", ["both", "tangent"])
@pytest.mark.parametrize("H,L,Lk,causal", [(4, 321, 321, False), (4, 512, 512, False), (16, 512, 512, True), (2, 385, 700, False), (2, 1000, 449, True)])
def test_split_blocks_of_up_to_eight_tiles(dtype, grads, H, L, Lk, causal):
    split_or_not(dtype, 128, grads, H, L, Lk, causal)


def split_or_not(dtype, D, grads, H, L, Lk, causal):
    print("case", dtype, D, grads, H, L, Lk, causal, flush=True)
    g = torch.Generator().manual_seed(L)
    q, qt, go, gt = (torch.randn(1, H, L, D, generator=g).to(dtype) for _ in range(4))
    k, v, kt, vt = (torch.randn(1, H, Lk, D, generator=g).to(dtype) for _ in range(4))
    cpu = [q, k, v, qt, kt, vt, go, gt]
    dev = [x.cuda() for x in cpu]
    if grads == "plain":
        dev[3:6], dev[7] = [None] * 3, None
    if grads == "tangent":
        dev[6] = None
    be, scale = _lib.backend(), D**-0.5
    p = _lib.make_problem(dev[0], None, _lib.MASK_NONE, causal, scale)
    assert _lib.load().jvpfa_bwd_split_workspace_bytes(C.byref(p), Lk, H, 0) > 0
    _lib.set_split(False)
    try:
        o, ot, M, mu = be.fwd(*dev[:6], None, _lib.MASK_NONE, causal, scale)
        one = be.bwd(*dev[:6], o, ot, M, mu, *dev[6:], None, _lib.MASK_NONE, causal, scale)
    finally:
        _lib.set_split(True)
    got = be.bwd(*dev[:6], o, ot, M, mu, *dev[6:], None, _lib.MASK_NONE, causal, scale)
    f = [x.double().numpy() for x in cpu]
    if grads == "plain":
        f[3], f[4], f[5], f[7] = f[3] * 0, f[4] * 0, f[5] * 0, f[7] * 0
    if grads == "tangent":
        f[6] = f[6] * 0
    ref = dense.backward(*f, causal=causal, scale=scale)
    ulp = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for name, a, b in zip(("dq", "dk", "dv"), got, one):
        a, b, want = a.double().cpu().numpy(), b.double().cpu().numpy(), ref[name]
        # fp32 sums in another order, rounded once: one rounding of the element type at most
        assert np.isfinite(a).all() and np.linalg.norm(a - b) <= ulp * np.linalg.norm(b) + 1e-6, name
        assert np.abs(a - want).max() <= 2e-2 * max(np.abs(want).max(), 1.0), name
