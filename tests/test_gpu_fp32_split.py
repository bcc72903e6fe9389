"""fp32 calls whose blocks' tiles are dealt to several workgroups: against the same calls on whole blocks and the dense oracle."""
import numpy as np
import pytest
import torch

from jvp_flash_attention_amd import _lib
from oracle import dense

from .test_gpu_split_merge import dealt_parts

pytestmark = pytest.mark.gpu


def _mask(kind, Z, H, L, Lk, g):
    if kind == "padding":
        return torch.arange(Lk) < torch.tensor([1, Lk // 3, Lk][:Z]).view(Z, 1, 1, 1), _lib.MASK_BOOL
    if kind == "documents":  # tiles that hold nothing, and key tiles of a share that nothing in it attends to
        d = (torch.arange(L) * 3 // L)[:, None] == (torch.arange(Lk) * 3 // Lk)[None, :]
        return d.expand(Z, 1, L, Lk).contiguous(), _lib.MASK_BOOL
    if kind == "bias":
        return torch.randn(Z, H, L, Lk, generator=g), _lib.MASK_ADD
    return None, _lib.MASK_NONE


def _step(dev, gs, mask, kind, causal, scale, six):
    be = _lib.backend()
    o, ot, M, mu = be.fwd(*dev, mask, kind, causal, scale)
    grads = be.bwd(*dev, o, ot, M, mu, *gs, mask, kind, causal, scale, six)
    return [o, ot, M, mu, *grads]


# ends inside tiles and blocks; more shares than some blocks have tiles; blocks of one tile; keys that no query sees; rows of a bias
# that are and are not on 16-byte boundaries
SHAPES = [(1, 2, 900, 900, "causal"), (2, 3, 130, 2000, "none"), (1, 2, 2000, 130, "none"), (1, 2, 1100, 2000, "causal"), (1, 3, 1400, 400, "causal"),
          (3, 2, 1025, 1025, "padding"), (2, 2, 1200, 1104, "documents"), (1, 2, 1040, 1040, "bias"), (1, 2, 1033, 901, "bias"), (1, 1, 3300, 3300, "causal")]


# ... of which stay whole, as too short to be worth another launch on 256 compute units: head dim, queries, keys, tangents
WHOLE_FORWARDS = {(D, 2000, 130, dual) for D in (32, 64, 128) for dual in (False, True)} - {(128, 2000, 130, True)}
WHOLE_FORWARDS |= {(32, 1400, 400, True), (32, 1400, 400, False), (64, 1400, 400, False)}
WHOLE_BACKWARDS = {(32, *n, False) for n in ((900, 900), (1100, 2000), (1025, 1025), (1200, 1104), (1040, 1040), (1033, 901))}
WHOLE_FORWARDS |= WHOLE_BACKWARDS


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Z,H,L,Lk,kind", SHAPES)
@pytest.mark.parametrize("grads", ["plain", "both", "tangent", "six"])
def test_dealt_tiles_agree_with_whole_blocks(D, Z, H, L, Lk, kind, grads):
    print("case", D, Z, H, L, Lk, kind, grads, flush=True)
    g = torch.Generator().manual_seed(L + Lk + D)
    cpu = [torch.randn(Z, H, n, D, generator=g) for n in (L, Lk, Lk, L, Lk, Lk, L, L)]
    mask, mk = _mask(kind, Z, H, L, Lk, g)
    dev = [x.cuda() for x in cpu]
    scale, causal = D**-0.5, kind == "causal"
    if grads == "plain":
        dev[3:6], dev[7] = [None] * 3, None
    if grads == "tangent":
        dev[6] = None
    dmask = None if mask is None else mask.cuda()
    args = (dev[:6], dev[6:], dmask, mk, causal, scale, grads == "six")
    what = (D, L, Lk, grads != "plain")
    assert dealt_parts(*args) == (what not in WHOLE_FORWARDS, what not in WHOLE_BACKWARDS)
    got = _step(*args)
    _lib.set_split(False)
    try:
        one = _step(*args)
    finally:
        _lib.set_split(True)
    f = [x.double().numpy() for x in cpu]
    if grads == "plain":
        f[3], f[4], f[5], f[7] = f[3] * 0, f[4] * 0, f[5] * 0, f[7] * 0
    if grads == "tangent":
        f[6] = f[6] * 0
    m = None if mask is None else mask.numpy()
    want = dense.forward(*f[:6], mask=m, causal=causal, scale=scale)
    back = dense.backward(*f, mask=m, causal=causal, scale=scale)
    refs = [want["O"], want["Ot"], None, None, *(back[n] for n in ("dq", "dk", "dv", "dqt", "dkt", "dvt"))]
    for i, (a, b, w) in enumerate(zip(got, one, refs)):
        if a is None:
            continue
        a, b = a.double().cpu().numpy(), b.double().cpu().numpy()
        alive = np.isfinite(b)  # (M of a row without keys)
        assert np.array_equal(alive, np.isfinite(a)), i
        a, b = a[alive], b[alive]
        assert np.abs(a - b).max() <= 1e-5 * max(1.0, np.abs(b).max()), i  # sums of up to 3300 terms in another order: a few units of 2^-24 of a term each
        if w is not None:
            assert np.abs(a - w[alive]).max() <= 1e-4 * max(1.0, np.abs(w).max() / 8), i


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("kind", ["documents", "padding"])
def test_shares_do_not_depend_on_what_is_skipped(D, kind):
    """The same mask with and without tile lists and a key limit: not a bit changes."""
    Z, H, L, Lk = 2, 2, 600, 700
    g = torch.Generator().manual_seed(3)
    dev = [torch.randn(Z, H, n, D, generator=g).cuda() for n in (L, Lk, Lk, L, Lk, Lk, L, L)]
    mask, mk = _mask(kind, Z, H, L, Lk, g)
    full = mask.expand(Z, 1, L, Lk).contiguous().cuda()
    runs = []
    for m, lists in ((full, True), (full.clone(), False), (mask.cuda(), True)):
        _lib.set_tile_lists(lists)
        try:
            runs.append(_step(dev[:6], dev[6:], m, mk, False, D**-0.5, True))
        finally:
            _lib.set_tile_lists(True)
    for other in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(runs[0], other))


@pytest.mark.parametrize("D", [64, 128])
def test_infinities_stay_where_they_are(D):
    """An infinite value and a not-a-number, in a split call: the same outputs are not finite as on whole blocks, and the others agree."""
    L = 700
    g = torch.Generator().manual_seed(5)
    dev = [torch.randn(1, 2, L, D, generator=g).cuda() for _ in range(8)]
    dev[2][0, 0, 400, 3] = float("inf")
    dev[4][0, 1, 10, 0] = float("nan")
    runs = []
    for on in (True, False):
        _lib.set_split(on)
        try:
            runs.append(_step(dev[:6], dev[6:], None, _lib.MASK_NONE, True, D**-0.5, False))
        finally:
            _lib.set_split(True)
    for a, b in zip(*runs):
        if a is None:
            continue
        fa, fb = torch.isfinite(a), torch.isfinite(b)
        assert torch.equal(fa, fb)
        if fa.any():
            assert (a[fa] - b[fa]).abs().max().item() <= 1e-5 * max(1.0, b[fb].abs().max().item())
