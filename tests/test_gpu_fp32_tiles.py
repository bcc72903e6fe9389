"""fp32 kernels at the edges of their 32-row tiles and 128-row blocks, against the dense oracle."""
import numpy as np
import pytest
import torch

from jvp_flash_attention_amd import _lib
from oracle import dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("L,Lk", [(1, 1), (31, 33), (32, 32), (33, 31), (127, 129), (128, 64), (129, 96), (160, 255)])
@pytest.mark.parametrize("mask", ["none", "causal", "bool", "bias"])
def test_tile_edges(D, L, Lk, mask):
    print("case", D, L, Lk, mask, flush=True)
    g = torch.Generator().manual_seed(1000 * D + L)
    rand = lambda n: torch.randn(1, 2, n, D, generator=g)  # noqa: E731
    cpu = [rand(L), rand(Lk), rand(Lk), rand(L), rand(Lk), rand(Lk), rand(L), rand(L)]
    m, kind = None, _lib.MASK_NONE
    if mask == "bool":
        m, kind = torch.rand(1, 2, L, Lk, generator=g) < 0.7, _lib.MASK_BOOL
        m[..., 0] = True
    elif mask == "bias":
        m, kind = torch.randn(1, 1, L, Lk, generator=g), _lib.MASK_ADD
    f = [x.double().numpy() for x in cpu]
    opts = dict(mask=None if m is None else (m.numpy() if kind == _lib.MASK_BOOL else m.double().numpy()), causal=mask == "causal")
    fwd, bwd = dense.forward(*f[:6], **opts), dense.backward(*f, **opts)
    q, k, v, qt, kt, vt, go, gt = (x.cuda() for x in cpu)
    md = None if m is None else m.cuda()
    be = _lib.backend()
    o, ot, M, mu = be.fwd(q, k, v, qt, kt, vt, md, kind, mask == "causal", D**-0.5)
    six = be.bwd(q, k, v, qt, kt, vt, o, ot, M, mu, go, gt, md, kind, mask == "causal", D**-0.5, True)
    for name, got, want in (("O", o, fwd["O"]), ("Ot", ot, fwd["Ot"]), *zip(("dq", "dk", "dv", "dqt", "dkt", "dvt"), six, (bwd[n] for n in ("dq", "dk", "dv", "dqt", "dkt", "dvt")))):
        # the repository's fp32 bar, relative where the quantity is larger than one
        assert np.abs(got.double().cpu().numpy() - want).max() <= 1e-4 * max(1.0, np.abs(want).max()), name


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("grads", ["plain", "six"])
@pytest.mark.parametrize("first,row", [(0, 255), (1, 256), (2, 257), (3, 258), (1, 259)])
def test_bias_rows_wherever_they_start(D, grads, first, row):
    """Vector loads of a bias take rows and planes at any element: the same bits as from rows on 16-byte boundaries."""
    print("case", D, grads, first, row, flush=True)
    L, Lk, H = 131, 255, 2
    g = torch.Generator(device="cuda").manual_seed(D)
    rand = lambda n: torch.randn(1, H, n, D, generator=g, device="cuda")  # noqa: E731
    a = [rand(L), rand(Lk), rand(Lk), rand(L), rand(Lk), rand(Lk), rand(L), rand(L)]
    if grads == "plain":
        a[3:6], a[7] = [None] * 3, None
    bias = torch.randn(1, H, L, Lk, generator=g, device="cuda")
    be = _lib.backend()

    def step(first, row):
        flat = torch.full((first + H * L * row,), float("nan"), device="cuda")
        mask = flat[first:].as_strided((1, H, L, Lk), (H * L * row, L * row, row, 1))
        mask.copy_(bias)
        o, ot, M, mu = be.fwd(*a[:6], mask, _lib.MASK_ADD, False, D**-0.5)
        return o, ot, *be.bwd(*a[:6], o, ot, M, mu, *a[6:], mask, _lib.MASK_ADD, False, D**-0.5, grads == "six")

    for x, y in zip(step(first, row), step(0, 256)):
        assert x is y is None or torch.equal(x, y)


def test_key_rows_past_32_bits_of_bytes():
    """One query over 2^23 + 70 keys of 512 bytes: one of the first keys, then the last, has a logit of 64, all others 0, and so
    all the weight but e^-64 each.  The exponent 64 log2(e) = 92 is rounded to 92 * 2^-24 on either side of its difference
    with the row's log-sum-exp, so the weight is 1 within 2 * 92 * 2^-24 * ln 2 < 1e-5."""
    D, Lk = 128, 2**23 + 70
    q = torch.zeros(1, 1, 1, D, device="cuda")
    q[..., 0] = 8.0
    k = torch.zeros(1, 1, Lk, D, device="cuda")
    v = torch.zeros_like(k)
    be = _lib.backend()
    for at in (84, Lk - 1):  # 84: in the tile from whose start 2^23 + 6 rows follow
        k[0, 0, at, 0] = 8.0
        v[0, 0, at] = 1.0 + torch.arange(D, device="cuda") / D
        o, _, M, _ = be.fwd(q, k, v, None, None, None, None, _lib.MASK_NONE, False, 1.0)
        assert (o[0, 0, 0] / v[0, 0, at] - 1).abs().max() <= 1e-5
        go = torch.ones_like(q)
        dq, _, dv = be.bwd(q, k, v, None, None, None, o, None, M, None, go, None, None, _lib.MASK_NONE, False, 1.0)[:3]
        assert (dv[0, 0, at] - 1).abs().max() <= 1e-5
        assert dq.abs().max() <= 1e-5 * 8 * 192  # P (gO V - rowsum gO O) K: both of the difference are 192 times the weight
        dv[0, 0, at] = 0
        assert dv.abs().max() <= 1e-20
        k[0, 0, at], v[0, 0, at] = 0, 0
