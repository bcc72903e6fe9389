"""fp32 attention on the 16-bit matrix instructions (D <= 64: every operand as three bf16 parts)."""
import numpy as np
import pytest
import torch

from jvp_flash_attention_amd import _lib
from oracle import dense

pytestmark = pytest.mark.gpu

NAMES = ("O", "Ot", "dq", "dk", "dv", "dqt", "dkt", "dvt")


def run(cpu, mask=None, kind=_lib.MASK_NONE, causal=False):
    q, k, v, qt, kt, vt, go, gt = (x.cuda() for x in cpu)
    md = None if mask is None else mask.cuda()
    be = _lib.backend()
    scale = q.shape[-1] ** -0.5
    o, ot, M, mu = be.fwd(q, k, v, qt, kt, vt, md, kind, causal, scale)
    six = be.bwd(q, k, v, qt, kt, vt, o, ot, M, mu, go, gt, md, kind, causal, scale, True)
    return dict(zip(NAMES, (x.double().cpu().numpy() for x in (o, ot, *six))))


def inputs(D, L, Lk, H, Hk, seed):
    g = torch.Generator().manual_seed(seed)
    q, k = lambda: torch.randn(1, H, L, D, generator=g), lambda: torch.randn(1, Hk, Lk, D, generator=g)  # noqa: E731
    return [q(), k(), k(), q(), k(), k(), q(), q()]


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("L,Lk,Hk", [(1, 1, 2), (1, 65, 2), (40, 31, 2), (97, 64, 1), (129, 95, 2), (160, 161, 1), (260, 260, 2), (65, 700, 1)])
@pytest.mark.parametrize("mask", ["none", "causal", "bool", "bias"])
def test_error_is_that_of_fp32_sums(D, L, Lk, Hk, mask):
    """Sums of n fp32 products are off by about sqrt(n) 2^-24 in the 2-norm.  A result is behind at most three such sums (its
    own over L or Lk, a row statistic over Lk, a score over D), each amplified by at most the few units of spread of the scores:
    16 sqrt(L + Lk + D) 2^-24.  A part left out of a product is an error of 2^-17 or 2^-9."""
    print("case", D, L, Lk, Hk, mask, flush=True)
    cpu = inputs(D, L, Lk, 2, Hk, 100 * D + L)
    g = torch.Generator().manual_seed(L)
    m, kind = None, _lib.MASK_NONE
    if mask == "bool":
        m, kind = torch.rand(1, 2, L, Lk, generator=g) < 0.7, _lib.MASK_BOOL
        m[..., 0] = True
    elif mask == "bias":
        m, kind = torch.randn(1, 2, L, Lk, generator=g), _lib.MASK_ADD
    f = [x.double().numpy() for x in cpu]
    opts = dict(mask=None if m is None else (m.numpy() if kind == _lib.MASK_BOOL else m.double().numpy()), causal=mask == "causal")
    want = {**dense.forward(*f[:6], **opts), **dense.backward(*f, **opts)}
    got = run(cpu, m, kind, mask == "causal")
    tol = 16 * np.sqrt(L + Lk + D) * 2.0**-24
    for n in NAMES:
        # (a gradient that cancels to nothing, as dq where a row has one key, is held to the terms it is the sum of: of size one)
        norm = max(np.linalg.norm(want[n]), np.sqrt(want[n].size))
        assert np.linalg.norm(got[n] - want[n]) <= tol * norm, n


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("where", ["v", "vt", "k", "go", "gt", "q"])
def test_values_that_have_no_parts(D, bad, where):
    """Infinities, NaN and what rounds to infinity: results are those of fp32 arithmetic on the values themselves."""
    print("case", D, bad, where, flush=True)
    L, Lk = 200, 150
    cpu = inputs(D, L, Lk, 1, 1, 7)
    i = ("q", "k", "v", "qt", "kt", "vt", "go", "gt").index(where)
    cpu[i][0, 0, 5, 3] = bad
    f = [x.double().numpy() for x in cpu]
    with np.errstate(all="ignore"):
        want = {**dense.forward(*f[:6]), **dense.backward(*f)}
    got = run(cpu)
    for n in NAMES:
        w = want[n]
        if bad == 3.4e38 and (n, where) != ("O", "v"):
            continue  # the other quantities are sums that pass the largest fp32 value on their way
        if where in ("q", "k") and n not in ("O", "Ot"):
            continue  # (a row without a log-sum-exp takes no part in the backward)
        if n in ("O", "Ot") and where in ("v", "vt"):  # the same columns are not finite, and no others
            assert (np.isfinite(got[n]) == np.isfinite(w)).all(), n
        if (n, where) in (("O", "v"), ("Ot", "vt")):  # ... and the same values stand in them
            assert np.allclose(got[n], w, rtol=1e-4, atol=1e-4, equal_nan=True), n
        ok = np.isfinite(w)
        assert np.allclose(got[n][ok], w[ok], rtol=1e-3, atol=1e-3), n
