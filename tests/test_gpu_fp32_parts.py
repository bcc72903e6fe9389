"""fp32 attention on the 16-bit matrix instructions (D <= 64: every operand as three bf16 parts)."""
import numpy as np
import pytest
import torch

from jvp_flash_attention_amd import _lib
from oracle import dense, dropout

pytestmark = pytest.mark.gpu

NAMES = ("O", "Ot", "dq", "dk", "dv", "dqt", "dkt", "dvt")


def run(cpu, mask=None, kind=_lib.MASK_NONE, causal=False, drop=(0.0, 0)):
    q, k, v, qt, kt, vt, go, gt = (None if x is None else x.cuda() for x in cpu)
    md = None if mask is None else mask.cuda()
    be = _lib.backend()
    scale = q.shape[-1] ** -0.5
    o, ot, M, mu = be.fwd(q, k, v, qt, kt, vt, md, kind, causal, scale, *drop)
    grads = be.bwd(q, k, v, qt, kt, vt, o, ot, M, mu, go, gt, md, kind, causal, scale, qt is not None, *drop)
    return {n: x.double().cpu().numpy() for n, x in zip(NAMES, (o, ot, *grads)) if x is not None}


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
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("where", ["v", "vt", "k", "go", "gt", "q"])
def test_values_that_have_no_parts(D, bad, where):
    """Infinities and NaN: results are those of fp32 arithmetic on the values themselves."""
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
        if where in ("q", "k") and n not in ("O", "Ot"):
            continue  # (a row without a log-sum-exp takes no part in the backward)
        if n in ("O", "Ot") and where in ("v", "vt"):  # the same columns are not finite, and no others
            assert (np.isfinite(got[n]) == np.isfinite(w)).all(), n
        if (n, where) in (("O", "v"), ("Ot", "vt")):  # ... and the same values stand in them
            assert np.allclose(got[n], w, rtol=1e-4, atol=1e-4, equal_nan=True), n
        ok = np.isfinite(w)
        assert np.allclose(got[n][ok], w[ok], rtol=1e-3, atol=1e-3), n


# a tensor with one entry of 3.4e38 in row 5, and the tensors whose column 3 is zero so that every result stays finite
ALONE = {"q": ("k", "kt"), "k": ("q", "qt"), "v": ("go", "gt"), "qt": ("k",), "kt": ("q",), "vt": ("gt",), "go": ("v",), "gt": ("v", "vt")}


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("where,call", [(w, c) for c in ("dual", "plain", "mask", "causal", "grouped", "dropout") for w in ALONE
                                        if c != "plain" or w in ("q", "k", "v", "go")])
def test_a_finite_value_whose_first_part_is_not(D, where, call):
    """3.4e38 rounds to infinity in bf16, and no result may show it: the sums it has a share in start over with the fp32
    instructions.  Bound: that of fp32 sums (above), column by column."""
    print("case", D, where, call, flush=True)
    names, L, Lk, H = ("q", "k", "v", "qt", "kt", "vt", "go", "gt"), 200, 150, 4 if call == "grouped" else 1
    x = dict(zip(names, inputs(D, L, Lk, H, 1, 9)))
    for n in ("qt", "kt", "vt"):
        x[n] *= 1e-2  # |S'| < 1/4, so that P S' V stays finite
    for n in ("go", "gt"):
        x[n] *= 1e-3  # |dS|, |dS'| < 1/4
    for n in ALONE[where]:
        x[n][..., 3] = 0
    if where in ("v", "vt"):
        x["k"][0, 0, 5] = 0  # a key of small weight: the sums of P V stay finite before they are divided, dropout's factor included
    x[where][0, 0, 5, 3] = 3.4e38
    if call == "plain":
        x["qt"] = x["kt"] = x["vt"] = x["gt"] = None
    mask, kind = None, _lib.MASK_NONE
    if call == "mask":
        mask, kind = torch.rand(1, 1, L, Lk, generator=torch.Generator().manual_seed(3)) < 0.7, _lib.MASK_BOOL
        mask[..., 5] = True
    drop = (0.25, 17) if call == "dropout" else (0.0, 0)
    f = [None if t is None else t.double().numpy() for t in x.values()]
    opts = dict(mask=None if mask is None else mask.numpy(), causal=call == "causal", keep_scale=dropout.keep_scale(1, H, L, Lk, *drop) if drop[0] else None)
    want = {**dense.forward(*f[:6], **opts), **dense.backward(*f, **opts)}
    got = run(list(x.values()), mask, kind, call == "causal", drop)
    assert set(got) == set(NAMES if call != "plain" else ("O", "dq", "dk", "dv"))
    tol = 16 * np.sqrt(L + Lk + D) * 2.0**-24
    for n, a in got.items():
        w = want[n]
        assert np.isfinite(w).all() and np.abs(w).max() < 3.4e38, "the case itself"
        size = 1.0 if n in ("O", "Ot") else 1e-3  # of the terms, where they cancel to nothing
        norms = np.maximum(np.linalg.norm(w, axis=-2), size * np.sqrt(w.shape[-2]))
        assert (np.linalg.norm(a - w, axis=-2) <= tol * norms).all(), n
