"""Backwards whose dk/dv and dq workgroups share one launch against those that take two: a few heads on their own fill a
fraction of the GPU and go in one; the same heads among many others go in two."""
import pytest
import torch

from jvp_flash_attention_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("grads", ["plain", "o and tangent", "tangent", "six"])
@pytest.mark.parametrize("kind", ["none", "causal", "packed mask", "padding", "grouped", "dropout"])
def test_alone_and_among_others(dtype, D, grads, kind):
    print("case", dtype, D, grads, kind, flush=True)
    few, L = 4, 520  # 5 blocks of 128 rows a head, the last of 8 rows
    # blocks past every limit on one launch: 2048 at D <= 64; elsewhere a multiple of 256 units (then two launches round up to
    # nothing) past 2.5 of them (five heads of 256 columns make 45 blocks of 64 rows)
    many = 424 if D <= 64 else 256
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
    drop = (0.2, 11) if kind == "dropout" else (0.0, 0)
    be, causal, scale = _lib.backend(), kind == "causal", D**-0.5

    def step(n):
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

    for name, alone, among in zip(("dq", "dk", "dv", "dqt", "dkt", "dvt"), step(few), step(many)):
        if alone is None:
            continue
        a, b = alone.float(), among[:, : alone.shape[1]].float()
        # the same products in the same type, row statistics added in another order at most, O and O' possibly from kernels
        # that split the keys: a rounding of the element type of a term of the row's size here and there
        ulp = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
        assert torch.isfinite(a).all() and ((a - b).norm() <= 2 * ulp * b.norm()).item(), name
