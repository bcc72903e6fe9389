"""The pipelined forward at D = 64: rows around its shortest length, tile ends, and keys split over workgroups."""
import numpy as np
import pytest
import torch

from jvp_flash_attention_amd import _lib
from oracle import dense

from .test_gpu_split_merge import dealt_parts

pytestmark = pytest.mark.gpu

TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def run(dt, Z, H, Hk, L, Lk, causal, dual, scale=0.125):
    print("case", dt, Z, H, Hk, L, Lk, causal, dual, flush=True)
    g = torch.Generator().manual_seed(L + Lk)
    q, qt = (torch.randn(Z, H, L, 64, generator=g).to(TYPES[dt]) for _ in range(2))
    k, v, kt, vt = (torch.randn(Z, Hk, Lk, 64, generator=g).to(TYPES[dt]) for _ in range(4))
    cpu = [q, k, v] + ([qt, kt, vt] if dual else [])
    dev = [x.cuda() for x in cpu] + [None] * (6 - len(cpu))
    ref = dense.forward(*(x.double().numpy() for x in cpu), causal=causal, scale=scale)
    return dev, ref, _lib.backend().fwd(*dev, None, _lib.MASK_NONE, causal, scale)


def check(got, ref, dual):
    for name, x in (("O", got[0]), ("Ot", got[1])) if dual else (("O", got[0]),):
        err = np.abs(x.double().cpu().numpy() - ref[name]).max()
        assert err <= 2e-2 * np.abs(ref[name]).max(), (name, err)
    assert np.abs(got[2].double().cpu().numpy() - ref["M"]).max() < 1e-4 * max(1.0, np.abs(ref["M"]).max())
    if dual:
        assert np.abs(got[3].double().cpu().numpy() - ref["mu"]).max() < 1e-4 * max(1.0, np.abs(ref["mu"]).max())


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("L,Lk,causal", [(1, 511, False), (1, 512, False), (130, 513, False), (129, 543, False), (33, 545, False), (512, 575, True),
                                         (577, 577, True), (640, 640, True), (700, 512, True)])
def test_tile_ends(dt, L, Lk, causal):
    for scale in (0.125, -0.3):
        _, ref, got = run(dt, 2, 18, 9, L, Lk, causal, True, scale) if L < 200 else run(dt, 3, 16, 16, L, Lk, causal, True, scale)
        check(got, ref, True)


@pytest.mark.parametrize("dual", [True, False])
@pytest.mark.parametrize("Z,H,Hk,L,Lk,causal", [(1, 1, 1, 1000, 1024, False), (1, 2, 1, 300, 1025, False), (1, 2, 2, 2100, 2100, True), (2, 1, 1, 64, 4100, False)])
def test_keys_split_over_workgroups(dual, Z, H, Hk, L, Lk, causal):
    dev, ref, got = run("bf16", Z, H, Hk, L, Lk, causal, dual)
    check(got, ref, dual)
    assert dealt_parts(dev, (None, None), None, _lib.MASK_NONE, causal, 0.125)[0] == (dual or Lk >= 32 * 64)  # (short calls without tangents stay whole)
    _lib.set_split(False)
    try:
        one = _lib.backend().fwd(*dev, None, _lib.MASK_NONE, causal, 0.125)
    finally:
        _lib.set_split(True)
    assert (got[2] - one[2]).abs().max().item() <= 1e-5
    for a, b in zip(got[:2], one[:2]):
        if a is not None:  # one rounding of the element type apart
            assert ((a.float() - b.float()).abs() <= 2 * 2.0**-7 * b.float().abs().clamp_min(1.0)).all()
