"""Causal launches deal their blocks longest first over batches of heads (``xcd_remap``): every block of every head is
worked on exactly once, for head counts around the dealing's limits, against the same scores masked explicitly."""
import pytest
import torch

from jvp_flash_attention_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.bfloat16, 128), (torch.bfloat16, 256), (torch.float32, 32)])
@pytest.mark.parametrize("B,H", [(1, 1), (1, 3), (1, 8), (3, 4), (2, 12), (5, 8), (1, 136), (25, 8)])
@pytest.mark.parametrize("L", [100, 129, 700])
def test_every_block_once(dtype, D, B, H, L):
    print("case", dtype, D, B, H, L, flush=True)
    g = torch.Generator(device="cuda").manual_seed(B * H + L)
    q, k, v, qt, kt, vt, go, gt = (torch.randn(B, H, L, D, generator=g, device="cuda").to(dtype) for _ in range(8))
    mask = torch.ones(L, L, dtype=torch.bool, device="cuda").tril()[None, None]
    be = _lib.backend()

    def step(m, kind, causal):
        o, ot, M, mu = be.fwd(q, k, v, qt, kt, vt, m, kind, causal, D**-0.5)
        return (o, ot, M, mu, *be.bwd(q, k, v, qt, kt, vt, o, ot, M, mu, go, gt, m, kind, causal, D**-0.5)[:3])

    for name, a, b in zip(("O", "Ot", "M", "mu", "dq", "dk", "dv"), step(None, _lib.MASK_NONE, True), step(mask, _lib.MASK_BOOL, False)):
        # same products, possibly other kernels and reference points: the repository's bars for one element type
        bar = 2e-2 if dtype != torch.float32 else 1e-4
        a, b = a.double(), b.double()
        scale = b.abs().amax(dim=tuple(range(2, b.dim())), keepdim=True).clamp_min(1.0)  # per head: a block left out shows
        assert torch.isfinite(a).all() and ((a - b).abs() <= bar * scale).all(), name
