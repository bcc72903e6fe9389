"""One pass over a boolean mask (``jvpfa_mask_scan``) against numpy, and the forward and dq kernels on its packed copy
against the same kernels on the mask's bytes."""
import numpy as np
import pytest
import torch

from jvp_flash_attention_amd import _lib, attention

pytestmark = pytest.mark.gpu


def _mask(shape, seed, strided=False):
    g = torch.Generator().manual_seed(seed)
    m = torch.rand(shape, generator=g) < 0.02
    m[..., : shape[2] // 3, shape[3] // 2:] = False  # tiles that hold nothing
    m = m.cuda()
    return m.transpose(2, 3).contiguous().transpose(2, 3) if strided else m


@pytest.mark.parametrize("Lq,Lk", [(512, 64), (1, 513), (577, 577), (640, 63), (100, 1000)])
@pytest.mark.parametrize("planes", [(2, 3), (2, 1), (1, 1)])
@pytest.mark.parametrize("strided", [False, True])
def test_scan_matches_numpy(Lq, Lk, planes, strided):
    print("case", Lq, Lk, planes, strided, flush=True)
    mask = _mask((*planes, Lq, Lk), Lq + Lk, strided)
    mask[0, 0] = False  # a plane that attends to nothing
    q = torch.empty(2, 3, Lq, 64, dtype=torch.bfloat16, device="cuda")
    scan = _lib.mask_scan(q, mask, _lib.MASK_BOOL, Lk)
    m = mask.reshape(-1, Lq, Lk).cpu().numpy()
    nqt, nkt = -(-Lq // 64), -(-Lk // 64)
    full = np.zeros((m.shape[0], 64 * nqt, 64 * nkt), bool)
    full[:, :Lq, :Lk] = m
    tiles = full.reshape(-1, nqt, 64, nkt, 64).any((2, 4))
    assert np.array_equal(scan.attends.cpu().numpy(), m.any((1, 2)).astype(np.int32))
    # words: 32 entries along the packed axis, entry i in bit i
    weights = (1 << np.arange(32, dtype=np.uint64)).astype(np.uint64)
    words_q = (full.reshape(-1, 64 * nqt, nkt, 2, 32).astype(np.uint64) @ weights)[:, :Lq].transpose(0, 2, 1, 3)
    words_k = (full.reshape(-1, nqt, 2, 32, 64 * nkt).transpose(0, 1, 4, 2, 3).astype(np.uint64) @ weights)[:, :, :Lk]
    assert np.array_equal(scan.bits_q.cpu().numpy().view(np.uint32).astype(np.uint64), words_q.reshape(-1))
    assert np.array_equal(scan.bits_k.cpu().numpy().view(np.uint32).astype(np.uint64), words_k.reshape(-1))
    for got, t in ((scan.tiles_q, tiles), (scan.tiles_k, tiles.transpose(0, 2, 1))):
        pad = t.shape[1] % 2
        owned = np.pad(t, ((0, 0), (0, pad), (0, 0))).reshape(t.shape[0], -1, 2, t.shape[2]).any(2)
        got = got.cpu().numpy().reshape(owned.shape[0], owned.shape[1], owned.shape[2] + 1)
        for p in range(owned.shape[0]):
            for b in range(owned.shape[1]):
                want = np.flatnonzero(owned[p, b]) if owned[p, b].any() else np.array([0])
                assert got[p, b, 0] == len(want) and np.array_equal(got[p, b, 1: 1 + len(want)], want)


def _compare(dtype, D, Z, H, Hk, Lq, Lk, dual, with_go=True, six=None):
    """Every output of a step, from the packed copies and from the mask's bytes."""
    g = torch.Generator(device="cuda").manual_seed(D + Lq)
    rand = lambda h, n: torch.randn(Z, h, n, D, generator=g, device="cuda").to(dtype)  # noqa: E731
    q, k, v, qt, kt, vt, go, gt = rand(H, Lq), rand(Hk, Lk), rand(Hk, Lk), rand(H, Lq), rand(Hk, Lk), rand(Hk, Lk), rand(H, Lq), rand(H, Lq)
    mask = torch.rand(Z, H, Lq, Lk, generator=g, device="cuda") < 0.7
    be = _lib.backend()

    def step(m):
        t = (qt, kt, vt) if dual else (None,) * 3
        o, ot, M, mu = be.fwd(q, k, v, *t, m, _lib.MASK_BOOL, False, -0.3 if Lk == 70 else D**-0.5)
        return (o, ot, M, mu, *be.bwd(q, k, v, *t, o, ot, M, mu, go if with_go else None, gt if dual else None, m, _lib.MASK_BOOL, False,
                                      -0.3 if Lk == 70 else D**-0.5, want_tangent_grads=dual if six is None else six))

    packed = step(mask)
    _lib.set_mask_bits(False)
    try:
        from_bytes = step(mask.clone())
    finally:
        _lib.set_mask_bits(True)
    for name, a, b in zip(("O", "Ot", "M", "mu", "dq", "dk", "dv", "dqt", "dkt", "dvt"), packed, from_bytes):
        assert (a is None and b is None) or torch.equal(a, b), name


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 32), (torch.float16, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("Lq,Lk,Hk", [(513, 513, 4), (128, 577, 2), (600, 70, 4)])
@pytest.mark.parametrize("dual", [False, True])
def test_packed_copy_changes_no_bit(dtype, D, Lq, Lk, Hk, dual):
    print("case", dtype, D, Lq, Lk, Hk, dual, flush=True)
    _compare(dtype, D, 2, 4, Hk, Lq, Lk, dual)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 32), (torch.float16, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("Z,H", [(1, 4), (4, 16)])  # both roles in one launch; a grid that fills the GPU
@pytest.mark.parametrize("grads", ["o", "tangent", "both"])
def test_packed_copy_changes_no_bit_of_three_gradients(dtype, D, Z, H, grads):
    print("case", dtype, D, Z, H, grads, flush=True)
    _compare(dtype, D, Z, H, H, 577, 577, grads != "o", grads != "tangent", False)


def test_packed_copies_are_made_where_kernels_of_the_call_read_them():
    q = torch.randn(1, 2, 513, 64, device="cuda").to(torch.bfloat16)
    leaf = q.clone().requires_grad_()
    wide = torch.randn(1, 2, 513, 256, device="cuda").to(torch.bfloat16).requires_grad_()
    mask = torch.rand(1, 1, 513, 513, device="cuda") < 0.9

    def made(x, p=0.0, m=None):
        m = mask.clone() if m is None else m
        o = attention(x, x, x, attn_mask=m, dropout_p=p)
        return m, o, m._jvpfa_scan.bits_q is not None, hasattr(m, "_jvpfa_bits")

    assert made(q)[2:] == (True, False)
    assert made(leaf)[2:] == (True, True)
    assert made(leaf, 0.25)[2:] == (False, True)
    assert made(q, 0.25)[2:] == (False, False)
    assert made(wide)[2:] == (False, False)
    # what is missing is made when a later call asks for it
    m = made(q, 0.25)[0]
    assert made(q, m=m)[2:] == (True, False)
    want, got = made(leaf)[1], made(leaf, m=m)
    assert got[2:] == (True, True) and torch.equal(got[1], want)
    grads = [torch.autograd.grad(o, leaf, torch.ones_like(o))[0] for o in (got[1], want)]
    assert torch.equal(*grads)
