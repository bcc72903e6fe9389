"""The native path of eager calls (``csrc/torch_binding.cpp``): which gradients arrive, what it refuses, and masks that change."""
import contextlib
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwAD
import torch.utils.checkpoint

from jvp_flash_attention_amd import JVPAttn, _lib, attention
from oracle import dense

pytestmark = pytest.mark.gpu


def _inputs(D, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(2, 3, 75, D, generator=g).to(dtype) for _ in range(8)]


@pytest.mark.parametrize("D,dtype", [(16, torch.bfloat16), (64, torch.float16), (32, torch.float32)])
@pytest.mark.parametrize("of", ["o", "ot", "both"])
@pytest.mark.parametrize("six", [False, True])
def test_gradients_of_either_output_or_both(D, dtype, of, six):
    """A gradient that does not arrive counts as zero; without one for O' the tangent inputs get zeros."""
    print("case", D, dtype, of, six, flush=True)
    cpu = _inputs(D, dtype)
    leaves = [x.cuda().requires_grad_(i < 3 or six) for i, x in enumerate(cpu[:6])]
    go, gt = cpu[6].cuda(), cpu[7].cuda()
    with fwAD.dual_level():
        o, ot = fwAD.unpack_dual(JVPAttn.fwd_dual(*(fwAD.make_dual(p, t) for p, t in zip(leaves[:3], leaves[3:]))))
        outs, gs = {"o": ((o,), (go,)), "ot": ((ot,), (gt,)), "both": ((o, ot), (go, gt))}[of]
        grads = torch.autograd.grad(outs, leaves[: 6 if six else 3], gs)
    f = [x.double().numpy() for x in cpu]
    f[6] = f[6] if of != "ot" else np.zeros_like(f[6])
    f[7] = f[7] if of != "o" else np.zeros_like(f[7])
    want = dense.backward(*f)
    for name, got in zip(("dq", "dk", "dv", "dqt", "dkt", "dvt"), grads):
        w = want[name]
        bar = 1e-4 if dtype == torch.float32 else 2e-2 * np.abs(w).max()
        assert np.abs(got.double().cpu().numpy() - w).max() <= bar, name


def test_a_second_derivative_is_refused():
    q, k, v = (x.cuda().requires_grad_() for x in _inputs(64, torch.bfloat16)[:3])
    o = attention(q, k, v)
    go = torch.ones_like(o, requires_grad=True)
    (dq,) = torch.autograd.grad(o, q, go, create_graph=True)
    with pytest.raises(RuntimeError, match="once_differentiable"):
        dq.float().sum().backward()


@pytest.mark.parametrize("dual", [False, True])
def test_gradients_of_constants_are_constants_under_create_graph(dual):
    """Where no arriving gradient requires grad, create_graph gives plain tensors that go on being used."""
    q, k, v, *t = (x.cuda() for x in _inputs(64, torch.bfloat16)[:6])
    q.requires_grad_()
    w = torch.randn_like(q).requires_grad_()
    with fwAD.dual_level():
        if dual:
            out = JVPAttn.fwd_dual(*(fwAD.make_dual(a, b) for a, b in zip((q, k, v), t)))
            o, ot = fwAD.unpack_dual(out)
            loss = o.float().sum() + ot.float().sum()
        else:
            loss = attention(q, k, v).float().sum()
        (dq,) = torch.autograd.grad(loss, q, create_graph=True)
    assert not dq.requires_grad
    (dq * w).sum().backward()
    assert torch.equal(w.grad, dq)


@pytest.mark.parametrize("tangents_require_grad", [False, True])
def test_dual_tensors_of_any_origin_get_their_gradients(tangents_require_grad):
    """Leaves, results of other operators and transposed views, dual or not, against the same values as contiguous leaves."""
    cpu = _inputs(64, torch.bfloat16)
    go, gt = cpu[6].cuda(), cpu[7].cuda()

    def step(lay, back):
        leaves = [lay(x.cuda()).requires_grad_(i < 3 or tangents_require_grad) for i, x in enumerate(cpu[:6])]
        with fwAD.dual_level():
            q, k, v, qt, kt, _ = (back(x) for x in leaves)
            v = v * 1  # a result, without a tangent
            out = JVPAttn.fwd_dual(fwAD.make_dual(q, qt), fwAD.make_dual(k, kt), v)
            o, ot = fwAD.unpack_dual(out)
            grads = torch.autograd.grad((o, ot), leaves[: 5 if tangents_require_grad else 3], (go, gt))
        assert fwAD._current_level < 0 and out.shape == go.shape
        return [o.detach(), ot.detach(), *(back(g) for g in grads)]

    want = step(lambda x: x, lambda x: x)
    got = step(lambda x: x.transpose(1, 2).contiguous(), lambda x: x.transpose(1, 2))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_a_primal_changed_in_place_before_its_backward_is_noticed():
    q, k, v, qt, kt, vt, go, _ = (x.cuda() for x in _inputs(64, torch.bfloat16))
    q.requires_grad_()
    with fwAD.dual_level():
        out = JVPAttn.fwd_dual(*(fwAD.make_dual(a, b) for a, b in zip((q, k, v), (qt, kt, vt))))
        o, _ = fwAD.unpack_dual(out)
        k.mul_(2)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(o, q, go)


def test_arguments_are_refused_with_the_reason():
    q, k, v = (x.cuda() for x in _inputs(64, torch.bfloat16)[:3])
    with pytest.raises(AssertionError, match="one dtype"):
        attention(q, k.half(), v)
    with pytest.raises(AssertionError, match="HEAD_DIM_K"):
        attention(*(x[..., :48] for x in (q, k, v)))
    with pytest.raises(AssertionError, match="dropout_p"):
        attention(q, k, v, dropout_p=1.5)


def test_the_backward_under_compiled_autograd():
    """The node's backward reads device pointers: compiled autograd has to call it as it is, not to trace it."""
    from torch._dynamo import compiled_autograd

    q, k, v = (x.cuda().requires_grad_() for x in _inputs(64, torch.bfloat16)[:3])
    go = torch.ones_like(q)
    want = torch.autograd.grad(attention(q, k, v, causal=True), (q, k, v), go)
    o = attention(q, k, v, causal=True)
    with compiled_autograd._enable(torch.compile(backend="eager")):
        o.backward(go)
    assert all(torch.equal(t.grad, w) for t, w in zip((q, k, v), want))


@pytest.mark.parametrize("dtype,D,H,L", [(torch.bfloat16, 64, 2, 520), (torch.bfloat16, 64, 32, 577), (torch.bfloat16, 256, 2, 520),
                                         (torch.float32, 64, 2, 520)])
@pytest.mark.parametrize("kind", ["rows", "keys"])
@pytest.mark.parametrize("dropout", [0.0, 0.25])
def test_a_backward_reads_the_mask_as_it_then_is(dtype, D, H, L, kind, dropout):
    """A mask refilled between forward and backward: every kernel of the backward sees the new one, as one backward() of the
    backend with that mask does.  (The new mask attends to no tile that the old one attends to, and to the keys past the old
    one's last.)"""
    print("case", dtype, D, H, L, kind, dropout, flush=True)
    g = torch.Generator(device="cuda").manual_seed(L)
    Z = 4
    q, k, v, go = (torch.randn(Z, H, L, D, generator=g, device="cuda").to(dtype) for _ in range(4))
    q, k, v = (x.requires_grad_() for x in (q, k, v))
    shape = (Z, 1, L if kind == "rows" else 1, L)
    first = (torch.arange(L, device="cuda") < 200).expand(shape).contiguous()
    second = ~first
    be, scale = _lib.backend(), D**-0.5
    mask = first.clone()
    torch.manual_seed(3)
    o = attention(q, k, v, attn_mask=mask, dropout_p=dropout)
    mask.copy_(second)
    got = torch.autograd.grad(o, (q, k, v), go)
    torch.manual_seed(3)
    drop = dict(dropout_p=dropout, dropout_seed=int(torch.randint(0, 2**62, (1,)).item()) if dropout else 0)
    plain = [x.detach() for x in (q, k, v)]
    none = (None,) * 3
    o2, _, M, _ = be.fwd(*plain, *none, first, _lib.MASK_BOOL, False, scale, *drop.values())
    assert torch.equal(o2, o)
    want = be.bwd(*plain, *none, o2, None, M, None, go, None, second, _lib.MASK_BOOL, False, scale, **drop)
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        assert torch.equal(a, b), name
    assert torch.count_nonzero(got[1][:, :, :192]) == 0 and torch.count_nonzero(got[1][:, :, 256:]) > 0


def test_a_backward_looks_at_a_forgotten_mask_again():
    """A write that no version counter shows, then forget_mask, between forward and backward."""
    L = 520
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v, go = (torch.randn(1, 2, L, 64, generator=g, device="cuda").to(torch.bfloat16) for _ in range(4))
    q, k, v = (x.requires_grad_() for x in (q, k, v))
    mask = (torch.arange(L, device="cuda") < 200).expand(1, 1, L, L).contiguous()
    second = ~mask
    o = attention(q, k, v, attn_mask=mask)
    version = mask._version
    mask.data.copy_(second)
    assert mask._version == version
    _lib.forget_mask(mask)
    got = torch.autograd.grad(o, (q, k, v), go)
    mask.data.copy_(~second)
    o = attention(q, k, v, attn_mask=mask.clone())
    other = ~second
    want_o = attention(q, k, v, attn_mask=other)
    other.copy_(second)
    assert all(torch.equal(a, b) for a, b in zip(got, torch.autograd.grad(want_o, (q, k, v), go)))


@pytest.mark.parametrize("dtype,D,Lq,Lk,kind", [(torch.bfloat16, 64, 577, 577, "rows"), (torch.float16, 128, 600, 520, "rows"),
                                                (torch.float32, 32, 520, 520, "rows"), (torch.bfloat16, 256, 520, 520, "rows"),
                                                (torch.bfloat16, 64, 70, 1000, "keys"), (torch.bfloat16, 128, 65, 17000, "keys")])
def test_a_graph_replays_with_refilled_masks(dtype, D, Lq, Lk, kind):
    """A captured forward and backward looks at the mask on every replay, whatever eager calls on the same mask leave behind
    in between."""
    print("case", dtype, D, Lq, Lk, kind, flush=True)
    g = torch.Generator(device="cuda").manual_seed(D + Lk)
    rand = lambda n: torch.randn(2, 2, n, D, generator=g, device="cuda").to(dtype)  # noqa: E731
    q, k, v, qt, kt, vt, go, gt = rand(Lq), rand(Lk), rand(Lk), rand(Lq), rand(Lk), rand(Lk), rand(Lq), rand(Lq)
    leaves = [x.requires_grad_() for x in (q, k, v)]

    def fresh():
        if kind == "keys":
            return torch.arange(Lk, device="cuda") < torch.randint(1, Lk + 1, (2, 1, 1, 1), generator=g, device="cuda")
        m = torch.rand(2, 1, Lq, Lk, generator=g, device="cuda") < 0.5
        cut = int(torch.randint(1, Lk, (1,), generator=g, device="cuda"))
        m[0, :, : Lq // 2, cut:] = False  # tiles come and go
        m[1, :, Lq // 2:, :cut] = False
        return m

    mask = fresh()

    def step():
        with fwAD.dual_level():
            out = JVPAttn.fwd_dual(*(fwAD.make_dual(a, b) for a, b in zip(leaves, (qt, kt, vt))), attn_mask=mask)
            o, ot = fwAD.unpack_dual(out)
            return [o.detach(), ot.detach(), *torch.autograd.grad((o, ot), leaves, (go, gt))]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for rep in range(4):
        if rep:
            mask.copy_(fresh())
        if rep % 2:  # an eager call first, which leaves its own lists and copies behind, and memory that is used again
            want = step()
            junk = [torch.full((1 << 16,), -1, dtype=torch.int32, device="cuda") for _ in range(8)]
        graph.replay()
        torch.cuda.synchronize()
        got = [x.clone() for x in captured]
        if not rep % 2:
            want = step()
            junk = None
        torch.cuda.synchronize()
        for i, (a, b) in enumerate(zip(got, want)):
            assert torch.equal(a, b), (rep, i)
    del junk


def test_saved_tensor_hooks_and_checkpointing_change_nothing():
    q, k, v, qt, kt, vt, go, gt = (x.cuda() for x in _inputs(64, torch.bfloat16))
    mask = torch.rand(2, 1, 75, 75, device="cuda") < 0.5
    leaves = [x.requires_grad_() for x in (q, k, v)]
    packed = []

    def step(hooks):
        with fwAD.dual_level():
            with hooks:
                o, ot = fwAD.unpack_dual(JVPAttn.fwd_dual(*(fwAD.make_dual(a, b) for a, b in zip(leaves, (qt, kt, vt))), attn_mask=mask))
            return [o.detach(), ot.detach(), *torch.autograd.grad((o, ot), leaves, (go, gt))]

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    want = step(contextlib.nullcontext())
    hooked = step(torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()))
    assert len(packed) >= 10  # q, k, v, their tangents, O, O', M, mu
    assert all(torch.equal(a, b) for a, b in zip(hooked, want))
    want = torch.autograd.grad(attention(q, k, v, causal=True), leaves, go)
    o = torch.utils.checkpoint.checkpoint(attention, q, k, v, None, 0.0, True, use_reentrant=False)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o, leaves, go), want))


def test_threads_on_streams_of_their_own_share_a_mask():
    """(First-order steps: torch keeps one forward-mode level for all threads.)"""
    mask = torch.rand(2, 1, 530, 530, generator=torch.Generator(device="cuda").manual_seed(9), device="cuda") < 0.5

    def step(seed, mask):
        g = torch.Generator(device="cuda").manual_seed(seed)
        q, k, v, go = (torch.randn(2, 3, 530, 64, generator=g, device="cuda").to(torch.bfloat16) for _ in range(4))
        q, k, v = (x.requires_grad_() for x in (q, k, v))
        o = attention(q, k, v, attn_mask=mask)
        return [o.detach(), *torch.autograd.grad(o, (q, k, v), go)]

    want = [step(seed, mask) for seed in range(4)]
    for shared in (mask, mask.clone()):  # scanned by the calls above; scanned by whichever thread comes first
        torch.cuda.synchronize()

        def work(seed, shared=shared):
            with torch.cuda.stream(torch.cuda.Stream()):
                got = [step(seed, shared) for _ in range(3)]
                torch.cuda.current_stream().synchronize()
                return got

        with ThreadPoolExecutor(4) as pool:
            for steps, w in zip(pool.map(work, range(4)), want):
                for got in steps:
                    assert all(torch.equal(a, b) for a, b in zip(got, w))
