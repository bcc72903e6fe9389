"""Causal blocks dealt to workgroups by length: the deal itself on the CPU, and forwards and backwards that go by it on the GPU."""
import os

import pytest
import torch

from jvp_flash_attention_amd import _lib, build
from oracle import dense

from .test_gpu_split_merge import dealt_parts
from .test_launch_rules import run


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")
def test_every_share_is_dealt_once(tmp_path):
    """Ranks 0 .. workgroups() - 1 of a head are the shares of its orders, each once; shares() of an order agrees."""
    text = """
  int bad = 0;
  for (int most = 1; most <= 8; ++most)
    for (int step = most > 1; step <= 9; ++step)
      for (int first = 0; first < 20; first += 3)
        for (int last = first + 1; last < 41; ++last) {
          const Deal d = {most, step, first, last};
          int n = 0, seen[41][8] = {};
          for (int o = first; o < last; ++o) n += d.shares(o);
          bad += n != d.workgroups();
          for (int r = 0; r < n; ++r) {
            const Share s = share_of(d, r);
            const bool in = s.order >= first && s.order < last && s.index >= 0 && s.index < s.count;
            bad += !in || s.count != d.shares(s.order) || seen[s.order][s.index]++ != 0;
          }
        }
  std::printf("%d ", bad);
"""
    assert run(tmp_path, text) == [0]


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")
def test_deals_of_backwards(tmp_path):
    """Whole blocks where they fill the units or are short, more shares the longer a block is, and bounded partial results."""
    shapes = [(D, dual, H, L, Lk) for D in (32, 64, 128) for dual in (0, 1) for H in (1, 3, 16, 40) for L in (100, 777, 3000, 30000) for Lk in (64, 1000, 30000)]
    text = "  int bad = 0, split = 0;\n"
    for D, dual, H, L, Lk in shapes:
        text += f"""  {{ const BwdDeal d = bwd_deal(false, {D}, 1, {H}, {L}, {Lk}, true, {dual}, 256);
    const int bq = {(L + 127) // 128}, bk = {(Lk + 127) // 128};
    bad += d.q.most < 1 || d.q.most > 8 || d.k.most < 1 || d.k.most > 8 || (d.q.most > 1 && d.q.step < 1) || (d.k.most > 1 && d.k.step < 1);
    bad += d.q.last != bq || d.k.last != bq || d.k.first != bq - std::min(bq, bk);
    bad += d.any() && {H} * (d.q.most * bq + 2 * d.k.most * bk) > 6 * 256 + 2 * 256 * 8;
    split += d.any(); }}
"""
    bad, split = run(tmp_path, text + '  std::printf("%d %d", bad, split);\n')
    assert bad == 0 and 0 < split < len(shapes)
    whole = ", ".join(f"bwd_deal(false, {D}, 4, 16, 2048, 2048, true, true, 256).any()" for D in (32, 64, 128))
    assert run(tmp_path, f'  for (bool b : {{{whole}}}) std::printf("%d ", b ? 1 : 0);\n') == [0, 0, 0]


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")
def test_equal_shares_are_as_long_as_planned(tmp_path):
    """Odd lengths, too: no share of any block is longer, and no block is cut into more than it needs."""
    text = "  int bad = 0, odd = 0;\n  struct P { int D, Z, H, L, dtype, causal, mask_kind; float dropout_p; };\n"
    for D, dual, H, L in [(128, 1, 3, 728), (128, 1, 7, 1635), (64, 0, 3, 5000), (128, 0, 12, 1997), (128, 1, 2, 6201), (64, 1, 5, 3427)]:
        text += f"""  {{ const BwdSplitPlan e = bwd_split_plan({D}, 1, {H}, {L}, {L}, true, {dual}, 256);
    const BwdDeal d = make_bwd_deal({D}, 1, {H}, {L}, {L}, true, {dual}, 256);
    odd += e.tiles_q % 2;
    for (int o = 0; o < d.q.last; ++o) bad += d.q.shares(o) != (2 * o + 2 + e.tiles_q - 1) / e.tiles_q; }}
"""
    for H, L in [(12, 693), (12, 651), (5, 676), (3, 680)]:
        text += f"""  {{ const P p = {{128, 1, {H}, {L}, 0, 1, 0, 0.f}}; const SplitPlan s = fwd_split_plan_16(p, {L}, false, 256);
    const int n = {(L + 63) // 64}, per = (n + s.chunks - 1) / s.chunks;
    for (int o = 0; o < {(L + 127) // 128}; ++o) bad += s.chunks < 2 || Deal{{s.chunks, s.chunk_tiles, 0, {(L + 127) // 128}}}.shares(o) != (std::min(2 * o + 2, n) + per - 1) / per; }}
"""
    bad, odd = run(tmp_path, text + '  std::printf("%d %d", bad, odd);\n')
    assert bad == 0 and odd > 3


# D, tangents, heads, rows of a causal forward, and the shares of its longest block on 256 compute units
FORWARDS = [(128, 0, 6, 1111, 3), (128, 0, 4, 1111, 3), (128, 0, 3, 1667, 5), (128, 0, 6, 1484, 4), (64, 0, 5, 1985, 4), (64, 0, 3, 1985, 4), (64, 1, 8, 1103, 3),
            (128, 1, 8, 2048, 3), (128, 1, 2, 8192, 3), (64, 0, 3, 7421, 4), (64, 0, 1, 14336, 4), (128, 1, 6, 4096, 2), (64, 0, 1, 16384, 6), (64, 0, 1, 8483, 7), (64, 1, 10, 1400, 4)]


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")
def test_no_more_shares_than_the_merge_is_worth(tmp_path):
    text = "  struct P { int D, Z, H, L, dtype, causal, mask_kind; float dropout_p; };\n"
    for D, dual, H, L, _ in FORWARDS:
        text += f'  {{ const P p = {{{D}, 1, {H}, {L}, 0, 1, 0, 0.f}}; std::printf("%d ", fwd_split_plan_16(p, {L}, {dual}, 256).chunks); }}\n'
    assert [(x, y) for x, y in zip(FORWARDS, run(tmp_path, text)) if x[-1] != y] == []


# calls that comments quote a time for, in shares or whole, on 256 compute units: direction, type (2: fp32), D, tangents, batch, heads, rows, causal, dealt
QUOTED = [
    *((0, "fwd", 128, d, 1, h, n, 1, x) for h, n, x2 in ((8, 2048, (1, 1)), (12, 2048, (0, 1)), (6, 4096, (1, 1)), (2, 8192, (1, 1))) for d, x in enumerate(x2)),
    *((0, "fwd", 64, d, 1, h, n, 1, x) for h, n, x2 in ((12, 1500, (0, 1)), (6, 4096, (1, 1)), (2, 8192, (1, 1)), (1, 16384, (1, 1))) for d, x in enumerate(x2)),
    *((0, "bwd", 128, d, 1, h, n, 1, x) for h, n, x2 in ((12, 1024, (0, 0)), (16, 1024, (0, 0)), (9, 2048, (0, 1)), (7, 2500, (1, 1)), (2, 12000, (1, 1))) for d, x in enumerate(x2)),
    *((0, "bwd", 64, d, 1, h, n, 1, x) for h, n, x2 in ((16, 1024, (0, 0)), (6, 4096, (1, 1)), (1, 30000, (1, 1)), (3, 5000, (1, 1))) for d, x in enumerate(x2)),
    *((0, "bwd", 32, d, 1, h, n, 1, x) for h, n, x2 in ((12, 1024, (0, 0)), (6, 4096, (1, 1)), (1, 8192, (1, 1))) for d, x in enumerate(x2)),
    *((2, "fwd", D, d, z, h, n, c, x) for D, z, h, n, c, x2 in ((64, 1, 8, 512, 0, (0, 1)), (64, 1, 2, 4096, 1, (1, 1)), (64, 2, 6, 777, 0, (0, 1)), (128, 1, 8, 512, 0, (1, 1)),
                                                          (128, 1, 16, 1024, 0, (1, 1)), (128, 1, 40, 1000, 0, (1, 1)), (32, 1, 12, 1024, 1, (0, 1))) for d, x in enumerate(x2)),
    *((2, "bwd", D, d, z, h, n, c, x) for D, z, h, n, c, x2 in ((64, 1, 8, 512, 0, (0, 1)), (64, 1, 12, 1024, 1, (1, 1)), (64, 3, 4, 640, 0, (0, 1)), (64, 1, 2, 4096, 1, (1, 1)),
                                                          (128, 1, 8, 512, 0, (1, 1)), (128, 1, 12, 1024, 1, (1, 1)), (32, 1, 2, 4096, 1, (1, 1))) for d, x in enumerate(x2)),
    (2, "bwd", 64, 1, 1, 4, 900, 0, 1), (2, "bwd", 64, 1, 1, 2, 300, 0, 0),
]


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")
def test_calls_with_a_quoted_time_are_dealt_or_whole(tmp_path):
    text = "  struct P { int D, Z, H, L, dtype, causal, mask_kind; float dropout_p; };\n"
    for kind, way, D, dual, Z, H, L, causal, _ in QUOTED:
        if way == "fwd":
            plan = f"fwd_split_plan_{'f32' if kind else 16}(p, {L}, {dual}, 256).chunks > 1"
        else:
            plan = f"make_bwd_deal{'_f32' if kind else ''}({D}, {Z}, {H}, {L}, {L}, {causal}, {dual}, 256).any()"
        text += f'  {{ const P p = {{{D}, {Z}, {H}, {L}, {kind}, {causal}, 0, 0.f}}; (void)p; std::printf("%d ", {plan} ? 1 : 0); }}\n'
    assert [x for x, y in zip(QUOTED, run(tmp_path, text)) if x[-1] != y] == []


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")
def test_order_of_a_launch_goes_by_the_units_of_the_device(tmp_path):
    """280 workgroups of 4 heads: heads side by side on 256 units, the shares of a block on 304; either way each once."""
    text = """  for (int units : {256, 304}) {
    int seen[4][70] = {}, bad = 0;
    for (int b = 0; b < 280; ++b) {
      const HeadRank r = deal_heads(b, 4, 280, more_than_units(280, units));
      bad += r.head < 0 || r.head > 3 || r.rank < 0 || r.rank > 69 || seen[r.head][r.rank]++;
    }
    std::printf("%d %d ", bad, deal_heads(1, 4, 280, more_than_units(280, units)).head);
  }
"""
    assert run(tmp_path, text) == [0, 1, 0, 0]


# few workgroups, more than there are units (heads that are and are not a multiple of 8), keys and queries of unequal number
SHAPES = [(1, 4, 1100, 1100), (1, 3, 4200, 4200), (2, 4, 2100, 2100), (1, 2, 900, 2000), (1, 3, 2000, 900)]


# ... whose forwards stay whole on 256 compute units: always at D = 32, which has no kernel for it; at D = 64 head dim, queries, keys, tangents
WHOLE_FORWARDS = {(64, 1100, 1100, False), (64, 2100, 2100, False), (64, 900, 2000, False), (64, 2000, 900, False), (64, 2000, 900, True)}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Z,H,L,Lk", SHAPES)
@pytest.mark.parametrize("grads", ["plain", "both", "tangent"])
def test_dealt_blocks_agree_with_whole_ones(dtype, D, Z, H, L, Lk, grads):
    """Against the same kernels on whole blocks, and a slab of rows of O, O' against the dense oracle."""
    print("case", dtype, D, Z, H, L, Lk, grads, flush=True)
    g = torch.Generator(device="cuda").manual_seed(L + D)
    rand = lambda n: torch.randn(Z, H, n, D, generator=g, device="cuda").to(dtype)  # noqa: E731
    q, qt, go, gt, k, v, kt, vt = rand(L), rand(L), rand(L), rand(L), rand(Lk), rand(Lk), rand(Lk), rand(Lk)
    t = (None,) * 3 if grads == "plain" else (qt, kt, vt)
    be, scale = _lib.backend(), D**-0.5
    parts = dealt_parts((q, k, v, *t), (go, gt if grads != "plain" else None), None, _lib.MASK_NONE, True, scale)
    assert parts == (D > 32 and (D, L, Lk, grads != "plain") not in WHOLE_FORWARDS, True)
    fwd = lambda: be.fwd(q, k, v, *t, None, _lib.MASK_NONE, True, scale)  # noqa: E731
    got = fwd()
    _lib.set_split(False)
    try:
        one = fwd()
        bwd = lambda: be.bwd(q, k, v, *t, *one, go if grads != "tangent" else None, gt if grads != "plain" else None,  # noqa: E731
                             None, _lib.MASK_NONE, True, scale)
        whole = bwd()
    finally:
        _lib.set_split(True)
    dealt = bwd()
    ulp = 2.0**-7 if dtype == torch.bfloat16 else 2.0**-10
    for a, b in zip(got[2:], one[2:]):
        assert b is None or (a - b).abs().max().item() <= 1e-5 * max(1.0, b.abs().max().item())
    # P is rounded against another reference point in each share, so either side has for every key an error of its own of up to half a unit of p, as
    # good as independent: 0.3 units of the entry's size by root mean square (0.2 for a uniform error, times the square root of 2), and the result's own
    # rounding.  O' has two products that are rounded so.  Five times that for the worst of 2 million entries, against its row's root mean square.
    for a, b, products in zip(got[:2], one[:2], (1, 2)):
        if b is not None:
            a, b = a.double(), b.double()
            assert (a - b).norm() <= products * ulp / 2 * b.norm()
            assert ((a - b).abs() <= ulp * b.abs() + products * 2 * ulp * b.square().mean(-1, keepdim=True).sqrt()).all()
    for a, b in zip(dealt[:3], whole[:3]):  # the same P and dS, sums in fp32 in another order, each rounded once
        assert (a.float() - b.float()).norm() <= ulp / 2 * b.float().norm()
        assert ((a.float() - b.float()).abs() <= ulp * b.float().abs() + 1e-5 * b.float().abs().max()).all()
    rows = slice(max(0, L - 70), L)  # the last rows: the block with most shares
    f = [x[:1, :1].double().cpu().numpy() for x in (q, k, v, qt, kt, vt)]
    keep = torch.arange(Lk)[None, :] <= torch.arange(L)[rows][:, None]
    ref = dense.forward(f[0][:, :, rows], f[1], f[2], f[3][:, :, rows], f[4], f[5], mask=keep[None, None].numpy(), scale=scale)
    for x, name in ((got[0], "O"), (got[1], "Ot")):
        if x is not None:
            want = ref[name]
            assert abs(x[:1, :1, rows].double().cpu().numpy() - want).max() <= 2e-2 * abs(want).max()
