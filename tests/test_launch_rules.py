"""The rules that say how a backward is launched, on the CPU."""
import os
import subprocess

import pytest

from jvp_flash_attention_amd import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")


def run(tmp_path, text, **env):
    """What a program with `text` in its main prints, numbers apart."""
    src, exe = tmp_path / "rules.hip", tmp_path / "rules"
    src.write_text('#include <cstdio>\n#include "split.hpp"\nusing namespace jvpfa;\nint main() {\n' + text + "}\n")
    subprocess.run([build.HIPCC, *build.FLAGS, "-I", build.CSRC, str(src), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], env={**os.environ, **env}, capture_output=True, text=True)
    assert r.returncode == 0, r.returncode
    return [int(x) for x in r.stdout.split()]


def test_device_that_cannot_be_asked(tmp_path):
    """Two launches, whatever the grid (and no division by the number of units)."""
    text = "  int one = 0;\n  for (long long b : {1LL, 255LL, 300LL, 5000LL})\n    for (int f = 0; f < 32; ++f) {\n"
    for D in (32, 64, 128, 256):
        text += f"""
      one += launch_both<{D}, BWD_PLAIN>(b, 2 * b, f & 1, f & 2 ? MASK_BITS : MASK_NONE, f & 4, false, f & 8, f & 16);
      one += launch_both<{D}, BWD_DUAL>(2 * b, b, f & 1, f & 2 ? MASK_BOOL : MASK_NONE, f & 4, f & 8, false, f & 16);
      one += launch_both_f32<{D}, BWD_PLAIN>(b, 3 * b, f & 1) + launch_both_f32<{D}, BWD_DUAL>(3 * b, b, f & 2);
"""
    assert run(tmp_path, text + '    }\n  std::printf("%d %d", device_cus(), one);\n', HIP_VISIBLE_DEVICES="-1") == [0, 0]


# D, mode, what the call has, and blocks of either role with what was faster on 256 compute units: 1 one launch, 0 two
SIDES = [
    (32, "DUAL", "bits", {256: 1, 336: 1, 384: 0, 512: 0, 2048: 0}),
    (32, "DUAL", "bool", {512: 1, 2048: 1}),
    (32, "DUAL", "", {512: 1, 2048: 1}),
    (32, "PLAIN", "bits", {512: 1, 2048: 1}),
    (64, "PLAIN", "bits", {256: 1, 320: 1, 384: 0, 1024: 0}),
    (64, "PLAIN", "bool", {288: 1, 1024: 1}),
    (64, "DUAL", "bits two", {512: 1, 2048: 1}),
    (64, "DUAL", "bool", {256: 1, 392: 1, 448: 0, 512: 0, 640: 1, 1024: 0}),
    (32, "DUAL", "drop", {320: 1, 384: 0}),
    (32, "DUAL", "drop causal", {384: 1, 448: 0}),
    (32, "TANGENT", "drop", {448: 1, 640: 1}),
    (64, "PLAIN", "drop", {256: 1, 288: 0, 384: 0}),
    (64, "PLAIN", "drop causal", {384: 1, 448: 0}),
    (32, "DUAL", "six", {336: 1, 384: 0, 512: 0}),
    (32, "DUAL", "six causal", {384: 1, 448: 0}),
    (32, "DUAL", "six bits", {512: 1}),
    (64, "DUAL", "six", {384: 1, 448: 0, 512: 0, 640: 1, 704: 0}),
    (64, "DUAL", "six causal", {512: 1, 640: 1}),
    (64, "DUAL", "grouped", {384: 1, 448: 0, 512: 0, 704: 0}),
    (64, "DUAL", "grouped causal", {512: 1, 640: 0}),
    (64, "DUAL", "grouped alone", {512: 1, 640: 1, 768: 0}),  # gradients of O' alone
    (64, "PLAIN", "grouped", {1024: 1, 1536: 1}),
    (128, "DUAL", "", {128: 1, 288: 1, 2048: 0}),
    (128, "DUAL", "causal", {512: 1, 1024: 0}),
]


def test_one_launch_or_two(tmp_path):
    text, want, names = "", [], []
    for D, mode, has, sides in SIDES:
        f = {x: str(x in has.split()).lower() for x in ("causal", "drop", "six", "grouped", "two", "alone")}
        mask = "MASK_BITS" if "bits" in has else "MASK_BOOL" if "bool" in has else "MASK_NONE"
        for blocks, one in sides.items():
            call = f"launch_both<{D}, BWD_{mode}>({blocks}, {blocks}, {f['causal']}, {mask}, {f['drop']}, {f['six']}, {f['grouped']}, {f['two']}, {f['alone']}, 256)"
            text += f'  std::printf("%d ", {call} ? 1 : 0);\n'
            want.append(one)
            names.append(call)
    got = run(tmp_path, text)
    assert [n for n, a, b in zip(names, got, want) if a != b] == []


# the same in fp32; "uneven": causal or a boolean mask
SIDES_F32 = [
    (32, "PLAIN", "", {168: 1, 448: 1, 2048: 1}),
    (32, "TANGENT", "", {168: 1, 448: 1}),
    (32, "DUAL", "", {160: 1, 176: 0, 208: 0, 224: 1, 256: 1, 416: 1, 448: 0, 640: 1, 768: 0}),
    (64, "DUAL", "", {136: 1, 168: 0, 192: 0, 240: 1, 256: 1, 288: 1, 384: 1, 480: 0, 640: 1, 768: 0}),
    (64, "PLAIN", "", {160: 1, 192: 1, 224: 1, 448: 0, 2048: 0}),
    (64, "DUAL", "uneven", {160: 1, 256: 1, 448: 1, 512: 1, 640: 1, 768: 0}),
    (128, "DUAL", "", {144: 1, 192: 1, 256: 1, 320: 1, 416: 1, 576: 1, 640: 1, 1024: 0}),
]


def test_one_launch_for_roles_of_unequal_length(tmp_path):
    """D = 64, dual: few blocks of one role fit beside many of the other, where as many again of them would not."""
    calls = {f"launch_both<64, BWD_DUAL>({a}, {b}, false, MASK_BOOL, false, false, false, false, false, 256)": one
             for a, b, one in ((512, 64, 1), (96, 512, 1), (512, 512, 0), (512, 420, 0), (640, 64, 1), (768, 64, 0))}
    calls["launch_both<64, BWD_DUAL>(512, 16, false, MASK_NONE, false, false, false, true, false, 256)"] = 1  # 4000 queries over 64 keys, uncapped
    got = run(tmp_path, "".join(f'  std::printf("%d ", {c} ? 1 : 0);\n' for c in calls))
    assert [c for c, a in zip(calls, got) if a != calls[c]] == []


def test_one_launch_or_two_in_fp32(tmp_path):
    calls = {f"launch_both_f32<{D}, BWD_{mode}>({n}, {n}, {str(has == 'uneven').lower()}, 256)": one
             for D, mode, has, sides in SIDES_F32 for n, one in sides.items()}
    got = run(tmp_path, "".join(f'  std::printf("%d ", {c} ? 1 : 0);\n' for c in calls))
    assert [c for c, a in zip(calls, got) if a != calls[c]] == []


# D, dual, heads, queries, keys, causal, and the shares of a block of dq and of dk/dv on 256 compute units
SHARES = [
    # blocks of up to 8 tiles: cut where that is a tenth faster, whole where it is a tenth slower
    (128, 1, 1, 512, 512, 0, 2, 2), (128, 1, 12, 512, 512, 0, 2, 2), (128, 1, 16, 512, 512, 0, 1, 1), (128, 1, 16, 512, 512, 1, 2, 2),
    (128, 1, 4, 384, 384, 0, 2, 2), (128, 1, 8, 384, 384, 0, 1, 1), (128, 1, 8, 384, 384, 1, 2, 2), (128, 1, 12, 384, 384, 1, 1, 1),
    (128, 1, 4, 320, 1500, 1, 1, 1), (128, 1, 8, 1000, 512, 0, 1, 2), (128, 1, 4, 512, 2000, 0, 3, 1), (128, 1, 2, 512, 2000, 0, 6, 2),  # one role cut is no gain if the other stays long
    (128, 1, 1, 256, 256, 0, 1, 1), (128, 1, 4, 1024, 1024, 0, 4, 4), (128, 1, 1, 65536, 65536, 1, 1, 1),
    # causal: more shares than units only while the blocks unsplit leave units idle
    (128, 0, 16, 1500, 1500, 1, 1, 1), (128, 1, 16, 1500, 1500, 1, 1, 1), (128, 1, 10, 1500, 1500, 1, 1, 1), (128, 1, 8, 1500, 1500, 1, 2, 2),
    (128, 1, 8, 2048, 2048, 1, 3, 3), (128, 0, 10, 2048, 2048, 1, 1, 1), (128, 1, 6, 4096, 4096, 1, 1, 1), (128, 1, 4, 4096, 4096, 1, 3, 3),
    (128, 1, 12, 1500, 700, 1, 1, 2), (64, 1, 16, 2000, 512, 1, 1, 2),  # (one role cut is less to pay for)
    (64, 1, 12, 2048, 2048, 1, 1, 1), (64, 1, 6, 3000, 3000, 1, 2, 2), (64, 1, 8, 2048, 2048, 1, 3, 3), (64, 0, 12, 2048, 2048, 1, 2, 2), (32, 1, 10, 2048, 2048, 1, 2, 2),
    # D = 64 without tangents: not for four tiles
    (64, 0, 16, 512, 512, 0, 1, 1), (64, 0, 2, 512, 512, 0, 1, 1), (64, 1, 8, 512, 512, 0, 2, 2), (64, 0, 4, 777, 777, 0, 3, 3), (64, 0, 1, 512, 2000, 0, 8, 2),
]


def test_shares_of_small_backwards(tmp_path):
    text = "".join(f'  {{ const BwdSplitPlan s = bwd_split_plan({D}, 1, {H}, {L}, {Lk}, {c}, {dual}, 256); std::printf("%d %d ", s.chunks_q, s.chunks_k); }}\n'
                   for D, dual, H, L, Lk, c, _, _ in SHARES)
    got = run(tmp_path, text)
    assert [(x, got[2 * i], got[2 * i + 1]) for i, x in enumerate(SHARES) if (got[2 * i], got[2 * i + 1]) != x[-2:]] == []


def test_capped_kernel_for_both_roles(tmp_path):
    """Queries, keys, heads, causal: capped where the launch has more work than its longest block for every unit."""
    sides = {(2048, 2048, 8, 0): 0, (777, 777, 20, 0): 1, (1000, 1000, 24, 0): 1, (1500, 700, 20, 0): 0, (1000, 512, 28, 0): 0, (1000, 512, 96, 0): 1,
             (512, 2000, 14, 0): 1, (512, 1000, 24, 0): 1, (512, 1000, 20, 0): 0,
             (2048, 2048, 14, 1): 0, (1500, 1500, 20, 1): 0, (777, 777, 32, 1): 0, (512, 512, 48, 1): 0, (512, 512, 56, 1): 1, (340, 340, 80, 1): 1,
             (640, 640, 48, 1): 1, (2048, 2048, 16, 1): 1, (512, 2000, 16, 1): 1, (1, 1, 1, 1): 0}
    got = run(tmp_path, "".join(f'  std::printf("%d ", both_two_wgs({L}, {Lk}, {h}, {c}, 256) ? 1 : 0);\n' for L, Lk, h, c in sides))
    assert [x for x, y in zip(sides, got) if y != sides[x]] == []


PLANS = """
  long long made = 0;
  auto plan = [&](int size) { return remembered<int, 1>({size}, [&] { ++made; return 3 * size; }); };
"""


def test_plans_are_remembered_for_as_many_shapes_as_a_model_has(tmp_path):
    """Sixteen shapes in turn, again and again: each is planned once, and every answer is that of its sizes."""
    text = PLANS + """
  int bad = 0;
  for (int i = 0; i < 1600; ++i) bad += plan(100 + i % 16 * 37) != 3 * (100 + i % 16 * 37);
  const int first = made;
  for (int i = -1000; i < 1000; ++i) bad += plan(i * 7919) != 3 * (i * 7919) || plan(i * 7919) != 3 * (i * 7919);
  std::printf("%d %d %d", bad, first, (int)(made - first));
"""
    assert run(tmp_path, text) == [0, 16, 2000]


def test_plans_are_remembered_however_many_were_made(tmp_path):
    """More plans than a 32-bit count holds, each of another size: the last one is still found where it was put."""
    text = PLANS + """
  const long long many = (1LL << 31) + 19;
  long long sum = 0;
  for (long long i = 0; i < many; ++i) sum += plan((int)(unsigned)i) != 3 * (int)(unsigned)i;
  const long long before = made;
  const int size = 12345;
  sum += plan(size) != 3 * size, sum += plan(size) != 3 * size;
  std::printf("%d %d", (int)sum, (int)(made - before));
"""
    assert run(tmp_path, text) == [0, 1]
