"""A launch variant's number keeps its shape (CPU): tuning files name variants by
number, and one written earlier has to select what it measured.  The shapes that the
draw's dispatch compiles under each number are the ones below and those of the table
in profiles/autotune.md; numbers past the fixed shapes choose one by rule."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# knob: shapes (lanes per sample, vectors per lane, threads) of its numbers 0, 1, ...
SHAPES = {
    "sts_draw.fp64.r16": [(16, 5, 1024), (8, 9, 1024), (32, 3, 1024), (8, 9, 512)],
    "sts_draw.fp64.r32": [(32, 9, 1024), (16, 17, 1024), (64, 5, 1024), (32, 9, 256), (16, 17, 512), (64, 5, 256)],
    "sts_draw.fp32.r16": [(16, 3, 1024), (8, 5, 1024), (32, 2, 1024), (8, 5, 512)],
    "sts_draw.fp32.r32": [(8, 17, 1024), (16, 9, 1024), (32, 5, 1024), (8, 17, 256), (8, 17, 512), (16, 9, 256),
                          (32, 5, 256)],
    "sts_draw.fp32.r64": [(64, 9, 1024), (32, 17, 1024), (32, 17, 512), (64, 9, 256)],
}
KNOB = {k: "kTuneDraw" + k.split(".")[1].upper().replace("FP", "F") + k.split(".")[2].upper() for k in SHAPES}
LAUNCH = r"DRAW_LAUNCH\(\w+, (\d+), (\d+), (\d+)\)"


def dispatched(text, knob):
    """Number -> shape of the fixed cases in the knob's switch; a plain default is number 0."""
    body = text[text.index(f"switch (tune_value({KNOB[knob]}))"):]
    depth, end = 0, 0
    for i, ch in enumerate(body[body.index("{"):], body.index("{")):
        depth += (ch == "{") - (ch == "}")
        if depth == 0:
            end = i
            break
    body = body[:end]
    out = {int(n): tuple(map(int, s)) for n, *s in re.findall(r"case (\d+): " + LAUNCH, body)}
    plain = re.search(r"default: " + LAUNCH, body)
    if plain and 0 not in out:
        out[0] = tuple(map(int, plain.groups()))
    return out


def test_numbers_keep_their_shapes():
    text = open(os.path.join(ROOT, "rdist_tensor_amd", "csrc", "kernels_sample.hip")).read()
    for knob, shapes in SHAPES.items():
        got = dispatched(text, knob)
        assert [got.get(n) for n in range(len(shapes))] == shapes, knob


def test_documented_numbers():
    from rdist_tensor_amd import abi
    text = open(os.path.join(ROOT, "profiles", "autotune.md")).read()
    counts = {k: n for k, (n, _) in abi.tuning().items()}
    for knob, shapes in SHAPES.items():
        row = next(l for l in text.split("\n") if l.startswith(f"| `{knob}`")).split("|")[2]
        fixed = {int(n): tuple(map(int, s)) for n, *s in re.findall(r"v(\d+) \((\d+), (\d+), (\d+)\)", row)}
        assert [fixed.get(n) for n in range(len(shapes))] == shapes, knob
        assert counts[knob] == max(map(int, re.findall(r"v(\d+)\b", row))) + 1, knob


def test_shipped_table_is_in_range():
    from rdist_tensor_amd import abi
    counts = {k: n for k, (n, _) in abi.tuning().items()}
    lines = [l.split("#")[0].split() for l in open(os.path.join(ROOT, "rdist_tensor_amd", "tuning.txt"))]
    table = {l[0]: int(l[1]) for l in lines if l}
    assert set(table) == set(counts)
    for knob, v in table.items():
        assert 0 <= v < counts[knob], knob
