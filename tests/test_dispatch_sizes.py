"""The sizes of tests/test_gpu_dispatch_shapes.py reach the shapes they are
listed under, by the constants and the order of the rules in the sources, on
the 256 compute units of an MI355X: a change of a rule that empties a group
fails here."""
import os
import re

from test_gpu_dispatch_shapes import ADJOINT_SIZES, FORWARD_SIZES, PASS_SIZES, SINGLE_SIZES

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "chmy.jl_amd", "csrc")
CUS, LANES = 256, 64


def source(name):
    with open(os.path.join(CSRC, name)) as f:
        return f.read()


def up(a, b):
    return -(-a // b)


def pass_shape(dims):
    src = source("stokes_multi2d.hip")
    shapes = {n: tuple(map(int, v.split(","))) for n, v in re.findall(r"using (\w+) = Shape2<([^>]*)>;", src)}
    body = src[src.index("static int shape2("):]
    order = re.findall(r"one_round<(\w+)>", body[:body.index("}")])
    assert set(order) | {"Dense2"} == set(shapes) == set(PASS_SIZES)
    for name in order:
        km, w, pt = shapes[name]
        if up(dims[0] + 2, LANES - 2 * km) * up(dims[1] + 2, w * pt - 2 * km) <= CUS:
            return name
    return "Dense2"


def regions(n, rx, ry, rows):
    return up(n[0], LANES - 2 * rx) * up(n[1], rows - 2 * ry)


def constants(src):
    return {k: int(v) for line in re.findall(r"^constexpr int (k\w+ = \d+(?:, k\w+ = \d+)*);", src, re.M)
            for k, v in re.findall(r"(k\w+) = (\d+)", line)}


def test_pass_sizes():
    for name, sizes in PASS_SIZES.items():
        assert [pass_shape(d) for d in sizes] == [name] * len(sizes)


def test_adjoint_sizes():
    src = source("sia.hip")
    ring = constants(src)["kAdjRing"]
    order = [tuple(map(int, m)) for m in re.findall(r"if \(fits\((\d+), (\d+)\)\) launch_adj_r<\1, \2, ", src)]
    assert order + [(16, 3)] == list(ADJOINT_SIZES)
    for want, sizes in ADJOINT_SIZES.items():
        for n in sizes:
            fit = [s for s in order if regions(n, 2 * ring, 2 * ring, s[0] * s[1]) +
                   regions(n, 4, 4, s[0] * (s[1] + 1)) <= CUS]
            assert (fit + [(16, 3)])[0] == want, n


def test_forward_sizes():
    c = constants(source("sia.hip"))
    assert {c["kSiaMax"], c["kSiaMany"]} == set(FORWARD_SIZES)
    for want, sizes in FORWARD_SIZES.items():
        for n in sizes:
            one = regions(n, 2 * c["kSiaMax"], 2 * c["kSiaMax"], c["kNWF"] * c["kRF2"]) <= CUS
            assert (c["kSiaMax"] if one else c["kSiaMany"]) == want, n


def test_single_step_sizes():
    src = source("sia.hip")
    c = constants(src)
    body = src[src.index("static void launch_steps("):]
    order = [(c[w], c[r], int(k)) for w, r, k in re.findall(r"if \((?:n == 1 && )?fits\((k\w+) \* (k\w+), (\d+)\)\)",
                                                            body[:body.index("\n}")])]
    last = (c["kNWF"], c["kRF2"])
    assert [o[:2] for o in order] + [last] == list(SINGLE_SIZES)
    for want, sizes in SINGLE_SIZES.items():
        for n in sizes:
            fit = [(w, r) for w, r, k in order if regions(n, 2, 2, w * r) <= k * CUS]
            assert (fit + [last])[0] == want, n
