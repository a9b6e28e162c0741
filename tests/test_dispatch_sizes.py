"""The sizes of tests/test_gpu_dispatch_shapes.py reach the shapes they are
listed under, by the constants and the order of the rules in the sources, on
the 256 compute units of an MI355X: a change of a rule that empties a group
fails here."""
import os
import re

from test_gpu_dispatch_shapes import PASS_SIZES

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


def test_pass_sizes():
    for name, sizes in PASS_SIZES.items():
        assert [pass_shape(d) for d in sizes] == [name] * len(sizes)
