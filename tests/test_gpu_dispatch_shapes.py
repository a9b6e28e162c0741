"""Every shape that the 2D multi-iteration passes choose from by grid size,
bitwise against single iterations.  The sizes are listed under the shape they reach; tests/test_dispatch_sizes.py
holds the lists to the shapes' constants in the sources."""
import numpy as np
import pytest

import chmy
from test_gpu_fused_pairs import GENERAL, _compare, _run

pytestmark = pytest.mark.gpu

# grids that end at, past and inside the shape's tiles
PASS_SIZES = {"Small2": [(49, 3), (101, 66)],
              "Flat2": [(160, 148), (161, 149)],
              "Mid2": [(414, 378), (415, 379), (400, 380)],
              "Large2": [(478, 638), (481, 639)],
              "Dense2": [(862, 558), (863, 559)]}

@pytest.fixture(scope="module")
def arch():
    return chmy.Arch(chmy.MI355XBackend())


@pytest.mark.parametrize("T,forcing", [(np.float64, None), (np.float64, "same"), (np.float32, "bf16")])
@pytest.mark.parametrize("exact,visc,rhog", [(False, "field", True), (True, "field", False), (False, "scalar", False)])
@pytest.mark.parametrize("dims,niter", [(PASS_SIZES["Mid2"][0], 13), (PASS_SIZES["Mid2"][1], 12),
                                        (PASS_SIZES["Mid2"][2], 7), (PASS_SIZES["Mid2"][1], 6)])
def test_passes_of_two_rows_a_thread_2d(arch, T, forcing, exact, visc, rhog, dims, niter):
    """Mid2 (52 x 20 own points, up to 6 iterations): whole passes, even
    splits and remainders."""
    g = chmy.UniformGrid(arch, origin=(-0.5, -0.5), extent=(1.0, 1.3), dims=dims)
    a = _run(arch, g, T, exact, visc, forcing, GENERAL, niter, True, 37, rhog=rhog)
    b = _run(arch, g, T, exact, visc, forcing, GENERAL, niter, False, 37, rhog=rhog)
    _compare(a, b, f"dims {dims} niter {niter}")


@pytest.mark.parametrize("shape,dims,niter", [(s, d, n) for s, ds in PASS_SIZES.items() if s != "Mid2"
                                              for d, n in zip(ds, (17, 12))])
def test_passes_of_the_other_shapes_2d(arch, shape, dims, niter):
    g = chmy.UniformGrid(arch, origin=(-0.5, -0.5), extent=(1.0, 1.3), dims=dims)
    a = _run(arch, g, np.float64, False, "field", None, GENERAL, niter, True, 41)
    b = _run(arch, g, np.float64, False, "field", None, GENERAL, niter, False, 41)
    _compare(a, b, f"{shape} dims {dims} niter {niter}")
