"""Every shape that the 2D multi-iteration passes and the SIA launches choose
from by grid size, bitwise against single iterations and single steps.  The
sizes are listed under the shape they reach; tests/test_dispatch_sizes.py
holds the lists to the shapes' constants in the sources."""
import numpy as np
import pytest
import torch

import chmy
from chmy.sia import SIA
from _helpers import dev
from test_gpu_fused_pairs import GENERAL, _compare, _run
from test_gpu_sia import _setup

pytestmark = pytest.mark.gpu

# grids that end at, past and inside the shape's tiles
PASS_SIZES = {"Small2": [(49, 3), (101, 66)],
              "Flat2": [(160, 148), (161, 149)],
              "Mid2": [(414, 378), (415, 379), (400, 380)],
              "Large2": [(478, 638), (481, 639)],
              "Dense2": [(862, 558), (863, 559)]}
# adjoint pairs: waves and rows of a region
ADJOINT_SIZES = {(8, 2): [(57, 11), (104, 52)], (12, 2): [(260, 180), (261, 181), (300, 200)], (16, 3): [(512, 437)]}
# forward steps a launch may take
FORWARD_SIZES = {5: [(250, 177)], 3: [(800, 520), (833, 541)]}
# single forward steps: waves and rows of a region
SINGLE_SIZES = {(4, 2): [(60, 4), (61, 5), (300, 196)], (8, 2): [(360, 372), (361, 373)], (16, 2): [(480, 476), (481, 477)],
                (16, 3): [(840, 616), (841, 617)]}


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


@pytest.mark.parametrize("dims,niter,forcing", [((1699, 1541), 4, None), ((1699, 1541), 6, None), ((1699, 1541), 7, None),
                                                ((1699, 1541), 13, None), ((1699, 1541), 22, None), ((1690, 1540), 6, None),
                                                ((1699, 1541), 6, "bf16"), ((2290, 2290), 8, "bf16"),
                                                ((2290, 2290), 17, "bf16")])
def test_fp32_exact_passes_of_five_and_two(arch, dims, niter, forcing):
    """FP32, exact form, at and below the size from which runs are cut into
    passes of five and two iterations: pairs only, a five and pairs, fives and
    pairs (the batch is the next pass's before a five, a launch before a pair).
    Bitwise; the random state overflows after 17 iterations, and a NaN counts as
    a NaN (IEEE 754 leaves its sign open: Inf - Inf by the order of operands)."""
    g = chmy.UniformGrid(arch, origin=(-0.5, -0.5), extent=(1.0, 1.3), dims=dims)
    a, b = ([np.where(np.isnan(x), np.float32("nan"), x) for x in
             _run(arch, g, np.float32, True, "field", forcing, GENERAL, niter, pairs, 43)] for pairs in (True, False))
    _compare(a, b, f"dims {dims} niter {niter}")


@pytest.mark.parametrize("npow", [3, 2])
@pytest.mark.parametrize("n", sum(ADJOINT_SIZES.values(), []) + sum(FORWARD_SIZES.values(), []))
def test_sia_gradient_over_shapes(arch, n, npow):
    """Seven steps and two checkpoints: segments of four states and of three,
    so that paired and single adjoint steps and riding steps mix.  The run
    against the per-point step, the reverse sweep against the five gather
    passes, bitwise."""
    g, og, H, hH, B, hB, A, hA = _setup(arch, n=n, seed=23)
    S = SIA(arch, g, hB.arr, logA=np.log(hA.arr), As=0.5, npow=npow, mb=(0.5, 0.3, 0.25))
    dt = 1e-2 * min(e / m for e, m in zip(g.extent, n)) ** 2
    dts = [dt * (1 + 0.1 * k) for k in range(7)]
    want = [hH.arr.copy()]
    S.reset(hH.arr)
    for d in dts:
        S.step(d)
        S.H.swap(S.H2)
        want.append(dev(S.H).copy())
    S.reset(hH.arr)
    S.forward(7, dts)
    assert np.array_equal(dev(S.H), want[7]) and np.array_equal(dev(S.H2), want[6])
    last = torch.from_numpy(want[7][2:-2, 2:-2].T.copy()).to(S.lam.data.device)
    obs = last * 0.97
    _, grad = S.gradient(hH.arr, obs, 7, dts, ncheck=2)
    lam = S.lam.interior().clone()
    for a in (S.grad, S.lam, S.lam2):
        a.data.zero_()
    S.lam.interior().copy_(last - obs)
    for k in reversed(range(7)):
        S.reset(want[k])
        S._adjoint_step(S.H, dts[k], passes=5)
    assert torch.equal(S.lam.interior(), lam) and torch.equal(S.grad.interior(), grad)


@pytest.mark.parametrize("npow", [3, 2])
@pytest.mark.parametrize("n", sum(SINGLE_SIZES.values(), []))
def test_sia_single_steps_over_shapes(arch, n, npow):
    """A run that keeps every state, one step a launch, against the per-point
    step and its Neumann batch, bitwise over the storage."""
    g, og, H, hH, B, hB, A, hA = _setup(arch, n=n, seed=29)
    S = SIA(arch, g, hB.arr, logA=np.log(hA.arr), As=0.5, npow=npow, mb=(0.5, 0.3, 0.25))
    dt = 1e-2 * min(e / m for e, m in zip(g.extent, n)) ** 2
    dts = [dt * (1 + 0.1 * k) for k in range(3)]
    S.reset(hH.arr)
    states = [S._field() for _ in range(4)]
    states[0].data.copy_(S.H.data)
    S.run(states, dts)
    for k, d in enumerate(dts):
        S.step(d)
        S.H.swap(S.H2)
        assert torch.equal(states[k + 1].data, S.H.data), k
