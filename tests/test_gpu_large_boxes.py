"""A box of 2^32 points (more work-items than one grid dimension takes): every
point is written once, bitwise the same expression in torch, band by band."""
import pytest
import torch

import chmy
from chmy import Center, Vertex

pytestmark = pytest.mark.gpu
N, BAND = 65534, 2048   # the Launcher box is N + 2 = 2^16 points a side


@pytest.fixture(scope="module")
def arch():
    return chmy.Arch(chmy.MI355XBackend())


def test_box_of_2_to_the_32_points(arch):
    """maxloc (flat per-point kernels) and left (the operators' kernel)."""
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 80 GB of free device memory")
    g = chmy.UniformGrid(arch, origin=(0.0, 0.0), extent=(1.0, 1.0), dims=(N, N))
    launch = chmy.Launcher(arch, g)
    src = chmy.Field(arch, g, (Center(), Center()), torch.float32)
    s = src.data
    cols = torch.arange(s.shape[1], device=s.device, dtype=torch.int32)
    for r in range(0, s.shape[0], BAND):
        rows = torch.arange(r, min(r + BAND, s.shape[0]), device=s.device, dtype=torch.int32)
        s[r:r + BAND] = ((rows[:, None] * 7919 + cols[None, :] * 104729) % 65521).float()
    for loc, kernel, args in (((Center(), Center()), chmy.kernels.maxloc, ()),
                              ((Vertex(), Center()), chmy.kernels.left, (0, g))):
        dst = chmy.Field(arch, g, loc, torch.float32)
        d = dst.data
        d.fill_(-1.0)
        launch(arch, g, (kernel, (dst, src, *args)))
        # the box 0..N+1 is storage 1..N+2 in both dims
        assert bool((d[0] == -1.0).all()) and bool((d[N + 3] == -1.0).all())
        for r in range(1, N + 3, BAND):
            e = min(r + BAND, N + 3)
            if kernel is chmy.kernels.left:
                want = s[r:e, 0:N + 2]
            else:
                a = torch.maximum(torch.maximum(s[r - 1:e - 1], s[r:e]), s[r + 1:e + 1])
                want = torch.maximum(torch.maximum(a[:, 0:N + 2], a[:, 1:N + 3]), a[:, 2:N + 4])
            assert torch.equal(d[r:e, 1:N + 3], want), f"{kernel.name} rows {r}..{e - 1}"
            assert bool((d[r:e, 0] == -1.0).all()) and bool((d[r:e, N + 3:] == -1.0).all())
        del dst, d
    del src, s
    torch.cuda.empty_cache()
