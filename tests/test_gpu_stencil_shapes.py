"""Stencils at the edges of their launch shapes: the lane splits of the one-lane-per-value kernels
(64, 32 or 16 lanes along the fastest axis, components innermost) and, from 2^20 cells on, the
marching kernels with tiles cut along k, along j and along both. Bit-exact against the oracle."""
import ctypes

import numpy as np
import pytest

import dare_amd as da
import oracle as orc
from conftest import bits_equal

pytestmark = pytest.mark.gpu

SHAPES = [([5, 7, 65], 1), ([4, 3, 17], 1), ([3, 6, 22], 3), ([2, 5, 16], 2), ([33, 65], 1), ([9, 21], 3), ([67], 2),
          ([24, 24, 24], 1), ([2, 2, 5], 1), ([130, 90, 97], 1), ([110, 121, 128], 1), ([128, 64, 130], 1)]


@pytest.mark.parametrize("lim", [da.VANLEER, da.MINMOD])
@pytest.mark.parametrize("n,ncomp", SHAPES)
def test_stencils_match_oracle(ctx, rng, n, ncomp, lim):
    import torch
    go = orc.grid(n, size=[0.7 + 0.2 * d for d in range(len(n))], ghost=2, ncomp=ncomp)
    g = da.Grid()
    ctypes.memmove(ctypes.byref(g), ctypes.byref(go), ctypes.sizeof(g))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    host = lambda t: t.cpu().numpy()
    phi = rng.normal(size=orc.lib().orc_num_cells_padded(ctypes.byref(go)) * ncomp)
    phi[rng.uniform(size=phi.size) < 0.2] = 1.0          # flat patches: 0/0 and infinite ratios
    modes = [[da.GHOST_DIRICHLET, da.GHOST_NEUMANN, da.GHOST_CONSTANT, da.GHOST_LEAVE][f % 4] for f in range(2 * len(n))]
    values = [0.25 * f for f in range(6)]
    filled = orc.ghost_fill(go, phi, modes, values)
    pd = dev(phi)
    da.ghost_fill(ctx, g, pd, modes, values)
    assert bits_equal(host(pd), filled)
    vel = [rng.uniform(-1, 1, size=orc.lib().orc_num_faces(ctypes.byref(go), d)) for d in range(len(n))]
    vd = [dev(v) for v in vel]
    out = pd.clone()
    da.tvd_explicit_step(ctx, g, lim, pd, vd, 1e-3, out)
    assert bits_equal(host(out), orc.tvd_explicit_step(go, lim, filled, vel, 1e-3))
    exp = orc.grad_faces(go, filled)
    fd = [torch.full((e.size,), np.nan, dtype=torch.float64, device="cuda") for e in exp]
    da.grad_faces(ctx, g, pd, fd)
    for d in range(len(n)):
        assert bits_equal(host(fd[d]), exp[d]), d
    div = torch.zeros_like(pd)
    da.div_faces(ctx, g, fd, div)
    assert bits_equal(host(div), orc.div_faces(go, exp))
    if lim == da.VANLEER:
        exp = orc.tvd_face_flux(go, lim, filled, vel)
        da.tvd_face_flux(ctx, g, lim, pd, vd, fd)
        for d in range(len(n)):
            assert bits_equal(host(fd[d]), exp[d]), d
        x = rng.normal(size=g.num_cells * ncomp)
        f2 = pd.clone()
        da.copy_to_field(ctx, g, dev(x), f2)
        assert bits_equal(host(f2), orc.copy_to_field(go, x, filled))


@pytest.mark.parametrize("n,ncomp", [([61, 67, 87], 3), ([64, 65, 127], 2), ([1025, 1027], 1), ([513, 700], 3),
                                     ([1048577], 1), ([700001], 2), ([1, 1, 1], 1), ([2, 1, 1], 3), ([3, 2], 2),
                                     ([161, 162, 163], 1), ([66000, 4, 5], 1), ([3, 263000, 2], 1)])
def test_paired_gradient_and_divergence_match_oracle(ctx, rng, n, ncomp):
    """A lane takes two neighbours of a line of cells and components: odd and even lines, the pair that
    ends one cell and starts the next, and the last cell's far faces."""
    import torch
    go = orc.grid(n, size=[0.7 + 0.2 * d for d in range(len(n))], ghost=2, ncomp=ncomp)
    g = da.Grid()
    ctypes.memmove(ctypes.byref(g), ctypes.byref(go), ctypes.sizeof(g))
    phi = rng.normal(size=orc.lib().orc_num_cells_padded(ctypes.byref(go)) * ncomp)
    pd = torch.from_numpy(phi).cuda()
    exp = orc.grad_faces(go, phi)
    fd = [torch.full((e.size,), np.nan, dtype=torch.float64, device="cuda") for e in exp]
    da.grad_faces(ctx, g, pd, fd)
    for d in range(len(n)):
        assert bits_equal(fd[d].cpu().numpy(), exp[d]), d
    div = torch.zeros_like(pd)
    da.div_faces(ctx, g, fd, div)
    assert bits_equal(div.cpu().numpy(), orc.div_faces(go, exp))


@pytest.mark.parametrize("n,ncomp", [([40, 112, 240], 1), ([11, 333, 301], 1), ([21, 161, 163], 2), ([13, 167, 173], 3),
                                     ([9, 113, 1031], 1)])
def test_gradient_and_divergence_dealt_to_the_dies_match_oracle(ctx, rng, n, ncomp):
    """From 2^20 entries a plane's tiles go to the dies in runs that move on every eight planes: 28 tiles
    and more, run lengths that differ by one tile, a last group of planes cut short."""
    test_paired_gradient_and_divergence_match_oracle(ctx, rng, n, ncomp)


@pytest.mark.parametrize("lim", [da.CDS, da.UPWIND])
@pytest.mark.parametrize("n,ncomp", [([5, 7, 65], 1), ([3, 6, 22], 3), ([33, 65], 2), ([67], 1), ([130, 90, 97], 1),
                                     ([200, 121, 150], 1)])
def test_limiters_of_one_value_match_oracle(ctx, rng, n, ncomp, lim):
    """The step of CDS and UPWIND reads the next neighbours alone; on the march (the last two shapes, 8 and
    19 planes a work-group) it loads the next plane ahead only where the march is long."""
    test_stencils_match_oracle(ctx, rng, n, ncomp, lim)


def test_tvd_step_of_more_planes_than_a_launch_takes(ctx, rng):
    """Fewer cells than the march starts at, but more planes than a grid's third extent."""
    import torch
    n = [66000, 3, 5]
    go = orc.grid(n, size=[66.0, 0.3, 0.5], ghost=2)
    g = da.Grid()
    ctypes.memmove(ctypes.byref(g), ctypes.byref(go), ctypes.sizeof(g))
    phi = rng.normal(size=orc.lib().orc_num_cells_padded(ctypes.byref(go)))
    vel = [rng.uniform(-1, 1, size=orc.lib().orc_num_faces(ctypes.byref(go), d)) for d in range(3)]
    pd, vd = torch.from_numpy(phi).cuda(), [torch.from_numpy(v).cuda() for v in vel]
    out = pd.clone()
    da.tvd_explicit_step(ctx, g, da.VANLEER, pd, vd, 1e-3, out)
    assert bits_equal(out.cpu().numpy(), orc.tvd_explicit_step(go, da.VANLEER, phi, vel, 1e-3))


@pytest.mark.parametrize("lim", [da.MINMOD, da.VANLEER, da.UPWIND])
def test_streaming_tvd_march_matches_oracle(ctx, rng, lim):
    """From 4 M cells on the march streams, without loads a plane ahead for minmod; tiles cut along k and j."""
    test_stencils_match_oracle(ctx, rng, [131, 165, 195], 1, lim)
