"""GPU tests of the neighbour-list kernels and the near lists where they can
go wrong: both list kernels (one lane and 16 lanes per particle), rows of
more candidates than a mask or a queue holds, radii of several sizes,
positions outside the grid, grids of one or two cells, and displacements on
both sides of the near lists' bound."""
import numpy as np
import pytest
import torch

from granular_gpu_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _scene(kind, n, seed):
    rng = np.random.default_rng(seed)
    L = float(scenes.CELL_LENGTH)
    cells = {"thin": (1, 2, 40), "one": (1, 1, 1)}.get(kind, (9, 7, 11))
    space = tuple(L * c * 0.999 for c in cells)
    pos = rng.random((n, 3)) * np.array(space)
    mass = np.ones(n, np.float32)
    if kind == "radii":
        mass = rng.choice(np.array([0.125, 1.0, 8.0], np.float32), n)
    if kind == "outside":  # a tenth beyond the walls, some far
        far = rng.random(n) < 0.1
        pos[far] += rng.normal(0.0, 3.0, (int(far.sum()), 3))
        pos[:3] = [[1e6, 0.1, 0.1], [-1e9, 0.1, 0.1], [0.1, 3e7, 0.1]]
    if kind == "dense":    # hundreds in a few cells
        pos[: n // 2] = (0.13 + 0.05 * rng.random((n // 2, 3)))
    vel = rng.normal(0.0, 0.3, (n, 3)).astype(np.float32)
    walls = (rng.random((60, 3)) * np.array(space)).astype(np.float32)
    return scenes.Scene(name=kind, pos=pos.astype(np.float32), vel=vel, mass=mass, boundary=walls,
                        space=space, cell_length=scenes.CELL_LENGTH, cells=cells,
                        dt=np.float32(0.002), gravity=(0.0, -9.8, 0.0),
                        density=scenes.DENSITY_R001, radius=0.01)


CASES = [("box", 1, 3), ("box", 63, 4), ("box", 65, 5), ("box", 4099, 6), ("radii", 4099, 7),
         ("outside", 3000, 8), ("dense", 1500, 9), ("thin", 900, 10), ("one", 70, 11)]


@pytest.mark.parametrize("kind,n,seed", CASES)
@pytest.mark.parametrize("block", [0, 64, 256])  # 0: 16 lanes per particle at these sizes
def test_lists_equal_oracle(gpu, kind, n, seed, block):
    from granular_gpu_amd.device import PlainSim
    s = _scene(kind, n, seed)
    gmax, bmax = 1600, 64
    sim = PlainSim(s, stab=3, solver=5, gmax=gmax, bmax=bmax)
    sim.params.nlist_block = block
    sim.grid_build()
    sim.predict()
    torch.cuda.synchronize()
    cap = sim.cap + 1
    x0, off = sim.view(0, n).cpu().numpy(), sim.view(1, n).cpu().numpy()
    meta = sim.view(2, n, dtype=torch.int32).cpu().numpy()
    gl = sim.view(3, gmax * cap, dtype=torch.int32, width=1).reshape(gmax, cap)[:, :n].cpu().numpy()
    bl = sim.view(4, bmax * cap, dtype=torch.int32, width=1).reshape(bmax, cap)[:, :n].cpu().numpy()
    p = po.params_from(s, skin=0.0075)
    bpos, bcs = po.sorted_boundary(s.boundary, s.cell_length, s.cells)
    ogc, obc, obase = (np.empty(n, np.int32) for _ in range(3))
    ogl, obl = np.empty(n * gmax, np.int32), np.empty(n * bmax, np.int32)
    po.load().oracle_nlist_f32(n, np.ascontiguousarray(x0).reshape(-1),
                               np.ascontiguousarray(off).reshape(-1), bpos.shape[0],
                               bpos.reshape(-1), sim.cs.cpu().numpy(), bcs, p, gmax, bmax, ogc,
                               ogl, obc, obl, obase)
    assert np.array_equal(meta[:, 0], ogc) and np.array_equal(meta[:, 1], obc)
    ogl, obl = ogl.reshape(n, gmax), obl.reshape(n, bmax)
    for i in range(n):
        assert np.array_equal(gl[: min(ogc[i], gmax), i], ogl[i, : min(ogc[i], gmax)])
        assert np.array_equal(bl[: min(obc[i], bmax), i], obl[i, : min(obc[i], bmax)])


@pytest.mark.parametrize("kind,n,seed", CASES)
@pytest.mark.parametrize("mu", [(0.0, 0.0), (0.5, 0.4), (0.0, 0.3)])
def test_steps_equal_oracle(gpu, kind, n, seed, mu):
    # 3 steps of overlapping particles: corrections of millimetres, so near
    # lists, full lists and stencil scans all occur
    from granular_gpu_amd.device import PlainSim
    s = _scene(kind, n, seed)
    sim = PlainSim(s, stab=3, solver=5, mu_s=mu[0], mu_k=mu[1])
    sim.step(3)
    gp, gv, _ = sim.host()
    p = po.params_from(s, 3, 5, mu[0], mu[1])
    bpos, bcs = po.sorted_boundary(s.boundary, s.cell_length, s.cells)
    op, ov = po.plain_steps_f32(s.pos, s.vel, s.mass, bpos, bcs, p, 3)[:2]
    assert np.array_equal(gp, op) and np.array_equal(gv, ov)


@pytest.mark.parametrize("kind,n,seed", CASES)
@pytest.mark.parametrize("nlist_block,sweep_block", [(64, 64), (256, 256), (0, 64), (64, 0)])
@pytest.mark.parametrize("refresh", [False, True])
def test_every_pair_of_kernels_equals_oracle(gpu, kind, n, seed, nlist_block, sweep_block,
                                             refresh):
    # each list build (64, 256: one lane a particle, as for large sets) with
    # each sweep, near lists included; refreshed within the step too
    from granular_gpu_amd._lib import GG_FLAG_LIST_REFRESH
    from granular_gpu_amd.device import PlainSim
    s = _scene(kind, n, seed)
    sim = PlainSim(s, stab=3, solver=5, mu_s=0.5, mu_k=0.4,
                   flags=GG_FLAG_LIST_REFRESH if refresh else 0)
    sim.params.nlist_block, sim.params.sweep_block = nlist_block, sweep_block
    sim.step(3)
    gp, gv, _ = sim.host()
    p = po.params_from(s, 3, 5, 0.5, 0.4)
    bpos, bcs = po.sorted_boundary(s.boundary, s.cell_length, s.cells)
    op, ov = po.plain_steps_f32(s.pos, s.vel, s.mass, bpos, bcs, p, 3)[:2]
    assert np.array_equal(gp, op) and np.array_equal(gv, ov)
