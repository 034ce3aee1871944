"""GPU tests of the list path against the oracle at the ends of its ranges:
radii beyond what the list build's quantised test holds, frictions and masses
outside the short arithmetic's domain, positions that are not finite."""
import numpy as np
import pytest
import torch

from granular_gpu_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _run(s, steps=2, mu=(0.5, 0.4), nlist_block=0, sweep_block=0, flags=0):
    from granular_gpu_amd.device import PlainSim
    sim = PlainSim(s, stab=3, solver=5, mu_s=mu[0], mu_k=mu[1], flags=flags)
    sim.params.nlist_block, sim.params.sweep_block = nlist_block, sweep_block
    sim.step(steps)
    gp, gv, _ = sim.host()
    ctr = sim.view(8, 64, dtype=torch.int32, width=1).reshape(-1).cpu().numpy()
    p = po.params_from(s, 3, 5, *mu)
    bpos, bcs = po.sorted_boundary(s.boundary, s.cell_length, s.cells)
    op, ov = po.plain_steps_f32(s.pos, s.vel, s.mass, bpos, bcs, p, steps)[:2]
    return gp, gv, op, ov, ctr[1:9]


def _equal(a, b):
    return np.array_equal(a, b, equal_nan=True)


def _with_large(side, cells_of_radius, count, seed):
    """A lattice block with `count` particles of a radius of several cells,
    each fast enough to cross some cells within the step: the lists are
    built on the predicted positions, the cells on the present ones."""
    s = scenes.plain_box(side, max(0.7, 0.022 * side), seed=seed)
    rng = np.random.default_rng(seed)
    k = rng.choice(s.n, count, replace=False)
    s.mass[k] = (cells_of_radius * s.cell_length / 0.01) ** 3
    d = rng.normal(size=(count, 3))
    d *= rng.uniform(1.0, 4.5, (count, 1)) * s.cell_length / np.linalg.norm(d, axis=1)[:, None]
    s.vel[k] = d / s.dt
    return s


@pytest.mark.parametrize("nlist_block,sweep_block", [(0, 0), (64, 0), (64, 64), (256, 256)])
@pytest.mark.parametrize("cells_of_radius", [3.5, 4.1, 5.0, 9.0])
def test_radii_of_several_cells(gpu, cells_of_radius, nlist_block, sweep_block):
    s = _with_large(20, cells_of_radius, 20, seed=int(10 * cells_of_radius))
    gp, gv, op, ov, _ = _run(s, 2, (0.5, 0.4), nlist_block, sweep_block)
    assert _equal(gp, op) and _equal(gv, ov)


def test_radii_of_several_cells_at_the_default_kernels_of_large_sets(gpu):
    s = _with_large(41, 5.0, 12, seed=3)
    assert s.n > 65536
    gp, gv, op, ov, _ = _run(s, 1)
    assert _equal(gp, op) and _equal(gv, ov)


def test_scenes_over_a_long_concatenated_table(gpu):
    # ten scenes in grids of 60^3 cells: their tables are one of 2.2 million
    # cells, their positions no larger than one scene's grid
    from granular_gpu_amd.device import SceneBatch
    scs, fr = [], []
    for k in range(10):
        s = scenes.plain_box(6 + k % 5, 2.4, seed=1 + k)
        s.vel[:] = np.random.default_rng(k).normal(0.0, 0.5, s.vel.shape)
        if k == 3:  # some in the grid's far corner
            s.pos[::2] += np.float32(1.9)
        scs.append(s)
        fr.append((0.3 + 0.05 * k, 0.2 + 0.05 * k))
    assert sum(c.cells[0] * c.cells[1] * c.cells[2] for c in scs) > 2_000_000
    for block in (0, 64):
        sb = SceneBatch(scs, fr)
        sb.params.nlist_block = block
        sb.step(6)
        for k, s in enumerate(scs):
            gp, gv, _ = sb.scene(k)
            p = po.params_from(s, 3, 5, *fr[k])
            bpos, bcs = po.sorted_boundary(s.boundary, s.cell_length, s.cells)
            op, ov = po.plain_steps_f32(s.pos, s.vel, s.mass, bpos, bcs, p, 6)[:2]
            assert _equal(gp, op) and _equal(gv, ov), (block, k)


def _pile(side, seed, shake=0.2):
    """A block a little compressed: contacts everywhere, lists mostly valid."""
    s = scenes.plain_box(side, max(0.7, 0.022 * side), seed=seed)
    rng = np.random.default_rng(seed)
    s.pos[:] = (0.15 + 0.97 * (s.pos - 0.15)).astype(np.float32)
    s.vel[:] = rng.normal(0.0, shake, s.vel.shape)
    return s


# (0: four lanes a particle at this size, 64: one)
@pytest.mark.parametrize("sweep_block", [0, 64])
@pytest.mark.parametrize("mu", [(0.5, 1e-7), (0.0, 9e-7), (0.3, 1e-30), (0.5, 3e6), (0.0, 1e20),
                                (0.5, -0.2), (1e25, 0.4)])
def test_frictions_outside_the_short_division(gpu, mu, sweep_block):
    s = _pile(16, 5)
    usual = _run(s, 2, (0.5, 0.4), 0, sweep_block)[4]
    gp, gv, op, ov, scans = _run(s, 2, mu, 0, sweep_block)
    assert _equal(gp, op) and _equal(gv, ov)
    # the lists are used as under an ordinary friction
    assert usual.max() < s.n // 2 and scans.max() < s.n // 2


@pytest.mark.parametrize("sweep_block", [0, 64])
@pytest.mark.parametrize("mass", [np.nan, np.inf, -1.0, 0.0, 1e30])
def test_one_odd_mass_leaves_the_others_their_lists(gpu, mass, sweep_block):
    s = _pile(20, 6)
    # beside a corner: an infinite radius reaches its whole stencil
    k = int(np.argmin(np.abs(s.pos - s.pos.min(axis=0)).sum(axis=1)))
    s.mass[k] = mass
    gp, gv, op, ov, scans = _run(s, 1, (0.5, 0.4), 64 if sweep_block else 0, sweep_block)
    assert _equal(gp, op) and _equal(gv, ov)
    assert scans.max() < s.n // 2


@pytest.mark.parametrize("nlist_block,sweep_block", [(0, 0), (64, 64)])
def test_positions_and_velocities_that_are_not_finite(gpu, nlist_block, sweep_block):
    s = _pile(16, 7)
    s.pos[5], s.pos[77, 1], s.pos[900] = np.nan, np.inf, [1e30, -1e30, 3e38]
    s.vel[11], s.vel[1234, 2], s.vel[2000] = np.nan, -np.inf, [1e25, 0.0, 0.0]
    gp, gv, op, ov, _ = _run(s, 2, (0.5, 0.4), nlist_block, sweep_block)
    assert _equal(gp, op) and _equal(gv, ov)
