"""GPU tests of the cell sort and the stencil passes over it where they can go
wrong: sets on both sides of the large-cell limits, cells of more members
than one thread per entry ranks (the sentinel and one inside), cell tables of
one and of several sub-tiles per scan tile, fine particles at a coarse
particle's or a wall's own position, and the learned upsampler on both sides
of the size from which its flags run beside the features."""
import numpy as np
import pytest
import torch

from granular_gpu_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _set(n, cells, crowd, seed):
    rng = np.random.default_rng(seed)
    L = float(scenes.CELL_LENGTH)
    space = tuple(L * c * 0.999 for c in cells)
    pos = rng.random((n, 3)) * np.array(space)
    pick = rng.permutation(n)
    pos[pick[:crowd]] = L * (1.0 + 0.9 * rng.random((crowd, 3)))        # one cell
    pos[pick[crowd:2 * crowd]] += 1e3                                     # the sentinel
    return scenes.Scene(name="cells", pos=pos.astype(np.float32), vel=np.zeros((n, 3), np.float32),
                        mass=np.ones(n, np.float32),
                        boundary=(rng.random((60, 3)) * np.array(space)).astype(np.float32),
                        space=space, cell_length=scenes.CELL_LENGTH, cells=cells,
                        dt=np.float32(0.002), gravity=(0.0, -9.8, 0.0),
                        density=scenes.DENSITY_R001, radius=0.01)


# (n, cells, members of each of two crowded cells); 90 x 80 x 75 cells are 264
# scan tiles
@pytest.mark.parametrize("n,cells,crowd", [
    (1, (3, 4, 5), 0), (4096, (9, 7, 11), 2000), (4097, (9, 7, 11), 1024), (4097, (9, 7, 11), 1025),
    (5000, (9, 7, 11), 1026), (70001, (40, 30, 35), 30000), (20000, (90, 80, 75), 3000)])
def test_cell_sort_equals_oracle(gpu, n, cells, crowd):
    from granular_gpu_amd.device import PlainSim
    s = _set(n, cells, crowd, n)
    sim = PlainSim(s)
    perm = torch.empty(n, dtype=torch.int32, device="cuda")
    _, want, cs = po.grid_build(s.pos, s.cell_length, s.cells)
    for _ in range(2):  # the scan's and the large cells' counters are left as found
        sim.pos[:n].copy_(torch.from_numpy(s.pos))
        sim.grid_build(perm)
        torch.cuda.synchronize()
        assert np.array_equal(perm.cpu().numpy(), want)
        assert np.array_equal(sim.cs.cpu().numpy(), cs)
        assert np.array_equal(sim.pos[:n].cpu().numpy(), s.pos[want])


@pytest.mark.parametrize("n", [1, 7, 3000])
def test_upsample_at_coincident_positions_bitexact(gpu, n):
    from granular_gpu_amd.device import FineSet, PlainSim
    s = _set(n, (9, 7, 11), 0, 5 + n)
    rng = np.random.default_rng(n)
    s.vel = rng.normal(0.0, 0.3, (n, 3)).astype(np.float32)
    _, perm, cs = po.grid_build(s.pos, s.cell_length, s.cells)
    s.pos, s.vel = np.ascontiguousarray(s.pos[perm]), np.ascontiguousarray(s.vel[perm])
    sim = PlainSim(s)
    sim.cs.copy_(torch.from_numpy(cs).cuda())
    bpos, bcs = po.sorted_boundary(s.boundary, s.cell_length, s.cells)
    f = np.concatenate([s.pos[rng.integers(0, n, 70)], bpos[:40],
                        s.pos[rng.integers(0, n, 40)] + np.float32(1e-20),
                        s.pos[rng.integers(0, n, 90)] + np.float32(0.004)]).astype(np.float32)
    v = rng.normal(0.0, 0.3, f.shape).astype(np.float32)
    fs = FineSet(sim, f, v)
    fs.upsample()
    gp, gv = fs.host()
    rp, rv = po.upsample_plain(f, v, s.pos, s.vel, cs, bpos, bcs, po.params_from(s), steps=1)
    assert np.array_equal(gp, rp) and np.array_equal(gv, rv)


def test_learned_flags_first_or_beside_agree(gpu):
    # 64^3 particles, then one more in the sentinel cell (after them in the
    # order): the other order of launches, the same values for the first 64^3
    from granular_gpu_amd.device import PlainSim
    from granular_gpu_amd.learned import LearnedUpsampler, MlpNet
    m = 64
    rng = np.random.default_rng(3)
    pos = (np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5
           + 0.2 * rng.random((m ** 3, 3))) * 0.02
    up = LearnedUpsampler(MlpNet(seed=7))
    got = []
    for extra in (0, 1):
        n = m ** 3 + extra
        s = _set(n, (33, 33, 33), 0, 1)
        s.boundary = _set(1, (33, 33, 33), 0, 1).boundary  # (of the same draw for both)
        s.pos = np.concatenate([pos, np.full((extra, 3), 50.0)]).astype(np.float32)
        s.vel = np.zeros((n, 3), np.float32)
        s.vel[: m ** 3] = np.random.default_rng(4).normal(0.0, 0.3, (m ** 3, 3))
        sim = PlainSim(s)
        sim.grid_build()
        count = torch.zeros(1, dtype=torch.int32, device="cuda")
        fine = [up.infer(sim, fallback_count=count).cpu().numpy()[: m ** 3] for _ in range(3)]
        assert all(np.array_equal(fine[0], x) for x in fine[1:])
        got.append((fine[0], int(count)))
    assert np.array_equal(got[0][0], got[1][0])
    assert 0 <= got[1][1] - got[0][1] <= 1
