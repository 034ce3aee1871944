"""GPU tests of the 16-lane stencil passes and of the claim finisher where
they can go wrong: few particles, more neighbours than the scan's list holds,
radii of several sizes, and chains of claims as long as a set, in the
finisher's on-chip and its global form; all against the oracle bit for bit."""
import ctypes as C

import numpy as np
import pytest
import torch

from granular_gpu_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _scene(pos, mass, cells):
    n = pos.shape[0]
    L = float(scenes.CELL_LENGTH)
    return scenes.Scene(name="t", pos=pos.astype(np.float32), vel=np.zeros((n, 3), np.float32),
                        mass=mass.astype(np.float32), boundary=np.zeros((1, 3), np.float32) + 0.01,
                        space=tuple(L * c for c in cells), cell_length=scenes.CELL_LENGTH,
                        cells=cells, dt=np.float32(0.002), gravity=(0.0, -9.8, 0.0),
                        density=scenes.DENSITY_R001, radius=0.01)


def _cloud(n, seed, crowd):
    rng = np.random.default_rng(seed)
    cells = (6, 5, 7)
    pos = rng.random((n, 3)) * (np.array(cells) * float(scenes.CELL_LENGTH))
    pos[: int(crowd * n)] = 0.1 + 0.06 * rng.random((int(crowd * n), 3))
    return _scene(pos, rng.choice([0.125, 1.0, 2.0, 8.0], n), cells)


def _lines(lines, length):
    # cand[i] = i + 1 along each line: every claim waits for the one before
    z = 0.02 + 0.03 * np.arange(length)
    pos = np.concatenate([np.stack([np.full(length, 0.02 + 0.05 * k), np.full(length, 0.02), z], 1)
                          for k in range(lines)])
    L = float(scenes.CELL_LENGTH)
    cells = (int(0.05 * lines / L) + 2, 1, int(z[-1] / L) + 2)
    return _scene(pos, np.ones(pos.shape[0]), cells)


def _sorted_sim(s):
    from granular_gpu_amd.device import AdaptiveSim
    sim = AdaptiveSim(s)
    sim.grid_build()
    torch.cuda.synchronize()
    n = sim.n
    g = lambda t: t[:n].cpu().numpy().copy()
    return sim, g(sim.pos), g(sim.vel), g(sim.mass), sim.cs.cpu().numpy()


def _mark(sim, max_mass=4.0):
    from granular_gpu_amd import _lib
    from granular_gpu_amd.device import _ptr, _stream
    _lib.check("gg_merge_mark", sim.lib.gg_merge_mark(
        C.byref(sim.set), C.byref(sim.ad), _ptr(sim.cs), max_mass, C.byref(sim.ws), _stream()))
    n = sim.n
    return (sim.remove[:n].cpu().numpy(), sim.merge[:n].cpu().numpy(), sim.mv[:n].cpu().numpy())


def _oracle_mark(s, pos, vel, mass, surf, sd, cs, max_mass=4.0):
    n = pos.shape[0]
    rem, mer, mv = np.zeros(n, np.int32), np.zeros(n, np.float32), np.zeros((n, 3), np.float32)
    po.load().oracle_merge_mark(n, pos.reshape(-1), mass, vel.reshape(-1), surf, sd, rem, mer,
                                mv.reshape(-1), cs, po.params_from(s, 3, 5), max_mass, None, None)
    return rem, mer, mv


@pytest.mark.parametrize("n,crowd", [(1, 0), (3, 0), (5, 1), (61, 0.5), (700, 0.0), (1500, 0.4),
                                     (2200, 0.9)])
def test_stencil_passes_equal_oracle(gpu, n, crowd):
    from granular_gpu_amd import _lib
    from granular_gpu_amd.device import _ptr, _stream
    s = _cloud(n, n, crowd)
    sim, pos, vel, mass, cs = _sorted_sim(s)
    p, lib = po.params_from(s, 3, 5), po.load()
    _lib.check("gg_surface", sim.lib.gg_surface(C.byref(sim.set), _ptr(sim.cs),
                                                C.byref(sim.params), C.byref(sim.ws), _stream()))
    _lib.check("gg_surface_distance", sim.lib.gg_surface_distance(
        C.byref(sim.set), _ptr(sim.cs), C.byref(sim.ws), _stream()))
    cover, surf, sd = np.zeros((n, 3), np.float32), np.zeros(n, np.int32), np.zeros(n, np.float32)
    lib.oracle_surface(n, pos.reshape(-1), mass, cs, p, cover.reshape(-1), surf)
    lib.oracle_surface_distance(n, pos.reshape(-1), surf, cs, p, sd)
    assert np.array_equal(sim.surface[:n].cpu().numpy(), surf)
    assert np.array_equal(sim.sd[:n].cpu().numpy(), sd)
    # marking with every particle deep, so that the crowd takes part
    surf[:], sd[:] = 0, 1e5
    sim.surface[:n], sim.sd[:n] = 0, 1e5
    for a, b in zip(_mark(sim, 16.0), _oracle_mark(s, pos, vel, mass, surf, sd, cs, 16.0)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [262144, 262145, 270001])
def test_surface_distance_on_both_sides_of_its_rule(gpu, n):
    # (16 lanes a particle up to 262,144, one above)
    from granular_gpu_amd import _lib
    from granular_gpu_amd.device import _ptr, _stream
    rng = np.random.default_rng(n)
    cells = (30, 31, 33)
    L = float(scenes.CELL_LENGTH)
    pos = rng.random((n, 3)) * (np.array(cells) * L)
    pos[:2000] = 0.5 + 0.05 * rng.random((2000, 3))
    pos[2000:2100] += 40.0  # outside the grid
    pos[2100] = np.nan
    s = _scene(pos, np.ones(n), cells)
    sim, pos, vel, mass, cs = _sorted_sim(s)
    surf = (rng.random(n) < 0.1).astype(np.int32)
    sim.surface[:n] = torch.from_numpy(surf).cuda()
    _lib.check("gg_surface_distance", sim.lib.gg_surface_distance(
        C.byref(sim.set), _ptr(sim.cs), C.byref(sim.ws), _stream()))
    sd = np.zeros(n, np.float32)
    po.load().oracle_surface_distance(n, pos.reshape(-1), surf, cs, po.params_from(s, 3, 5), sd)
    assert np.array_equal(sim.sd[:n].cpu().numpy(), sd)


def test_positions_and_masses_that_are_not_finite(gpu):
    from granular_gpu_amd import _lib
    from granular_gpu_amd.device import _ptr, _stream
    s = _cloud(900, 4, 0.4)
    s.pos[3], s.pos[40, 1], s.pos[500] = np.nan, np.inf, [1e30, -1e30, 0.1]
    s.mass[[7, 300, 700, 701]] = [np.nan, np.inf, -1.0, 0.0]
    sim, pos, vel, mass, cs = _sorted_sim(s)
    n = s.n
    p, lib = po.params_from(s, 3, 5), po.load()
    _lib.check("gg_surface", sim.lib.gg_surface(C.byref(sim.set), _ptr(sim.cs),
                                                C.byref(sim.params), C.byref(sim.ws), _stream()))
    _lib.check("gg_surface_distance", sim.lib.gg_surface_distance(
        C.byref(sim.set), _ptr(sim.cs), C.byref(sim.ws), _stream()))
    cover, surf, sd = np.zeros((n, 3), np.float32), np.zeros(n, np.int32), np.zeros(n, np.float32)
    lib.oracle_surface(n, pos.reshape(-1), mass, cs, p, cover.reshape(-1), surf)
    lib.oracle_surface_distance(n, pos.reshape(-1), surf, cs, p, sd)
    assert np.array_equal(sim.surface[:n].cpu().numpy(), surf)
    assert np.array_equal(sim.sd[:n].cpu().numpy(), sd)
    surf[:], sd[:] = 0, 1e5
    sim.surface[:n], sim.sd[:n] = 0, 1e5
    for a, b in zip(_mark(sim, 16.0), _oracle_mark(s, pos, vel, mass, surf, sd, cs, 16.0)):
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f")


# the last four leave the launched rounds some hundred thousand claims: in
# chains so long that the finisher goes over to index order at once, after some
# rounds, or never
@pytest.mark.parametrize("lines,length", [(1, 2), (1, 3000), (3, 1365), (5, 1200), (5, 60000),
                                          (300, 1000), (3000, 100), (9000, 30)])
def test_claim_chains_equal_oracle(gpu, lines, length):
    # (up to 4096 undecided claims are finished on chip, more in memory)
    s = _lines(lines, length)
    sim, pos, vel, mass, cs = _sorted_sim(s)
    n = s.n
    surf, sd = np.zeros(n, np.int32), np.full(n, 1e5, np.float32)
    sim.surface[:n], sim.sd[:n] = 0, 1e5
    want = _oracle_mark(s, pos, vel, mass, surf, sd, cs)
    assert (want[0] == -1).sum() >= n - 2 * lines
    t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0.record()
    got = _mark(sim)
    t1.record()
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
    # linear in the claims: about half a microsecond each where they are taken
    # one after another, and a pass over the set; rounds that each take one link
    # of every chain would need a minute for the longest
    assert t0.elapsed_time(t1) < 20.0 + 2e-3 * n
