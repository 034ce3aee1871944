"""GPU test of the learned upsampler called from two threads at once, each on
a stream of its own: the results of the calls made one after another."""
import threading

import numpy as np
import pytest
import torch

from granular_gpu_amd import scenes

pytestmark = pytest.mark.gpu


def test_two_threads_on_their_own_streams(gpu):
    from granular_gpu_amd.device import PlainSim
    from granular_gpu_amd.learned import LearnedUpsampler, MlpNet
    net = MlpNet(seed=5)
    sims = []
    for k, side in enumerate((9, 13)):
        sim = PlainSim(scenes.plain_box(side, 1.0, r=0.02, seed=1 + k, dt=0.002, g=-9.8))
        sim.step(100)
        sim.grid_build()
        sims.append(sim)
    ups = [LearnedUpsampler(net) for _ in sims]
    want = [up.infer(sim).cpu().numpy() for up, sim in zip(ups, sims)]
    torch.cuda.synchronize()
    start = threading.Barrier(2)
    got = [[], []]

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            start.wait()
            for _ in range(30):
                got[k].append(ups[k].infer(sims[k]))
        st.synchronize()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        assert len(got[k]) == 30
        for x in got[k]:
            assert np.array_equal(x.cpu().numpy(), want[k])
