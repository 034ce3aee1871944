"""GPU tests of the fused training kernels at the edges of their chunks of 32
samples and tiles of 16, against the oracle's forward and backward."""
import ctypes as C
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _bits(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) & 0xFFFF).astype(np.uint16)


def _case(B):
    rng = np.random.default_rng(B)
    x = _bits(rng.standard_normal((B, 96)))
    t = (0.1 * rng.standard_normal((B, 24))).astype(np.float32)
    xf = (x.astype(np.uint32) << 16).view(np.float32)
    return x.view(np.int16), xf, t


@pytest.mark.parametrize("B", [1, 15, 17, 31, 32, 33, 97, 4129])
def test_forward_and_gradient_at_chunk_edges(gpu, B):
    # the largest difference are bfloat16 roundings flipped where the last
    # bits of the FP32 sums differ from the oracle's 64-bit ones: a sum of 128
    # terms is off by at most 2^-17 of their size, so at most one rounding in
    # 2^-9 / 2^-17 = 256 flips, by 2^-8 of its value: 2^-8 / 16 = 2.4e-4 of a
    # layer's norm, 1e-3 through the seven layers of a forward and a backward
    # pass.  A sample left out of the largest batch is 1 / sqrt(4129) = 1.6e-2
    # of it
    from granular_gpu_amd.learned import MlpNet, Trainer
    net = MlpNet(seed=3)
    tr = Trainer(net, batch=B)
    x, xf, t = _case(B)
    X, T = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    y = tr.forward(X).cpu().numpy()
    dW, db, sq = (v.cpu().numpy() for v in tr.grad(X, T))
    W, b = net.host_bf16()
    oy = po.mlp_forward(xf, W, b)
    loss, odW, odb = po.mlp_backward(xf, W, b, t)
    assert np.abs(y - oy).max() <= 1e-2 * np.abs(oy).max()
    assert sq.shape == (B,) and float(sq.sum()) / (24 * B) == pytest.approx(loss, rel=1e-3)
    for l, (k_in, n_out) in enumerate(po.MLP_DIMS):
        s = slice(po.MLP_WOFF[l], po.MLP_WOFF[l] + k_in * n_out)
        e = slice(po.MLP_BOFF[l], po.MLP_BOFF[l] + n_out)
        assert np.linalg.norm(dW[s] - odW[s]) <= 1e-3 * np.linalg.norm(odW[s])
        assert np.linalg.norm(db[e] - odb[e]) <= 1e-3 * np.linalg.norm(odb[e])


def test_products_keep_their_order(gpu):
    # golden outputs of the layers as separate products, each summed in
    # ascending steps of 16 with the bias added last.  Outputs are the same
    # bits.  Gradients differ by the order of FP32 sums over the samples only,
    # at most 512 2^-24 = 3e-5 of their norm were all terms of one sign and
    # size, typically its square root: 2e-6.  One flipped bfloat16 rounding in
    # a hundred of a layer is 2^-9 / 10 = 2e-4, so 1e-5 keeps them apart.
    from granular_gpu_amd.learned import MlpNet, Trainer, init_master
    want = np.load(Path(__file__).parent / "golden" / "training.npz")
    W, _ = init_master(3)
    b = (0.1 * np.random.default_rng(9).standard_normal(416)).astype(np.float32)
    b[408:] = 0.0
    for B in (33, 512):
        net = MlpNet(master=(W, b))
        tr = Trainer(net, batch=B)
        x, _, t = _case(B)
        X, T = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        if B == 33:
            assert np.array_equal(tr.forward(X).cpu().numpy(), want["y33"])
        else:
            db = tr.grad(X, T)[1].cpu().numpy().astype(np.float64)
            for l, (_, n_out) in enumerate(po.MLP_DIMS):
                e = slice(po.MLP_BOFF[l], po.MLP_BOFF[l] + n_out)
                ref = want["db512"][e].astype(np.float64)
                assert np.linalg.norm(db[e] - ref) <= 1e-5 * np.linalg.norm(ref)


@pytest.mark.parametrize("B", [33, 300])
def test_gradient_does_not_depend_on_scratch_width(gpu, B):
    # one block (no partial gradients), a few, all: the same sums grouped
    # differently, so 1e-5 of the norm (fp32 sums of at most 300 terms);
    # unaligned rows and scratch are accepted like aligned ones
    from granular_gpu_amd import _lib
    from granular_gpu_amd.device import _ptr, _stream
    from granular_gpu_amd.learned import NB, NW, MlpNet
    lib = _lib.load()
    net = MlpNet(seed=5)
    x, _, t = _case(B)
    pad = torch.zeros(B * 96 + 1, dtype=torch.int16, device="cuda")
    pad[1:] = torch.from_numpy(x).cuda().reshape(-1)
    T = torch.from_numpy(t).cuda()
    full = int(lib.gg_mlp_train_scratch_bytes(B))
    low = 5376 * B
    assert full >= low
    ref = None
    for X, size, off in [(pad[1:].clone(), full, 0), (pad[1:], full, 4), (pad[1:].clone(), low, 0),
                         (pad[1:].clone(), min(full, low + 400_000), 8)]:
        buf = torch.empty(size + off, dtype=torch.uint8, device="cuda")
        dW = torch.full((NW,), 7.0, device="cuda")
        db = torch.full((NB,), 7.0, device="cuda")
        _lib.check("gg_mlp_grad", lib.gg_mlp_grad(
            C.byref(net.struct), _ptr(X), _ptr(T), B, _ptr(dW), _ptr(db), None,
            C.c_void_p(buf.data_ptr() + off), size, _stream()))
        got = torch.cat([dW, db]).cpu().numpy().astype(np.float64)
        if ref is None:
            ref = got
        assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)
    buf = torch.empty(full, dtype=torch.uint8, device="cuda")
    assert lib.gg_mlp_grad(C.byref(net.struct), _ptr(pad), _ptr(T), B, _ptr(dW), _ptr(db), None,
                           _ptr(buf), low - 1, _stream()) == -4
