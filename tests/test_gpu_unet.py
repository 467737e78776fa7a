"""Learned initial guess on the GPU: the MFMA operand layout, the network's forward pass,
loss and every parameter gradient against the CPU oracle (oracle/unet_oracle.py with the
GPU's bf16 rounding points), and training on solver-generated pairs with the solver run
from the network's x0."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
import unet_oracle as UO  # noqa: E402

pytestmark = pytest.mark.gpu


def test_mfma_operand_layout(gpu):
    X = gpu
    rng = np.random.default_rng(0)
    a = rng.integers(-8, 9, size=(16, 32)).astype(np.float32)
    b = rng.integers(-8, 9, size=(32, 16)).astype(np.float32)
    assert np.array_equal(X.mfma_selftest(a, b), a @ b)  # small integers: exact


def layer_slices(channels):
    shapes = []
    for l in range(len(channels)):
        shapes += [(1 if l == 0 else channels[l - 1], channels[l]), (channels[l], channels[l])]
    for l in range(len(channels) - 1):
        shapes += [(channels[l + 1], channels[l]), (channels[l], channels[l])]
    out, o = [], 0
    for a, b in shapes:
        out.append(slice(o, o + 27 * a * b))
        o += 27 * a * b
        out.append(slice(o, o + b))
        o += b
    out.append(slice(o, o + channels[0] + 1))
    return out


@pytest.mark.parametrize("channels,size,batch", [((16, 32, 48), 8, 2),
                                                 ((16, 32, 48, 64), 8, 1),
                                                 ((16,), 6, 3),
                                                 # 64^3: the 16-channel convolutions run
                                                 # on LDS-staged tiles
                                                 ((16, 32), 64, 1)])
def test_loss_and_gradients_match_oracle(gpu, channels, size, batch):
    X = gpu
    net = X.UNet(channels, seed=7)
    p = net.get_params()
    # non-zero biases so that every bias path is exercised
    rng = np.random.default_rng(1)
    for sl in layer_slices(channels)[1::2]:
        p[sl] = rng.standard_normal(sl.stop - sl.start).astype(np.float32) * 0.1
    net.set_params(p)
    x = rng.standard_normal((batch, size, size, size)).astype(np.float32)
    t = rng.standard_normal((batch, size, size, size)).astype(np.float32)
    loss, g, y = net.loss_grad(x, t)
    ref = UO.UNet(channels, p.astype(np.float64))
    rloss, rg, ry = ref.loss_grad(x.astype(np.float64), t.astype(np.float64), use_bf16=True)
    assert abs(loss - rloss) <= 1e-3 * rloss
    assert np.linalg.norm(y - ry) <= 1e-2 * np.linalg.norm(ry)
    for sl in layer_slices(channels):
        gg, rr = g[sl], rg[sl]
        assert np.linalg.norm(gg - rr) <= 3e-2 * np.linalg.norm(rr) + 1e-9, sl


@pytest.mark.parametrize("channels,dims", [
    ((16, 32, 48, 64), (3, 8, 16, 24)),  # levels down to 1 x 2 x 3 voxels, several samples
    ((16, 32), (2, 6, 8, 32)),           # tiles of 32-voxel lines, data gradients too
    ((64,), (1, 5, 3, 7)),               # one level, no edge a power of two
    ((48, 16), (2, 6, 10, 34)),          # lines just over a box edge, 16 -> 48 upsampling
    ((32, 64), (1, 2, 2, 66)),
])
def test_gradients_on_ragged_volumes(gpu, channels, dims):
    # the weight gradient's boxes overhang these volumes.  Bound: bf16 operands (2^-9 each,
    # two per product) and activations rounded once per layer give about 1e-2 per tensor,
    # the bar of the test above
    X = gpu
    net = X.UNet(channels, seed=3)
    rng = np.random.default_rng(2)
    p = net.get_params()
    for sl in layer_slices(channels)[1::2]:
        p[sl] = rng.standard_normal(sl.stop - sl.start).astype(np.float32) * 0.1
    net.set_params(p)
    x = rng.standard_normal(dims).astype(np.float32)
    t = rng.standard_normal(dims).astype(np.float32)
    loss, g, y = net.loss_grad(x, t)
    ref = UO.UNet(channels, p.astype(np.float64))
    rloss, rg, ry = ref.loss_grad(x.astype(np.float64), t.astype(np.float64), use_bf16=True)
    assert abs(loss - rloss) <= 1e-3 * rloss
    assert np.linalg.norm(y - ry) <= 1e-2 * np.linalg.norm(ry)
    for sl in layer_slices(channels):
        assert np.linalg.norm(g[sl] - rg[sl]) <= 3e-2 * np.linalg.norm(rg[sl]) + 1e-9, sl


def test_training_and_solver_from_learned_x0(gpu):
    X = gpu
    N, nv = 32, 8
    row, col, val, _ = X.varcoef7(N, sigma=1.0, seed=3)
    levels = X.Amg(row, col, val, agg_num_levels=2, num_paths=2, coarse_size=500).export()
    prm = X.default_params(method="MergedPBiCGStab", smoother="Chebyshev", poly_order=4,
                           rel_tol=1e-8, max_iters=100)
    S = X.Solver(X.Hier(levels), prm, nv)
    pairs = []
    for q in range(6):
        b = X.rhs_bumps(100 + q, N, N, N, nv)
        db, dx = X.DeviceArray.from_host(b), X.DeviceArray(N ** 3 * nv)
        S.solve_device(db, dx)
        assert S.stats()[1].all()
        pairs.append((db, dx))
    net = X.UNet((16, 32, 48, 64), seed=1)
    hist = net.train(N, N, N, pairs, nv, crop=16, batch=8, steps=200, lr=2e-3, seed=5)
    assert np.isfinite(hist).all()
    assert hist[-20:].mean() < 0.5 * hist[:20].mean()
    # held-out right-hand sides: the error of x0 against the solver's solution (the
    # residual b - A x0 is not the measure: A scales the high-frequency part of the error
    # by up to 12/h^2, and that part is what the smoother removes first)
    b = X.rhs_bumps(999, N, N, N, nv)
    db = X.DeviceArray.from_host(b)
    dx0 = X.DeviceArray(N ** 3 * nv)
    net.infer(N, N, N, nv, db, dx0)
    x0 = dx0.to_host().reshape(-1, nv)
    it = {}
    sol = {}
    for name, start in (("zero", None), ("learned", x0.reshape(-1))):
        dx = X.DeviceArray.from_host(start) if start is not None else X.DeviceArray(N ** 3 * nv)
        S.solve_device(db, dx)
        st = S.stats()
        assert st[1].all()
        it[name] = st[0]
        sol[name] = dx.to_host().reshape(-1, nv)
    xs = sol["zero"]
    err = np.linalg.norm(x0 - xs, axis=0) / np.linalg.norm(xs, axis=0)
    # a short training run (200 steps on 16^3 crops of 48 pairs) already removes an
    # iteration; the error of x0 is reported, not bounded
    print("relative error of x0 per RHS:", np.round(err, 3), "iterations:", it)
    assert np.isfinite(err).all()
    assert it["learned"] <= it["zero"], it
    # both starts reach the same solution to the solver's tolerance
    assert (np.abs(sol["learned"] - xs).max(0) / np.abs(xs).max(0)).max() < 1e-6


def test_fused_upsampling_inference_is_identical(gpu):
    # inference reads the decoder's upsampled inputs through the convolution (no
    # upsampled tensor is written); the arithmetic is that of the materialised path
    X = gpu
    net = X.UNet((16, 32, 48), seed=3)
    net.output_scale = 0.5
    for n, nv in ((16, 3), (64, 2)):
        b = X.DeviceArray.from_host(np.random.default_rng(n).standard_normal(n ** 3 * nv))
        outs = []
        for fuse in (0, 1):
            X.set_option("unet_fuse_up", fuse)
            x = X.DeviceArray(n ** 3 * nv)
            net.infer(n, n, n, nv, b, x)
            outs.append(x.to_host())
        X.set_option("unet_fuse_up", 1)
        assert np.isfinite(outs[0]).all() and np.abs(outs[0]).max() > 0
        assert np.array_equal(outs[0], outs[1])


def test_upsampled_inputs_are_made_on_demand(gpu):
    # buffers of one shape first used with the fused upsampling, which needs no upsampled
    # tensors, then without it: inference and gradients are the same
    X = gpu
    net, n, nv = X.UNet((16, 32, 48), seed=4), 16, 2
    rng = np.random.default_rng(1)
    b = X.DeviceArray.from_host(rng.standard_normal(n ** 3 * nv))
    x, t = (rng.standard_normal((nv, n, n, n)).astype(np.float32) for _ in range(2))
    outs = []
    try:
        for fuse in (1, 0, 1):
            X.set_option("unet_fuse_up", fuse)
            o = X.DeviceArray(n ** 3 * nv)
            net.infer(n, n, n, nv, b, o)
            outs.append((o.to_host(),) + net.loss_grad(x, t)[1:])
    finally:
        X.set_option("unet_fuse_up", 1)
    assert np.abs(outs[0][0]).max() > 0
    for q in outs[1:]:
        for u, v in zip(outs[0], q):
            assert np.array_equal(u, v)


def test_tiled_convolution_is_identical(gpu):
    # forward convolutions with 16 or 32 output channels on volumes with w % 64 == h % 4 ==
    # d % 2 == 0 (48 channels: w % 32 == 0) read their input from LDS-staged tiles (plain,
    # and through the fused upsampling); products, k order and epilogue are those of the
    # per-tap gathers, so the result is bit-identical
    X = gpu
    try:
        # level-1 tiles (32 output channels) on the 128 x 32 x 16 grid: 16 -> 32, 32 -> 32
        # (2-line tiles) and the upsampled 48 -> 32 and 32 -> 32; level-2 tiles (48 output
        # channels, lines of 32 voxels): 32 -> 48, 48 -> 48 and the upsampled 64 -> 48
        for ch, fuse in (((16, 32, 48), 1), ((16, 32, 48), 0), ((16, 16, 32), 1),
                         ((16, 32, 32), 1), ((16, 32, 48, 64), 1)):
            net = X.UNet(ch, seed=5)
            net.output_scale = 0.5
            X.set_option("unet_fuse_up", fuse)
            for (nx, ny, nz), nv in (((64, 64, 64), 2), ((128, 32, 16), 3)):
                V = nx * ny * nz
                b = X.DeviceArray.from_host(np.random.default_rng(nx + nv).standard_normal(V * nv))
                outs = []
                for tile in (0, 1):
                    X.set_option("unet_conv_tile", tile)
                    x = X.DeviceArray(V * nv)
                    net.infer(nx, ny, nz, nv, b, x)
                    outs.append(x.to_host())
                assert np.isfinite(outs[0]).all() and np.abs(outs[0]).max() > 0
                assert np.array_equal(outs[0], outs[1]), (ch, fuse, nx, ny, nz)
    finally:
        X.set_option("unet_conv_tile", 1)
        X.set_option("unet_fuse_up", 1)


def test_narrow_tiles_are_identical(gpu):
    # 32-voxel lines (w % 64 != 0): tiles against the per-tap gathers, one z step per workgroup
    X = gpu
    net = X.UNet((16, 32), seed=5)
    try:
        for (nx, ny, nz), nv in (((32, 8, 8), 1), ((96, 16, 24), 4), ((32, 32, 32), 16)):
            V = nx * ny * nz
            b = X.DeviceArray.from_host(np.random.default_rng(nx + nv).standard_normal(V * nv))
            outs = []
            for tile in (0, 1):
                X.set_option("unet_conv_tile", tile)
                x = X.DeviceArray(V * nv)
                net.infer(nx, ny, nz, nv, b, x)
                outs.append(x.to_host())
            assert np.array_equal(outs[0], outs[1]), (nx, ny, nz)
    finally:
        X.set_option("unet_conv_tile", 1)


@pytest.mark.parametrize("channels,nx,ny,nz,nv", [
    ((32,), 64, 32, 32, 1),      # 512 workgroups of 128 voxels: three k steps ahead
    ((32,), 64, 32, 36, 1),      # more: own loads
    ((48,), 32, 8, 8, 1), ((48,), 32, 32, 36, 2), ((16, 32), 128, 64, 24, 1)])
def test_gather_convolution_by_size_is_identical(gpu, channels, nx, ny, nz, nv):
    # the per-tap gathers that load k steps ahead and those that do not, against the tiles
    X = gpu
    net, V = X.UNet(channels, seed=11), nx * ny * nz
    b = X.DeviceArray.from_host(np.random.default_rng(nz).standard_normal(V * nv))
    outs = []
    try:
        for tile in (0, 1):
            X.set_option("unet_conv_tile", tile)
            x = X.DeviceArray(V * nv)
            net.infer(nx, ny, nz, nv, b, x)
            outs.append(x.to_host())
    finally:
        X.set_option("unet_conv_tile", 1)
    assert np.isfinite(outs[0]).all() and np.abs(outs[0]).max() > 0
    assert np.array_equal(outs[0], outs[1])


def net16(X, seed):
    """one level of 16 channels (1 -> 16 and 16 -> 16) with non-zero biases"""
    net = X.UNet((16,), seed=seed)
    p = net.get_params()
    rng = np.random.default_rng(seed)
    for sl in layer_slices((16,))[1::2]:
        p[sl] = rng.standard_normal(sl.stop - sl.start).astype(np.float32) * 0.1
    net.set_params(p)
    return net


@pytest.mark.parametrize("nx,ny,nz,nv,mz", [
    # lines of 64 voxels, 512 voxels per tile
    (128, 128, 128, 1, 2), (128, 128, 64, 4, 4), (128, 128, 64, 8, 8),
    (64, 64, 12, 64, 2), (64, 64, 20, 64, 2), (64, 64, 24, 64, 4),
    # lines of 32, 256 voxels per tile
    (32, 64, 12, 64, 2), (96, 32, 16, 64, 4), (32, 64, 32, 64, 8), (32, 64, 24, 64, 4)])
def test_marching_tile_is_identical(gpu, nx, ny, nz, nv, mz):
    # the 16 -> 16 convolution walks mz z steps of 2 planes over its ring of 4 planes: mz
    # doubles up to 8 while it divides nz / 2 and at least 2048 workgroups are left
    X = gpu
    tiles, m = nx * ny * nz * nv // (512 if nx % 64 == 0 else 256), 1
    while m < 8 and (nz // 2) % (2 * m) == 0 and tiles // (2 * m) >= 2048:
        m *= 2
    assert m == mz
    net, V = net16(X, 7), nx * ny * nz
    b = X.DeviceArray.from_host(np.random.default_rng(nx + nz).standard_normal(V * nv))
    outs = []
    try:
        for tile in (0, 1):
            X.set_option("unet_conv_tile", tile)
            x = X.DeviceArray(V * nv)
            net.infer(nx, ny, nz, nv, b, x)
            outs.append(x.to_host())
    finally:
        X.set_option("unet_conv_tile", 1)
    assert np.isfinite(outs[0]).all() and np.abs(outs[0]).max() > 0
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("n,d,h,w", [(64, 24, 32, 32), (64, 16, 32, 64), (64, 32, 32, 32)])
def test_marching_tile_gradients_are_identical(gpu, n, d, h, w):
    # the same kernel on a data gradient, through the relu's mask (2, 2 and 4 z steps)
    X = gpu
    net, rng = net16(X, 8), np.random.default_rng(d)
    x, t = (rng.standard_normal((n, d, h, w)).astype(np.float32) for _ in range(2))
    outs = []
    try:
        for tile in (0, 1):
            X.set_option("unet_conv_tile", tile)
            outs.append(net.loss_grad(x, t))
    finally:
        X.set_option("unet_conv_tile", 1)
    assert outs[0][0] == outs[1][0]
    assert np.abs(outs[0][1]).max() > 0 and np.array_equal(outs[0][1], outs[1][1])
    assert np.array_equal(outs[0][2], outs[1][2])


@pytest.mark.parametrize("nv", [2, 3])
def test_inference_matches_oracle_forward(gpu, nv):
    # x0[:, k] = rms(b[:, k]) * o * net(b[:, k] / rms(b[:, k])) on a grid the LDS-staged
    # convolution tiles cover (the single-channel input layer included); nv = 2 takes the
    # vector head, nv = 3 the per-element one
    X = gpu
    channels = (16, 32)
    net = X.UNet(channels, seed=9)
    p = net.get_params()
    rng = np.random.default_rng(4)
    for sl in layer_slices(channels)[1::2]:
        p[sl] = rng.standard_normal(sl.stop - sl.start).astype(np.float32) * 0.1
    net.set_params(p)
    net.output_scale = 0.7
    nx, ny, nz = 64, 16, 8
    V = nx * ny * nz
    b = rng.standard_normal((V, nv))
    x0 = X.DeviceArray(V * nv)
    net.infer(nx, ny, nz, nv, X.DeviceArray.from_host(b.ravel()), x0)
    got = x0.to_host().reshape(V, nv)
    scale = np.sqrt((b ** 2).mean(0))
    inp = (b / scale).T.reshape(nv, nz, ny, nx)
    ref = UO.UNet(channels, p.astype(np.float64))
    _, _, ry = ref.loss_grad(inp, np.zeros_like(inp), use_bf16=True)
    exp = (scale[:, None] * 0.7 * ry.reshape(nv, V)).T
    assert np.linalg.norm(got - exp) <= 1e-2 * np.linalg.norm(exp)
