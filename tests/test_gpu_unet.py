"""The U-Net kernels (BF16 on the matrix cores, FP32 accumulation) against a
plain float32 PyTorch statement of the same network on the CPU
(tests/unet_ref.py): the output, the loss and every layer's parameter
gradient, on random inputs and parameters (biases non-zero), for box sizes
that take every tiling of the convolution: one wave per x row with idle
16-voxel groups, two waves (the x shift crosses waves through LDS), eight
and sixteen waves, and output channels split over two launches (1024 voxels
along x).
The bar is BF16's: relative L2 error of the output within 3e-2, of each
layer's gradient within 1e-1 with cosine similarity above 0.99 -- a wrong tap,
a transposed weight block or a misplaced channel slice gives errors of order
one.  A few Adam steps on a fixed batch lower the loss."""
import numpy as np
import pytest

import unet_ref

pytestmark = pytest.mark.gpu


def _setup(pkg, box, nb, seed):
    import torch
    nx, ny, nz = box
    rng = np.random.default_rng(seed)
    U = pkg.unet
    p = U.init_params(seed)
    sl = U.layer_slices()
    for name in U.NAMES + ("out",):
        p[sl[name][1]] = rng.normal(0.0, 0.1, sl[name][1].stop - sl[name][1].start)
    x = rng.standard_normal((nb, 8, nz, ny, nx)).astype(np.float32)
    xb = torch.from_numpy(x).to(torch.bfloat16)
    xp = torch.zeros((nb, nz + 2, ny + 2, nx + 2, 8), dtype=torch.bfloat16)
    xp[:, 1:-1, 1:-1, 1:-1, :] = xb.permute(0, 2, 3, 4, 1)
    # the kernels' weights are BF16: the reference takes the same rounded values
    pr = p.copy()
    for name in U.NAMES + ("out",):
        w = sl[name][0]
        pr[w] = torch.from_numpy(p[w]).to(torch.bfloat16).float().numpy()
    e = rng.standard_normal((nb, nz, ny, nx)).astype(np.float32)
    m = (rng.random((nb, nz, ny, nx)) < 0.7).astype(np.float32)
    return p, pr, xb.float(), xp, e, m


@pytest.mark.parametrize("box,nb", [((64, 8, 8), 2), ((128, 4, 8), 1), ((512, 4, 4), 1),
                                    ((1024, 4, 4), 1)])
def test_unet_forward_and_gradients_match_torch(pkg, box, nb):
    import torch
    U = pkg.unet
    nx, ny, nz = box
    p, pr, xf, xp, e, m = _setup(pkg, box, nb, 3)
    print(f"unet box {box} batch {nb}", flush=True)
    with U.UNet(nx, ny, nz, nb, train=True) as net:
        net.set_params(p)
        net.set_input(xp.cuda())
        y = torch.empty(nb * nz * ny * nx, dtype=torch.float32, device="cuda")
        net.forward(y)
        y = y.cpu().numpy().reshape(nb, nz, ny, nx)
        loss, g = net.gradients(torch.from_numpy(e.ravel()).cuda(), torch.from_numpy(m.ravel()).cuda())
    # an inference network (which stores neither the coarse outputs of the
    # layers it upsamples nor the last hidden layer, only their fused
    # products) gives the same output bit for bit
    with U.UNet(nx, ny, nz, nb, train=False) as net:
        net.set_params(p)
        net.set_input(xp.cuda())
        yi = torch.empty(nb * nz * ny * nx, dtype=torch.float32, device="cuda")
        net.forward(yi)
        yi = yi.cpu().numpy().reshape(nb, nz, ny, nx)
    assert np.array_equal(yi, y)
    prm = unet_ref.forward(U, pr, xf)
    for v in prm.values():
        v[0].requires_grad_(True)
        v[1].requires_grad_(True)
    yr = unet_ref.run(prm, xf)
    ey = np.linalg.norm(y - yr.detach().numpy()) / np.linalg.norm(yr.detach().numpy())
    print(f"output rel L2 {ey:.3e}", flush=True)
    assert ey <= 3e-2
    lr = unet_ref.loss(yr, torch.from_numpy(e), torch.from_numpy(m))
    lr.backward()
    assert abs(loss - lr.item()) <= 3e-2 * lr.item(), (loss, lr.item())
    gr = unet_ref.grad_vector(U, prm, U.param_count())
    sl = U.layer_slices()
    for name in U.NAMES + ("out",):
        for part in (0, 1):
            a, b = g[sl[name][part]], gr[sl[name][part]]
            rel = np.linalg.norm(a - b) / np.linalg.norm(b)
            cos = float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b)))
            print(f"{name} {'wb'[part]}: rel {rel:.3e} cos {cos:.5f}", flush=True)
            assert rel <= 1e-1 and cos >= 0.99, (name, part, rel, cos)


def test_unet_gradients_from_a_given_output_gradient_match_torch(pkg):
    """The backward pass from a caller's output gradient (the residual loss's
    path, cad_unet_gradients_dy): with dy random, every layer's gradient
    against the reference's gradient of sum(dy * y).  This checks the path of
    dy into the backward pass: a dy read in the wrong order or from the wrong
    buffer gives gradients unrelated to the reference's (cosine near 0).  An
    unmasked random dy sums to small gradients through much cancellation,
    which BF16 activations widen, so the bar is relative error 2e-1 and
    cosine 0.98 (measured worst: b3b's bias, 0.146 and 0.9896)."""
    import torch
    U = pkg.unet
    box, nb = (64, 8, 8), 2
    nx, ny, nz = box
    p, pr, xf, xp, e, m = _setup(pkg, box, nb, 5)
    dy = np.random.default_rng(9).standard_normal((nb, nz, ny, nx)).astype(np.float32)
    with U.UNet(nx, ny, nz, nb, train=True) as net:
        net.set_params(p)
        net.set_input(xp.cuda())
        y = torch.empty(nb * nz * ny * nx, dtype=torch.float32, device="cuda")
        net.forward(y)
        g = net.gradients_dy(torch.from_numpy(dy.ravel()).cuda())
    prm = unet_ref.forward(U, pr, xf)
    for v in prm.values():
        v[0].requires_grad_(True)
        v[1].requires_grad_(True)
    yr = unet_ref.run(prm, xf)
    (yr * torch.from_numpy(dy)).sum().backward()
    gr = unet_ref.grad_vector(U, prm, U.param_count())
    sl = U.layer_slices()
    for name in U.NAMES + ("out",):
        for part in (0, 1):
            a, b = g[sl[name][part]], gr[sl[name][part]]
            rel = np.linalg.norm(a - b) / np.linalg.norm(b)
            cos = float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b)))
            print(f"{name} {'wb'[part]}: rel {rel:.3e} cos {cos:.5f}", flush=True)
            assert rel <= 2e-1 and cos >= 0.98, (name, part, rel, cos)


def test_unet_adam_steps_lower_the_loss(pkg):
    import torch
    U = pkg.unet
    box, nb = (64, 8, 8), 2
    p, _, _, xp, e, m = _setup(pkg, box, nb, 5)
    nx, ny, nz = box
    with U.UNet(nx, ny, nz, nb, train=True) as net:
        net.set_params(p)
        net.set_input(xp.cuda())
        t, mk = torch.from_numpy(e.ravel()).cuda(), torch.from_numpy(m.ravel()).cuda()
        losses = [net.train_step(t, mk, 1e-3) for _ in range(40)]
    print(f"loss {losses[0]:.4f} -> {losses[-1]:.4f}", flush=True)
    assert losses[-1] < 0.8 * losses[0]
    assert np.all(np.isfinite(losses))


@pytest.mark.parametrize("box,nb", [((64, 4, 4), 1), ((192, 12, 20), 3), ((320, 36, 4), 1)])
def test_unet_weight_gradients_by_segments_and_runs(pkg, box, nb):
    """The weight gradients' blocks at the edges of their split: one row and
    one 16-voxel segment on the coarsest level, x segments with a remainder
    (96 = 64 + 32 and 160 = 2 x 64 + 32 voxels on the middle level), row runs
    with a remainder, fewer and more units than blocks.  The bar is the one
    above, BF16's (test_unet_weight_gradients_equal_the_exact_sums compares without
    rounding); the partial sums are added in a fixed order, so two calls give the
    same bits, apart from the output layer's 17 sums and what the loss's
    atomic sum moves: dy is given, so nothing."""
    import torch
    U = pkg.unet
    nx, ny, nz = box
    p, pr, xf, xp, e, m = _setup(pkg, box, nb, 7)
    with U.UNet(nx, ny, nz, nb, train=True) as net:
        net.set_params(p)
        net.set_input(xp.cuda())
        y = torch.empty(nb * nz * ny * nx, dtype=torch.float32, device="cuda")
        net.forward(y)
        dy = (2.0 * torch.from_numpy(m).cuda() * (y.view(nb, nz, ny, nx) - torch.from_numpy(e).cuda())).reshape(-1)
        torch.cuda.synchronize()
        g = net.gradients_dy(dy)
        g2 = net.gradients_dy(dy)
    prm = unet_ref.forward(U, pr, xf)
    for v in prm.values():
        v[0].requires_grad_(True)
        v[1].requires_grad_(True)
    yr = unet_ref.run(prm, xf)
    (yr * dy.cpu().view(nb, nz, ny, nx)).sum().backward()
    gr = unet_ref.grad_vector(U, prm, U.param_count())
    sl = U.layer_slices()
    for name in U.NAMES:
        for part in (0, 1):
            a, b = g[sl[name][part]], gr[sl[name][part]]
            rel = np.linalg.norm(a - b) / np.linalg.norm(b)
            print(f"{name} {'wb'[part]}: rel {rel:.3e}", flush=True)
            assert rel <= 1e-1, (name, part, rel)
            assert np.array_equal(a, g2[sl[name][part]]), (name, part)


def _exact_case(pkg, box, nb, seed):
    """Parameters, input and output gradient whose activations and gradients are
    all short binary fractions: an output channel takes one input channel, or one of
    each half, shifted by up to a voxel along x (weight 1, no bias), the input is 0 or 1,
    the output gradient a sparse -1, 0 or 1.  Poolings divide by 8, so every value has
    at most 8 significant bits (BF16 rounds nothing; checked here) and the weight
    gradients' FP32 sums are exact."""
    import torch
    nx, ny, nz = box
    rng = np.random.default_rng(seed)
    U = pkg.unet
    sl = U.layer_slices()
    p = np.zeros(U.param_count(), np.float32)
    for name in U.NAMES:
        w, _, (ci, co) = sl[name]
        k = np.zeros((27, ci, co), np.float32)
        if ci > co:
            chan = np.stack([rng.permutation(co), co + rng.permutation(co)])
        else:
            chan = np.concatenate([rng.permutation(ci) for _ in range(co // ci)])[None]
        for c in chan:
            k[rng.integers(12, 15, co), c, np.arange(co)] = 1.0
        p[w] = k.ravel()
    p[sl["out"][0]] = rng.choice([-1.0, 1.0], 16)
    x = torch.from_numpy((rng.random((nb, 8, nz, ny, nx)) < 0.2).astype(np.float32))
    xp = torch.zeros((nb, nz + 2, ny + 2, nx + 2, 8), dtype=torch.bfloat16)
    xp[:, 1:-1, 1:-1, 1:-1, :] = x.permute(0, 2, 3, 4, 1)
    dy = torch.from_numpy((rng.choice([-1.0, 1.0], (nb, nz, ny, nx)) * (rng.random((nb, nz, ny, nx)) < 0.05)).astype(np.float32))
    prm = unet_ref.forward(U, p, x)
    for v in prm.values():
        v[0].requires_grad_(True)
        v[1].requires_grad_(True)
    seen = []

    def keep(t):
        t.retain_grad()
        seen.append(t)
        return t

    relu, pool, up = torch.relu, torch.nn.functional.avg_pool3d, torch.nn.functional.interpolate
    try:
        torch.relu = lambda h: keep(relu(h))
        torch.nn.functional.avg_pool3d = lambda *a, **k: keep(pool(*a, **k))
        torch.nn.functional.interpolate = lambda *a, **k: keep(up(*a, **k))
        y = unet_ref.run(prm, x)
    finally:
        torch.relu, torch.nn.functional.avg_pool3d, torch.nn.functional.interpolate = relu, pool, up
    (y * dy).sum().backward()
    for t in seen:
        for v in (t.detach(), t.grad):
            assert torch.equal(v.bfloat16().float(), v)
    return p, xp, dy, unet_ref.grad_vector(U, prm, U.param_count())


@pytest.mark.parametrize("box,nb", [((64, 4, 4), 1), ((192, 12, 20), 3), ((320, 36, 4), 1), ((128, 8, 12), 2)])
def test_unet_weight_gradients_equal_the_exact_sums(pkg, box, nb):
    """Weight and bias gradients of every tap and channel, where no rounding takes
    part, equal the reference's: one voxel lost or taken twice at the edge of a
    segment, a run or a plane changes a sum by at least 2^-12.  (Between the BF16
    network and the FP32 one a layer's gradients differ by up to 0.1.)"""
    U = pkg.unet
    nx, ny, nz = box
    p, xp, dy, want = _exact_case(pkg, box, nb, 3)
    with U.UNet(nx, ny, nz, nb, train=True) as net:
        import torch
        net.set_params(p)
        net.set_input(xp.cuda())
        y = torch.empty(nb * nz * ny * nx, dtype=torch.float32, device="cuda")
        net.forward(y)
        g = net.gradients_dy(dy.reshape(-1).cuda())
    sl = U.layer_slices()
    for name in U.NAMES + ("out",):
        for part in (0, 1):
            a, b = g[sl[name][part]], want[sl[name][part]]
            print(f"{name} {'wb'[part]}: {np.count_nonzero(b)} of {b.size} not 0, {np.count_nonzero(a != b)} differ", flush=True)
            assert np.array_equal(a, b), (name, part, np.abs(a - b).max())
