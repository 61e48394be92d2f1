"""GPU: the network's backward pass with the activations' gradients formed by the
kernels that produce them, and batches gathered in one launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference_gradient(N, params, nels, samples, fixed):
    """Loss over the samples (x, f, target) and its gradient by float64 autograd on the
    CPU, per layer (w, b)."""
    import torch
    F = torch.nn.functional
    W, B, off = [], [], 0
    for cin, cout, k, _ in N.NET_LAYERS:
        n = cout * k**3 * cin
        w = N.bf16(params[off:off + n].reshape(cout, k, k, k, cin))
        W.append(torch.tensor(w, dtype=torch.float64, requires_grad=True))
        off += n
        B.append(torch.tensor(params[off:off + cout].astype(np.float64), requires_grad=True))
        off += cout

    def conv(li, t, act=True):
        z = F.conv3d(t, W[li].permute(0, 4, 1, 2, 3), B[li], padding=N.NET_LAYERS[li][3])
        return F.silu(z) if act else z

    pool = lambda t: F.avg_pool3d(t, 2)
    up = lambda t: F.interpolate(t, scale_factor=2, mode="nearest")
    feats = np.concatenate([N.network_features(nels, x, f, fixed) for x, f, _ in samples])
    t = torch.tensor(feats).permute(0, 4, 1, 2, 3)
    s0 = conv(1, conv(0, t))
    s1 = conv(3, conv(2, pool(s0)))
    s2 = conv(5, conv(4, pool(s1)))
    e3 = conv(7, conv(6, pool(s2)))
    d2 = conv(9, conv(8, torch.cat([up(e3), s2], 1)))
    d1 = conv(11, conv(10, torch.cat([up(d2), s1], 1)))
    d0 = conv(13, conv(12, torch.cat([up(d1), s0], 1)))
    out = conv(14, d0, act=False)[:, :3].permute(0, 2, 3, 4, 1).reshape(len(samples), -1)
    targets = np.stack([u.ravel() / np.sqrt(np.mean(u**2)) for _, _, u in samples])
    loss = ((out - torch.tensor(targets)) ** 2).mean()
    loss.backward()
    return loss.item(), [(w.grad.numpy(), b.grad.numpy()) for w, b in zip(W, B)]


def _weights(N, g, gain):
    """He weights, the levels below the finest scaled by `gain`, small random biases: the
    pooled paths carry a good part of the gradient."""
    out = []
    for i, (cin, cout, k, _) in enumerate(N.NET_LAYERS):
        w = g.standard_normal((cout, k**3, cin)) * np.sqrt(2.0 / (k**3 * cin))
        b = 0.1 * g.standard_normal(cout)
        if k == 2:
            w[3:] = b[3:] = 0  # 3 of 8 outputs in use
        if 2 <= i <= 11:
            w *= gain
        out += [w.ravel(), b]
    return np.concatenate(out).astype(np.float32)


def _sample(nels, g, b, load):
    """A sample unlike its neighbours: sparse and dense designs, loads of other sizes,
    smooth displacements of other signs."""
    x = np.clip(0.2 + 0.6 * (b % 2) + 0.2 * g.standard_normal(int(np.prod(nels))), 0.01, 1.0)
    X, Y, Z = (np.arange(n + 1) / n for n in nels)
    u = np.zeros((nels[2] + 1, nels[1] + 1, nels[0] + 1, 3))
    u[..., 1] = (-1) ** b * (1 + b % 5) * X**2 * (3 - X)
    u[..., 0] = X * (2 - X) * (Y[None, :, None] - 0.3)
    u[..., 2] = b % 5 * X**2 * (Z[:, None, None] - 0.5) + 0.3
    return x, load * g.standard_normal(u.size), u.ravel()


# 24x8x16 by the split kernels, 40x32x32 by LDS tiles
@pytest.mark.parametrize("nels,batch,gain", [((8, 8, 8), 3, 1.8), ((24, 8, 16), 3, 1.4),
                                             ((40, 32, 32), 2, 1.0)])
def test_gradient_values(T, gpu, nels, batch, gain):
    """Every layer's gradient over a batch of unlike samples.  BF16 storage of
    activations and their gradients moves it by up to 0.9 % of a layer's norm (float64
    autograd with and without the roundings); half a pooled, skipped or upsampled
    gradient, or another sample's, moves some layer by 10 % and more in the last two
    cases."""
    from oracle import nn_oracle as N
    import topopt_jl_amd.nn as NN
    net = NN.WarmStartNet(nels, max_batch=batch, max_samples=batch)
    g = np.random.default_rng(sum(nels))
    p = _weights(N, g, gain)
    net.set_params(p)
    samples = [_sample(nels, g, b, 0.2 + b) for b in range(batch)]
    for x, f, u in samples:
        net.add_sample(x, f, u)
    loss = net.train(steps=1, batch=batch, lr=1e-30)[0]
    grad = net.get_gradient()
    ref_loss, ref = _reference_gradient(N, p, nels, samples, net.fixed)
    assert abs(loss - ref_loss) < 0.01 * ref_loss
    off = 0
    for li, (w, b) in enumerate(ref):
        for name, r in (("w", w.ravel()), ("b", b)):
            d = grad[off:off + r.size] - r
            off += r.size
            assert np.linalg.norm(d) < 0.03 * np.linalg.norm(r), (li, name)
    assert off == p.size


@pytest.mark.parametrize("nels,batch", [((8, 8, 8), 1), ((24, 8, 16), 3), ((40, 32, 32), 2)])
def test_gradient_signs(T, gpu, nels, batch):
    """The first Adam step moves every parameter by lr against its gradient's sign.
    BF16 storage along 15 layers leaves an error of some percent of a layer's root
    mean square; entries above three quarters of it have their sign."""
    from oracle import nn_oracle as N
    import topopt_jl_amd.nn as NN
    net = NN.WarmStartNet(nels, max_batch=batch, max_samples=1, seed=4)
    g = np.random.default_rng(sum(nels))
    x = g.uniform(0.05, 1.0, net.ncells)
    f = NN.cantilever_load(nels, nels[1] // 2, nels[2] // 2) * 50.0
    f = f + 0.1 * g.standard_normal(f.size)
    u = g.standard_normal(net.nnodes * 3)
    net.add_sample(x, f, u)
    p = net.get_params().copy()
    net.train(steps=1, batch=batch, lr=1e-3, count=1)
    step = net.get_params() - p
    _, ref = _reference_gradient(N, p, nels, [(x, f, u)], net.fixed)
    off = 0
    for li, (w, b) in enumerate(ref):
        for name, r in (("w", w), ("b", b)):
            d = step[off:off + r.size]
            off += r.size
            big = np.abs(r.ravel()) > 0.75 * np.sqrt(np.mean(r**2))
            assert np.array_equal(np.sign(d[big]), -np.sign(r.ravel()[big])), (li, name)
    assert off == p.size


def test_batches_gathered(T, gpu):
    """A batch of more samples than one launch gathers (64): its loss and its gradient
    are the means of the samples' own.  The two samples of the second launch have loads
    that let them dominate both, so that others in their place would show."""
    from oracle import nn_oracle as N
    import topopt_jl_amd.nn as NN
    nels, n = (8, 8, 8), 66
    net = NN.WarmStartNet(nels, max_batch=n, max_samples=n)
    g = np.random.default_rng(0)
    net.set_params(_weights(N, g, 1.4))
    for i in range(n):
        net.add_sample(*_sample(nels, g, i, 0.2 + 0.01 * i if i < 64 else 10.0 * (i - 62)))
    one = [net.eval(i, 1) for i in range(n)]
    # the outputs by other tiles of the same sums: BF16 roundings that fall the other way
    tol = 0.01
    assert abs(net.eval(0, n) - np.mean(one)) < tol * np.mean(one)
    for j in (64, 65):
        for k in range(n):
            if k != j:
                assert abs(one[j] - one[k]) / n > 5 * tol * np.mean(one)
    net.train(steps=1, batch=n, lr=1e-30)
    grad, mean, last = net.get_gradient().astype(np.float64), 0.0, []
    for i in range(n):
        net.train(steps=1, batch=1, lr=1e-30, first=i, count=1)
        last.append(net.get_gradient().astype(np.float64) / n)
        mean = mean + last[-1]
    assert np.linalg.norm(grad - mean) < 0.03 * np.linalg.norm(mean)  # as above
    for j in (64, 65):
        assert np.linalg.norm(last[j] - last[j - 64]) > 0.15 * np.linalg.norm(mean)
