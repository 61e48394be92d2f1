"""GPU: the network's backward pass with the activations' gradients formed by the
kernels that produce them, and batches gathered in one launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference_gradient(N, params, nels, x, f, fixed, target):
    """Gradient of the loss by float64 autograd on the CPU, per layer (w, b)."""
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
    t = torch.tensor(N.network_features(nels, x, f, fixed)).permute(0, 4, 1, 2, 3)
    s0 = conv(1, conv(0, t))
    s1 = conv(3, conv(2, pool(s0)))
    s2 = conv(5, conv(4, pool(s1)))
    e3 = conv(7, conv(6, pool(s2)))
    d2 = conv(9, conv(8, torch.cat([up(e3), s2], 1)))
    d1 = conv(11, conv(10, torch.cat([up(d2), s1], 1)))
    d0 = conv(13, conv(12, torch.cat([up(d1), s0], 1)))
    out = conv(14, d0, act=False)[:, :3].permute(0, 2, 3, 4, 1).reshape(-1, 3)
    loss = ((out - torch.tensor(target.reshape(-1, 3))) ** 2).mean()
    loss.backward()
    return loss.item(), [(w.grad.numpy(), b.grad.numpy()) for w, b in zip(W, B)]


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
    _, ref = _reference_gradient(N, p, nels, x, f, net.fixed, u / np.sqrt(np.mean(u**2)))
    off = 0
    for li, (w, b) in enumerate(ref):
        for name, r in (("w", w), ("b", b)):
            d = step[off:off + r.size]
            off += r.size
            big = np.abs(r.ravel()) > 0.75 * np.sqrt(np.mean(r**2))
            assert np.array_equal(np.sign(d[big]), -np.sign(r.ravel()[big])), (li, name)
    assert off == p.size


def test_batches_gathered(T, gpu):
    """A batch of more samples than one launch gathers (64): the loss of all is the
    mean of the samples' own."""
    import topopt_jl_amd.nn as NN
    nels, n = (8, 8, 8), 70
    net = NN.WarmStartNet(nels, max_batch=n, max_samples=n, seed=2)
    g = np.random.default_rng(0)
    for i in range(n):
        net.add_sample(g.uniform(0.05, 1.0, net.ncells), NN.cantilever_load(nels, i % 9, 4),
                       g.standard_normal(net.nnodes * 3))
    one = [net.eval(i, 1) for i in range(n)]
    # FP32 outputs by other tiles of the same sums
    assert abs(net.eval(0, n) - np.mean(one)) < 1e-3 * np.mean(one)
    assert len(set(one)) == n
