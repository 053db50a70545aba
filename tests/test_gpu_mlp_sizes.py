"""The network kernels at the edges of their tiles: training batches around
the 16-sample blocks and 64-sample gradient chunks (against the float64
reference, with the tolerances of the whole-batch test: FP32 sums of up to 4096
products), and inference batches around the 16-cell tiles and 128-cell blocks
(a cell's outputs do not depend on the batch it is in)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(seed):
    import mlp as M
    from koral_amd.learn import Net
    rng = np.random.default_rng(seed)
    th = (M.init_params(seed) + 0.02 * rng.standard_normal(M.NPARAM)).astype(np.float32)  # biases too
    return M, th, Net(theta=th)


@pytest.mark.parametrize("B", [1, 15, 16, 17, 63, 64, 65, 129, 2051, 4095, 4096])
def test_training_batches(oracle, B):
    import torch
    M, th, net = _net(B)
    rng = np.random.default_rng(B + 1)
    X = rng.normal(size=(B, M.NIN)).astype(np.float32)
    T = rng.normal(size=(B, M.NOUT)).astype(np.float32)
    Xd, Td = torch.from_numpy(X.T.copy()).cuda(), torch.from_numpy(T.T.copy()).cuda()
    Y = net.forward(Xd).cpu().numpy().T
    Yr, _ = M.forward(th.astype(np.float64), X.astype(np.float64))
    assert np.abs(Y - Yr).max() < 1e-5 * np.abs(Yr).max()
    loss, g = net.grad(Xd, Td)
    lr, gr = M.loss_and_grad(th.astype(np.float64), X.astype(np.float64), T.astype(np.float64))
    assert abs(loss - lr) < 1e-5 * lr
    assert (np.abs(g.cpu().numpy() - gr) / (np.abs(gr) + 1e-3 * np.abs(gr).max())).max() < 1e-3
    # a smaller batch after a larger one reads none of its samples
    _, g2 = net.grad(Xd[:, :1].contiguous(), Td[:, :1].contiguous())
    _, gr2 = M.loss_and_grad(th.astype(np.float64), X[:1].astype(np.float64), T[:1].astype(np.float64))
    assert (np.abs(g2.cpu().numpy() - gr2) / (np.abs(gr2) + 1e-3 * np.abs(gr2).max())).max() < 1e-3


def test_inference_batches(oracle):
    import torch
    M, th, net = _net(5)
    F = torch.randn((M.NIN, 70001), device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    Y = net.infer(F)
    for n in (1, 15, 16, 17, 127, 128, 129, 65536, 70001):
        assert torch.equal(net.infer(F[:, :n].contiguous()), Y[:, :n]), n


@pytest.mark.parametrize("B", [1, 130, 1000])
def test_indexed_batches(oracle, B):
    """fit takes its mini-batches through the permutation: the same steps as
    on gathered copies, bit for bit."""
    import torch
    M, th, net = _net(9)
    from koral_amd.learn import Net
    other = Net(theta=th)
    N = 3 * B + B // 2
    g = torch.Generator("cuda").manual_seed(B)
    X = torch.randn((M.NIN, N), device="cuda", generator=g)
    T = torch.randn((M.NOUT, N), device="cuda", generator=g)
    net.fit(X, T, epochs=2, lr=1e-3, batch=B, seed=4)
    gen = torch.Generator("cuda").manual_seed(4)
    for _ in range(2):
        perm = torch.randperm(N, device="cuda", generator=gen)
        for b0 in range(0, N - B + 1, B):
            idx = perm[b0:b0 + B]
            other.step(X[:, idx].contiguous(), T[:, idx].contiguous(), lr=1e-3)
    assert np.array_equal(net.get()[0], other.get()[0])
