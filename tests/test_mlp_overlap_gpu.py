"""Network calls whose outputs lie over their inputs (include/nrg_mlp.h takes any
device pointers): the results of separate buffers, the forward's bit for bit, the
gradient's to the order of its row sums (1e-4, as in test_mlp_gpu.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMS = (13, 128, 3, 10)


def _net_and_batch(n):
    import torch
    from nrg_amd.surrogate import MLP, init_params
    net = MLP(DIMS[0], DIMS[3], DIMS[1], DIMS[2])
    net.set_params(init_params(DIMS[0], DIMS[3], DIMS[1], DIMS[2], seed=n))
    g = torch.Generator().manual_seed(n)
    x = torch.randn((n, DIMS[0]), generator=g).to("cuda:0")
    t = torch.randn((n, DIMS[3]), generator=g).to("cuda:0")
    return net, x, t


@pytest.mark.parametrize("n", [33, 70001])
@pytest.mark.parametrize("shift", [0, 3 * 13, -3 * 13])
def test_forward_over_its_input(n, shift):
    import torch
    from nrg_amd.capi import check
    net, x, _ = _net_and_batch(n)
    want = net.forward(x)
    buf = torch.zeros(n * DIMS[0] + 2 * abs(shift), device="cuda:0")
    xs = buf[abs(shift):abs(shift) + n * DIMS[0]]
    xs.copy_(x.reshape(-1))
    y = buf[abs(shift) + shift:abs(shift) + shift + n * DIMS[3]]
    torch.cuda.synchronize()
    check(net.lib, net.lib.nrg_mlp_forward_dev(net.h, n, xs.data_ptr(), y.data_ptr()))
    assert torch.equal(y.reshape(n, DIMS[3]), want)
    net.close()


@pytest.mark.parametrize("n", [33, 70001])
@pytest.mark.parametrize("over", ["y_out over x", "y_out over t", "grad over x", "grad over t"])
def test_gradient_over_its_inputs(n, over):
    import torch
    from nrg_amd.capi import check
    net, x, t = _net_and_batch(n)
    g_ref, loss_ref, y_ref = net.grad(x, t)
    size = max(net.num_params, n * DIMS[0])
    bx, bt = torch.zeros(size, device="cuda:0"), torch.zeros(size, device="cuda:0")
    bx[:x.numel()].copy_(x.reshape(-1))
    bt[:t.numel()].copy_(t.reshape(-1))
    inp = bx if over.endswith("x") else bt
    grad = inp if over.startswith("grad") else torch.zeros(size, device="cuda:0")
    y = inp if over.startswith("y_out") else torch.zeros(size, device="cuda:0")
    loss = torch.zeros(1, device="cuda:0")
    torch.cuda.synchronize()
    check(net.lib, net.lib.nrg_mlp_grad_dev(net.h, n, bx.data_ptr(), bt.data_ptr(), None, grad.data_ptr(),
                                            loss.data_ptr(), y.data_ptr()))
    rel = lambda a, b: float(torch.linalg.norm((a - b).double()) / torch.linalg.norm(b.double()))  # noqa: E731
    assert torch.equal(y[:n * DIMS[3]].reshape(n, DIMS[3]), y_ref)
    assert rel(grad[:net.num_params], g_ref) <= 1e-4 and rel(loss, loss_ref) <= 1e-6
    net.close()
