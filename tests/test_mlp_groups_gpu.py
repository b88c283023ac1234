"""Inference on many rows: a block of mlp_infer_kernel takes several groups of row
tiles in turn, and the next group's input is fetched and placed while one is at work.
A row's outputs do not depend on the others, so they are those of calls on pieces that
give each block one group (test_mlp_gpu.py holds those against the reference)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [64, 128, 256])
@pytest.mark.parametrize("layers", [1, 2, 3])
@pytest.mark.parametrize("n,n_in", [(40_001, 32), (100_003, 12), (262_144, 1)])
def test_rows_do_not_depend_on_their_group(hidden, layers, n, n_in):
    import torch
    from nrg_amd.surrogate import MLP, init_params
    net = MLP(n_in, 10, hidden, layers)
    net.set_params(init_params(n_in, 10, hidden, layers, seed=n))
    g = torch.Generator().manual_seed(n)
    x = torch.randn((n, n_in), generator=g).to("cuda:0")
    y = net.forward(x)
    for a in range(0, n, 8000):
        assert torch.equal(y[a:a + 8000], net.forward(x[a:a + 8000].contiguous())), a
    net.close()
