"""Device memory that the selector's network takes at creation: activations and gradients of its largest batch, the slices
of weight gradients that this batch uses, and the parameters with their moments."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import selector as sel
from tests import mlp_ref


@pytest.mark.gpu
def test_network_memory(gpu):
    import torch
    dims, rows = [18, 256, 256, 256, 28], 8192
    first = sel.MLP(dims, max_batch=rows, seed=1)  # the library's code is loaded, the runtime's staging memory there
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    net = sel.MLP(dims, max_batch=rows, seed=1)
    taken = before - torch.cuda.mem_get_info()[0]
    # outputs of every layer, gradients of all but the last, 13 slices (512 workgroups over 40 tiles), three arrays of
    # parameters; and 4 MB for the allocator's granules
    need = 4 * (rows * (2 * 3 * 256 + 28) + (13 + 3) * net.num_params)
    assert taken <= need + (4 << 20), (taken, need)
    net.close()
    first.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [[5, 3], [18, 256, 28], [7, 64, 64, 9]])
def test_calls_share_the_last_layers_buffer(gpu, dims):
    """The last layer's outputs and gradients are one buffer: forward passes between gradients change neither."""
    import torch
    n = 333
    rng = np.random.default_rng(3)
    net = sel.MLP(dims, max_batch=n, seed=2)
    x = torch.from_numpy(rng.standard_normal((n, dims[0])).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.standard_normal((n, dims[-1])).astype(np.float32)).cuda()
    m = torch.ones(n, dims[-1], device="cuda")
    y = net.forward(x)
    loss, g = net.gradients(x, t, m)
    assert torch.equal(net.forward(x), y)
    loss2, g2 = net.gradients(x, t, m)
    assert torch.equal(g, g2) and torch.equal(loss, loss2)
    p64 = net.params().astype(np.float64)
    y_ref = mlp_ref.forward(p64, dims, x.cpu().numpy().astype(np.float64))[-1]
    assert np.abs(y.cpu().numpy() - y_ref).max() <= 2e-4 * np.abs(y_ref).max()
    net.close()
