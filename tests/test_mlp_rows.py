"""The selector's network where a workgroup takes whole rows through all layers (widths up to 256), against the float64
reference, at widths and batches around its tiles; and a wider network, which runs layer by layer."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import selector as sel
from tests import mlp_ref

torch = pytest.importorskip("torch")


def cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("dims,n", [([1, 1], 1), ([3, 5, 2], 15), ([18, 16, 28], 16), ([17, 33, 65, 31], 17),
                                    ([64, 64, 64], 64), ([20, 255, 256, 28], 130), ([256, 256, 256], 1007),
                                    ([18, 256, 256, 256, 28], 4096), ([8, 40, 40, 40, 40, 40, 40, 4], 333),
                                    ([18, 257, 28], 100)])
def test_rows_match_numpy(gpu, dims, n):
    """Tolerances as for the layer-by-layer network: outputs within 2e-4 of their largest magnitude, gradients within
    1e-4 of their condition scale (float32 sums of at most a few thousand terms: about 1e-6 of it)."""
    rng = np.random.default_rng(n)
    net = sel.MLP(dims, max_batch=max(n, 8), seed=n)
    p = rng.uniform(-1, 1, net.num_params).astype(np.float32) / np.sqrt(max(dims)).astype(np.float32)
    net.set_params(p)
    x = rng.standard_normal((n, dims[0])).astype(np.float32)
    t = rng.standard_normal((n, dims[-1])).astype(np.float32)
    m = (rng.random((n, dims[-1])) > 0.25).astype(np.float32)
    p64 = p.astype(np.float64)
    y_ref = mlp_ref.forward(p64, dims, x.astype(np.float64))[-1]
    assert np.abs(net.forward(cuda(x)).cpu().numpy() - y_ref).max() <= 2e-4 * np.abs(y_ref).max()
    m[mlp_ref.near_kinks(p64, dims, x)] = 0
    loss, g = net.gradients(cuda(x), cuda(t), cuda(m))
    l_ref, g_ref, g_scale = mlp_ref.loss_and_grads(p64, dims, x, t, m, scale=True)
    assert float(loss.item()) == pytest.approx(l_ref, rel=1e-4, abs=1e-12)
    assert np.all(np.abs(g.cpu().numpy() - g_ref) <= 1e-4 * g_scale + 1e-12)
    # one Adam step from zero moments moves every parameter with a clear gradient by the learning rate against its sign
    net.train_step(cuda(x), cuda(t), cuda(m), 1e-3)
    moved = net.params().astype(np.float64) - p64
    clear = np.abs(g_ref) > 1e-3 * g_scale + 1e-6
    assert np.allclose(moved[clear], -1e-3 * np.sign(g_ref[clear]), rtol=0.05)
    net.close()


@pytest.mark.gpu
@pytest.mark.parametrize("fi,fo", [(28, 28), (40, 20), (20, 40)])
def test_output_over_input(gpu, fi, fo):
    """The outputs written over the inputs are those written elsewhere, whatever the two widths."""
    n = 1000
    net = sel.MLP([fi, 64, fo], max_batch=n, seed=1)
    buf = torch.empty(n * max(fi, fo), device="cuda")
    x = cuda(np.random.default_rng(2).standard_normal((n, fi)))
    want = net.forward(x)
    buf[:n * fi] = x.view(-1)
    stream = torch.cuda.current_stream().cuda_stream
    assert sel._lib.load().bine_mlp_forward(net._h, buf.data_ptr(), n, buf.data_ptr(), stream) == 0
    assert torch.equal(buf[:n * fo].view(n, fo), want)
    net.close()
