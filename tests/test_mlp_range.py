"""Gradients of the selector's network whose sums over the rows leave the range of floats while their means do not."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import selector as sel


@pytest.mark.gpu
@pytest.mark.parametrize("dims,n", [([4, 2], 8192), ([4, 16, 2], 8192), ([3, 16, 16, 5], 4000)])
def test_large_inputs(gpu, dims, n):
    import torch
    rng = np.random.default_rng(11)
    net = sel.MLP(dims, max_batch=n, seed=4)
    x = (rng.uniform(0.5, 1.0, (n, dims[0])) * 1e20).astype(np.float32)
    y = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    t = (y.astype(np.float64) - 5e16).astype(np.float32)  # every error has one sign: the sums are n times their terms
    loss, g = net.gradients(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda(), torch.ones(n, dims[-1], device="cuda"))
    g = g.cpu().numpy()
    d = y.astype(np.float64) - t
    p = net.params().astype(np.float64)
    layers, off = [], 0
    for k, m in zip(dims, dims[1:]):
        layers.append((p[off:off + k * m].reshape(m, k), p[off + k * m:off + k * m + m]))
        off += k * m + m
    acts = [x.astype(np.float64)]
    for w, b in layers[:-1]:
        acts.append(np.maximum(acts[-1] @ w.T + b, 0))
    ref, size = [], []  # the gradients, and the sums of their terms' magnitudes
    dz = 2.0 * d / d.size
    az = np.abs(dz)
    for l in range(len(layers) - 1, -1, -1):
        w = layers[l][0]
        ref[:0] = [(dz.T @ acts[l]).ravel(), dz.sum(0)]
        size[:0] = [(az.T @ np.abs(acts[l])).ravel(), az.sum(0)]
        if l:
            dz, az = (dz @ w) * (acts[l] > 0), (az @ np.abs(w)) * (acts[l] > 0)
    ref, size = np.concatenate(ref), np.concatenate(size)
    assert (size * n * dims[-1] / 2).max() > np.finfo(np.float32).max > 10 * size.max()
    assert np.isfinite(g).all() and np.isfinite(float(loss))
    # n terms added in some order: n units in the last place of their magnitudes
    assert (np.abs(g - ref) <= n * 2.0**-24 * size).all()
    net.close()
