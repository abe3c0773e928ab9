"""Gradients that a leaf keeps without a copy (products, bias sums, attention)
stay its own: a leaf used several times in one graph, a second backward over
the retained graph, and gradients changed in place afterwards."""
import numpy as np
import pytest

from tests.helpers import download, normal, upload

pytestmark = pytest.mark.gpu


def test_kept_gradients_are_not_shared():
    from qutai_amd import Tensor
    from qutai_amd.backends import amd
    from qutai_amd.nn import MultiHeadAttention

    x = Tensor(upload(normal(1, 64), "float32"), shape=(4, 16), requires_grad=True)
    w = Tensor(upload(normal(2, 256), "float32"), shape=(16, 16), requires_grad=True)
    b = Tensor(upload(normal(3, 16), "float32"), shape=(16,), requires_grad=True)
    g = Tensor(upload(normal(4, 64), "float32"), shape=(4, 16))
    y = (x @ w + b) @ w + x + b
    y.backward(g)
    first = [download(t.grad.storage) for t in (x, w, b)]
    xs, ws, bs, gs = (download(t.storage).astype(np.float64).reshape(t.shape) for t in (x, w, b, g))
    h, dh = xs @ ws + bs, gs @ ws.T
    for got, want in zip(first, (dh @ ws.T + gs, h.T @ gs + xs.T @ dh, dh.sum(0) + gs.sum(0))):
        assert np.abs(got.reshape(want.shape) - want).max() <= 1e-4 * np.abs(want).max()
    amd.scale_into(x.grad.storage, 0.0)
    assert download(g.storage).tobytes() == normal(4, 64).tobytes()
    for t in (x, w, b):
        t.grad = None
    y.backward(g)
    for t, want in zip((x, w, b), first):
        assert download(t.grad.storage).tobytes() == want.tobytes()

    layer = MultiHeadAttention(16, 2, causal=True, seed=1)
    z = Tensor(upload(normal(5, 160), "float32"), shape=(1, 10, 16), requires_grad=True)
    layer(z).backward(Tensor(upload(normal(6, 160), "float32"), shape=(1, 10, 16)))
    pointers = [p.grad.storage.ptr for p in (z, *layer.parameters())]
    assert len(set(pointers)) == len(pointers)


def test_checkpoint_of_a_sum_with_a_deferred_gradient():
    """x gets the checkpoint's gradient through the sum and then the Linear's
    deferred product, which reads that same gradient."""
    from qutai_amd import Tensor
    from qutai_amd.lm import activation_checkpoint, layers

    x, weight, w = (Tensor(upload(normal(7 + i, 256), "float32"), shape=(16, 16), requires_grad=True) for i in range(3))
    s = x + layers.linear(x, weight)
    g = Tensor(upload(normal(10, 256), "float32"), shape=(16, 16))
    activation_checkpoint(lambda t: t @ w, s, parameters=(w,)).backward(g)
    xs, weights, ws, gs = (download(t.storage).astype(np.float64).reshape(16, 16) for t in (x, weight, w, g))
    ds = gs @ ws.T
    for got, want in ((x, ds + ds @ weights), (weight, ds.T @ xs), (w, (xs + xs @ weights.T).T @ gs)):
        assert np.abs(download(got.grad.storage).reshape(16, 16) - want).max() <= 1e-4 * np.abs(want).max()
