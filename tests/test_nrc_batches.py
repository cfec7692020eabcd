"""The radiance cache's training step at the batch sizes where its kernels
split the rows differently, against the oracle."""
import numpy as np
import pytest

from oracle import nrc_ref as ref
from test_nrc import SHAPES, _batch, _field, _init_weights


# one row; below, at and past a chunk of 32 rows, a block of four chunks, and
# the chunk count from which dW is split over row ranges; a size past that
# with a ragged last chunk.  Every value that enters a product is rounded to
# bf16 (2^-9 relative), some 11 roundings deep in the wide network, so the
# gradients of two evaluations that round alike up to the order of their sums
# differ by at most 11 x 2^-9 = 0.021 of their norm (cosine 0.9998)
@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 129, 255, 257, 2081])
def test_gradient_at_the_chunks_edges(shape, n):
    from bulbit_amd.nrc import Nrc

    net = Nrc(seed=3, width=shape[0], layers=shape[1])
    w = _init_weights(20 + n, shape)
    net.set_weights(w)
    raw = _batch(n, 30 + n)
    t = _field(raw)
    loss, g = net.train(raw, t, apply=False, want_grad=True)
    lr, gr = ref.loss_and_grad(w, raw, t)
    net.close()
    assert abs(loss - lr) <= 2e-2 * lr
    assert g @ gr / np.linalg.norm(g) / np.linalg.norm(gr) > 0.999
    assert abs(np.linalg.norm(g) / np.linalg.norm(gr) - 1) < 0.022
