"""The radiance cache's training step at the batch sizes where its kernels
split the rows differently, against the oracle: each row beside an edge of the
split is counted once, and only once."""
import numpy as np
import pytest

from oracle import nrc_ref as ref
from test_nrc import SHAPES, _batch, _init_weights

# One row's target is far off and every other row's is its own prediction, so
# that the gradient and the loss are that row's alone: a row that is lost or
# taken twice changes both by their whole size.  Every value that enters a
# product is rounded to bf16 (2^-9 relative), some 11 roundings deep in the wide
# network, so two evaluations that round alike up to the order of their sums
# differ by at most 11 x 2^-9 of the gradient's norm; the loss holds the square
# of the error over that of the prediction, two of its roundings after the
# network's five.  (With sums in 64 bits the oracle's own gradients of 300 such
# rows move by 5e-4 at most.)
TOLERANCE = 11 * 2.0 ** -9
FAR_OFF = 1e4  # against other rows' errors of below 1e-3, from the order of the sums


def _problem(n, shape):
    w = _init_weights(20 + n % 1000, shape)
    raw = _batch(n, 30 + n % 1000)
    y, _ = ref.forward(w, raw)
    return w, raw, y


def _one_row(w, raw, y, row):
    """the loss and gradient of a batch of n rows whose other rows have no error"""
    t = y[row] + np.float32(FAR_OFF)
    loss, g = ref.loss_and_grad(w, raw[row:row + 1], t[None], rows=len(raw))
    return t, loss, g


def _edges(n):
    """the first and last row, and both sides of every edge of 16 and 32 rows,
    in large batches of a few of them and of the rows a grid takes at once"""
    step = 16 if n <= 300 else 32
    at = range(0, n, step) if n <= 3000 else [0, 32, 128, 4096, 32768, 65536 - 128, 65536 - 32, 65536, 65568, 65664]
    return sorted({r for e in at for r in (e - 1, e) if 0 <= r < n} | {n - 1})


# one row; below, at and past a chunk of 32 rows, a block of four chunks, the
# fused step's pass of 128 rows, and the chunk count from which dW is split over
# row ranges; a size past that with a ragged last chunk; and just past the
# 65,536 rows that the wide network's kernels take without looping, with one row
# and with a block and one row in the second turn
SIZES = [1, 31, 32, 33, 127, 129, 255, 257, 2081, 65537, 65536 + 4 * 32 + 1]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", SIZES)
def test_every_row_counts_once(shape, n):
    from bulbit_amd.nrc import Nrc

    w, raw, y = _problem(n, shape)
    net = Nrc(seed=3, width=shape[0], layers=shape[1])
    net.set_weights(w)
    for row in _edges(n):
        t = y.copy()
        t[row], lr, gr = _one_row(w, raw, y, row)
        loss, g = net.train(raw, t, apply=False, want_grad=True)
        assert abs(loss - lr) <= TOLERANCE * lr, row
        assert np.linalg.norm(g - gr) <= TOLERANCE * np.linalg.norm(gr), row
    net.close()


# the test's own premise, on the oracle: the rest of the batch adds less than a
# hundredth of the tolerance, and without the row nearly nothing is left
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", [33, 257, 2081])
def test_the_row_is_all_there_is(shape, n):
    w, raw, y = _problem(n, shape)
    row = n - 1
    t = y.copy()
    t[row], loss, g = _one_row(w, raw, y, row)
    jitter = np.random.default_rng(n).uniform(-1e-3, 1e-3, y.shape).astype(np.float32)
    jitter[row] = 0.0
    lb, gb = ref.loss_and_grad(w, raw, t + jitter)
    assert abs(lb - loss) <= 0.01 * TOLERANCE * loss
    assert np.linalg.norm(gb - g) <= 0.01 * TOLERANCE * np.linalg.norm(g)
    lost, gl = ref.loss_and_grad(w, raw[:-1], (t + jitter)[:-1], rows=n)  # the last row dropped
    assert abs(lost - loss) > 0.9 * loss and np.linalg.norm(gl - g) > 0.9 * np.linalg.norm(g)
