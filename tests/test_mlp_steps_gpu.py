"""A training step's gradient and Adam update on the device at batch sizes
around its tiles (16 rows per block, 64-row padding, slices of the batch of at
least 256 rows, K steps of 128), against the CPU reference.

Tolerance: bf16 operands, whose rounding of an activation (2^-8 relative)
reaches the gradient through two layers: 3e-2 relative (L2, per tensor), as for
the other batch sizes.  A bias or embedding gradient of a single row is a sum
of few such values, hence the floor of 1e-3 of the whole gradient's norm."""
import numpy as np
import pytest

import gz_native as gz
import mlp_oracle

pytestmark = pytest.mark.gpu


def batch_of(n, seed):
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 21, (n, 128)).astype(np.uint8)
    ends = rng.integers(1, 129, n)
    codes[np.arange(128)[None, :] >= ends[:, None]] = 20  # runs of one code
    t = ((codes[:, :32] < 5).sum(axis=1) * 0.25 + rng.normal(0, 0.1, n)).astype(np.float32)
    return codes, t


def check(flat_got, flat_want):
    at, whole = 0, np.linalg.norm(flat_want)
    for name, shape in mlp_oracle.SIZES:
        size = int(np.prod(shape))
        g, w = flat_got[at:at + size], flat_want[at:at + size]
        at += size
        err = np.linalg.norm(g - w)
        assert err <= 3e-2 * np.linalg.norm(w) + 1e-3 * whole, (name, err, np.linalg.norm(w))
    assert at == flat_want.size


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 255, 256, 511, 513, 640, 2049, 4097])
def test_gradient_at_batch_sizes(n):
    print("gradient: batch", n, flush=True)
    codes, t = batch_of(n, 50 + n)
    codes[0, :4] = 21, 30, 200, 255  # past the alphabet: as its last code
    flat = gz.Mlp.init_weights(5)
    mlp = gz.Mlp(flat)
    loss, grad = mlp.train_step(codes, t, 0.0, want_grad=True)
    _, want_loss, want = mlp_oracle.forward_backward(flat, np.minimum(codes, 20), t)
    assert abs(loss - want_loss) <= 2e-2 * want_loss + 1e-4
    check(grad, want)
    assert np.array_equal(mlp.weights(), flat)  # lr = 0
    # the gradient is not carried into the next step (float atomics: in any order)
    _, again = mlp.train_step(codes, t, 0.0, want_grad=True)
    assert np.linalg.norm(again - grad) <= 1e-5 * np.linalg.norm(grad)


@pytest.mark.parametrize("batch,steps", [(1, 3), (60, 5), (300, 4), (2100, 2)])
def test_epochs_are_steps_through_the_order(batch, steps):
    """Whole batches taken through the order, a remainder left out, twice on
    one object: the moments and the step number go on."""
    print("epochs: batch", batch, "steps", steps, flush=True)
    codes, t = batch_of(1500, batch)
    order = np.random.default_rng(batch).integers(0, 1500, batch * steps + batch // 2)
    order = order.astype(np.uint32)
    a, b = gz.Mlp(gz.Mlp.init_weights(2)), gz.Mlp(gz.Mlp.init_weights(2))
    for _ in range(2):
        mean, _ = b.train_epochs(codes, t, order, batch, 1e-3)
        losses = [a.train_step(codes[order[k:k + batch]], t[order[k:k + batch]], 1e-3)
                  for k in range(0, batch * steps, batch)]
        assert abs(mean - np.mean(losses)) <= 1e-3 * max(1.0, np.mean(losses))
    # as in the test of longer runs: Adam turns a near-zero gradient's noise
    # into lr-sized steps of either sign
    wa, wb = a.weights(), b.weights()
    assert np.linalg.norm(wa - wb) <= 1e-3 * np.linalg.norm(wa)
