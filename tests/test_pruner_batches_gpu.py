"""The pruner's persistent workgroups: batches of fewer samples than
workgroups, and of more (a workgroup then carries several samples, with its
weight gradients in registers over them). A sample's logits do not depend on
its batch; the gradients of a batch are the mean of its halves' (halving is
exact in bfloat16, so only the order of FP32 sums differs)."""
import numpy as np
import pytest

import mav1hip
from test_pruner_gpu import batch

pytestmark = pytest.mark.gpu


def params(net, seed):
    return np.random.default_rng(seed).normal(0, 0.05, net.n).astype(np.float32)


def run(net, x, q, labels):
    net.load(x, q, labels)
    logits, loss = net.forward()
    return logits, loss, net.backward()


@pytest.mark.parametrize("B", [2, 64, 256, 520, 770])
def test_batch_equals_its_halves(gpu, B):
    print(f"[pruner] batch {B}", flush=True)
    rng = np.random.default_rng(B)
    x, q, labels = batch(rng, B)
    net = mav1hip.Pruner(max_batch=B)
    net.set_params(params(net, 1))
    logits, loss, grads = run(net, x, q, labels)
    h = B // 2
    parts = [run(net, x[s], q[s], labels[s]) for s in (slice(0, h), slice(h, B))]
    assert np.array_equal(logits, np.concatenate([p[0] for p in parts]))
    assert abs(loss - 0.5 * (parts[0][1] + parts[1][1])) <= 1e-5 * abs(loss)
    mean = 0.5 * (parts[0][2].astype(np.float64) + parts[1][2])
    # FP32 sums of up to 770 * 1024 terms in another order: random walk of 2^-24 roundings, taken 16-fold
    scale = np.abs(mean).max()
    assert np.abs(grads - mean).max() <= 16 * 2.0**-24 * np.sqrt(B * 1024) * scale


def test_unlabelled_batch_has_zero_gradients(gpu):
    x, q, labels = batch(np.random.default_rng(7), 5)
    net = mav1hip.Pruner(max_batch=8)
    net.set_params(params(net, 2))
    logits, _, grads = run(net, x, q, labels)
    net.load(x, q)
    a = net.forward()[0]
    assert np.array_equal(a, logits)
    assert np.any(grads) and not np.any(net.backward())
    assert np.array_equal(a, net.forward()[0])
    # and a labelled batch after it has its own again
    assert np.array_equal(run(net, x, q, labels)[2], grads)
