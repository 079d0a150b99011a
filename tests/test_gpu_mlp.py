"""The warm-start network's MFMA kernels against its CPU oracle.

oracle/mlp_oracle.py rounds to BF16 at the same points as the GPU and is
exact FP64 elsewhere, so the GPU differs from it only by FP32 accumulation
order, its exp and reciprocal, and the rare BF16 rounding flips these cause.  Stated bounds:
outputs within 2e-3 normwise relative, loss within 1e-4 relative, every
layer's weight and bias gradient within 5e-3 normwise relative.  A short
training run must cut the loss on a smooth regression target tenfold.
"""
import numpy as np
import pytest

from oracle.mlp_oracle import KIN, KOUT, NIN, NOUT, MlpOracle
from tests.test_mlp_oracle import random_params

pytestmark = pytest.mark.gpu


def net(params=None):
    from oneflow_amd.mlp import Mlp
    m = Mlp(seed=3)
    if params is not None:
        m.set_params(params.astype(np.float32))
    return m


def test_forward_matches_oracle():
    rng = np.random.default_rng(1)
    p = random_params(rng, scale=1.0).astype(np.float32)
    x = rng.normal(0, 1, (1000, NIN)).astype(np.float32)  # not a multiple of 64: padded rows
    m = net(p)
    y = m.forward(x)
    yo = MlpOracle(p, bf16=True).forward(x)
    e = float(np.linalg.norm(y - yo) / np.linalg.norm(yo))
    print(f"\n[mlp] forward rel err {e:.3e}", flush=True)
    assert e <= 2e-3, e


@pytest.mark.parametrize("n", [1050, 70_000, 70_050])
def test_one_kernel_forward_equals_layered(n):
    """The one-kernel forward pass (activations in LDS) against one GEMM
    kernel per layer: the same bits.  1050 and 70,050 samples leave the last
    128-sample workgroup half filled; 70,000 takes the layered pass's large
    tiles."""
    rng = np.random.default_rng(7)
    p = random_params(rng, scale=1.0).astype(np.float32)
    x = rng.normal(0, 1, (n, NIN)).astype(np.float32)
    m = net(p)
    m.set_forward_variant(0)
    y0 = m.forward(x)
    m.set_forward_variant(1)
    y1 = m.forward(x)
    print(f"\n[mlp] one-kernel forward, n={n}: max |diff| {float(np.max(np.abs(y1 - y0))):.3e}", flush=True)
    assert np.array_equal(y0, y1)


def test_gradients_match_oracle():
    rng = np.random.default_rng(2)
    p = random_params(rng, scale=1.0).astype(np.float32)
    x = rng.normal(0, 1, (777, NIN)).astype(np.float32)
    t = rng.normal(0, 1, (777, NOUT)).astype(np.float32)
    m = net(p)
    loss, g = m.gradients(x, t)
    lo, go = MlpOracle(p, bf16=True).gradients(x, t)
    assert abs(loss - lo) <= 1e-4 * abs(lo), (loss, lo)
    o = 0
    worst = 0.0
    for l, (i, k) in enumerate(zip(KIN, KOUT)):
        for name, cnt in (("W", i * k), ("b", k)):
            a, b = g[o:o + cnt], go[o:o + cnt]
            e = float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))
            worst = max(worst, e)
            assert e <= 5e-3, (l, name, e)
            o += cnt
    print(f"\n[mlp] loss {loss:.6e} vs {lo:.6e}; worst gradient block rel err {worst:.3e}", flush=True)


def test_training_reduces_loss():
    rng = np.random.default_rng(3)
    x = rng.uniform(-1, 1, (20000, NIN)).astype(np.float32)
    t = np.stack([np.sin(2 * x[:, 0]) * x[:, 1], np.cos(x[:, 2] + x[:, 3]), x[:, 4] ** 2 - x[:, 5],
                  np.tanh(3 * x[:, 6]), x[:, 7] * x[:, 8]], axis=1).astype(np.float32)
    m = net()
    losses = m.train(x, t, batch=4096, steps=400, lr=2e-3)
    first, last = float(losses[:5].mean()), float(losses[-20:].mean())
    print(f"\n[mlp] training loss {first:.4e} -> {last:.4e}", flush=True)
    assert np.all(np.isfinite(losses)) and last < 0.1 * first, (first, last)


@pytest.mark.parametrize("n", [1, 15, 17, 4095, 4096, 4097, 8192, 8193, 8255])
def test_one_kernel_forward_shapes(n):
    """Every workgroup shape of the one-kernel forward at its edges, against
    the layered pass: the same bits, an infinite and a NaN input included."""
    rng = np.random.default_rng(n)
    x = rng.normal(0, 1, (n, NIN)).astype(np.float32)
    x[0, 3], x[n // 2, 8] = np.inf, np.nan
    m = net(random_params(rng, scale=1.0).astype(np.float32))
    m.set_forward_variant(0)
    y0 = m.forward(x)
    m.set_forward_variant(1)
    y1 = m.forward(x)
    assert np.array_equal(y0, y1, equal_nan=True)


@pytest.mark.parametrize("n", [1, 63, 65, 1050, 2048, 4096, 4097, 131072])
def test_gradient_shapes(n):
    """Both workgroup shapes of the gradient kernel, one and several splits of
    the weight products (one layer at a time from 65 splits), and a ragged last
    64 samples, against the oracle.  Tolerance: all elements of a block one
    bf16 step (2^-8 = 4e-3) apart."""
    rng = np.random.default_rng(n)
    p = random_params(rng, scale=1.0).astype(np.float32)
    x = rng.normal(0, 1, (n, NIN)).astype(np.float32)
    t = rng.normal(0, 1, (n, NOUT)).astype(np.float32)
    loss, g = net(p).gradients(x, t)
    lo, go = MlpOracle(p, bf16=True).gradients(x, t)
    assert abs(loss - lo) <= 1e-4 * abs(lo), (loss, lo)
    o = 0
    for l, (i, k) in enumerate(zip(KIN, KOUT)):
        for name, cnt in (("W", i * k), ("b", k)):
            a, b = g[o:o + cnt], go[o:o + cnt]
            e = float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))
            assert e <= 5e-3, (l, name, e)
            o += cnt


@pytest.mark.parametrize("n,batch", [(70, 64), (5000, 4096), (9000, 8192)])
def test_training_keeps_weight_copies(n, batch):
    """After training, every copy of the weights (fp32, bf16, both operand
    orders, transposed) holds the same network: the two forward forms and the
    gradients equal those of a net given the trained parameters, bit for bit."""
    rng = np.random.default_rng(n)
    x = rng.normal(0, 1, (n, NIN)).astype(np.float32)
    t = rng.normal(0, 1, (n, NOUT)).astype(np.float32)
    m = net()
    m.train(x, t, batch=batch, steps=3, lr=1e-3)
    ref = net(m.params())
    for v in (0, 1):
        m.set_forward_variant(v)
        ref.set_forward_variant(v)
        assert np.array_equal(m.forward(x), ref.forward(x))
    (l0, g0), (l1, g1) = m.gradients(x, t), ref.gradients(x, t)
    assert l0 == l1 and np.array_equal(g0, g1)


@pytest.mark.parametrize("n", [262143, 262144, 262145, 393217, 1048576, 1048577])
def test_piped_forward(n):
    """Many host samples pass through in pieces (copies beside the computing):
    the same bits as calls of fewer samples, twice in a row with other inputs."""
    rng = np.random.default_rng(n)
    m = net(random_params(rng, scale=1.0).astype(np.float32))
    for _ in range(2):
        x = rng.normal(0, 1, (n, NIN)).astype(np.float32)
        y = m.forward(x)
        parts = np.concatenate([m.forward(x[i:i + 100000]) for i in range(0, n, 100000)])
        assert y.shape == (n, parts.shape[1]) and np.array_equal(y, parts)
