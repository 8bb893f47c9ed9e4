"""The training step's update at the edges of its row groups, with and without
Adam, and many networks on one context.  The gradient pass leaves a row per
workgroup of 64 samples (at most 512); of the update's eight threads per column
each takes every eighth row, eight at a time: 1, 3, 8, 9, 16, 17, 57, 60, 64,
65, 125 and 512 rows."""
import numpy as np
import pytest

from psb_project_amd import learned
from tests.test_gpu_learned import he_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 17, 64, 144, 512, 513, 1024, 1030, 3648, 3840, 4096,
                                   4097, 8000, 40000])
def test_gradient_and_adam_of_one_step(ctx, oracle, batch):
    rng = np.random.default_rng(batch)
    ns = max(batch, 500)
    feat = rng.normal(size=(8, ns)).astype(np.float32)
    target = rng.normal(size=ns).astype(np.float32)
    idx = rng.choice(ns, batch, replace=False).astype(np.uint32)
    w = he_params(10)
    df, dt, di = ctx.to_device(feat), ctx.to_device(target), ctx.to_device(idx)
    mean, std = np.zeros(8, np.float32), np.ones(8, np.float32)
    m = learned.PressureMLP(ctx)
    m.set_params(w)
    m.set_normalization(mean, std, 1.0)
    loss = m.train_step(df.ptr, dt.ptr, ns, di.ptr, batch, apply_adam=False)
    g = m.grad()
    gref, lref = oracle.mlp_grad(w, mean, std, feat, target, idx, emulate_bf16=True)
    assert loss == pytest.approx(lref, rel=1e-3)
    assert np.linalg.norm(g - gref) / np.linalg.norm(gref) < 1e-2
    # the same gradient through Adam: first step, bias-corrected moments
    m.zero_grad()
    m.train_step(df.ptr, dt.ptr, ns, di.ptr, batch, lr=1e-3)
    f = np.float32
    m1, m2 = (f(1) - f(0.9)) * g, (f(1) - f(0.999)) * g * g
    want = w - f(1e-3) * (m1 / f(1 - 0.9)) / (np.sqrt(m2 / f(1 - 0.999)) + f(1e-8))
    got = m.params()
    assert np.allclose(got, want, rtol=0, atol=2e-7 * (1 + np.abs(w).max()))
    assert not m.grad().any()
    # the fragments hold the new weights: a fresh network given them agrees
    out = [ctx.array(4 * ns) for _ in range(2)]
    m.forward(df.ptr, ns, out[0].ptr)
    k = learned.PressureMLP(ctx)
    k.set_params(got)
    k.set_normalization(mean, std, 1.0)
    k.forward(df.ptr, ns, out[1].ptr)
    ctx.sync()
    a, b = (o.download(np.float32, ns) for o in out)
    assert np.array_equal(a, b)
    m.close()
    k.close()


def test_many_networks_on_one_context(ctx, oracle):
    """More networks than the context has lines for their losses (48), alive
    together, trained in turn, some replaced: every loss is its own."""
    rng = np.random.default_rng(4)
    ns = 700
    feat = rng.normal(size=(8, ns)).astype(np.float32)
    target = rng.normal(size=ns).astype(np.float32)
    df, dt = ctx.to_device(feat), ctx.to_device(target)
    mean, std = np.zeros(8, np.float32), np.ones(8, np.float32)

    def made(seed):
        m = learned.PressureMLP(ctx)
        m.set_params(he_params(seed))
        m.set_normalization(mean, std, 1.0)
        return m

    nets = [(k, made(k)) for k in range(60)]
    for k in (3, 50, 58):
        nets[k][1].close()
        nets[k] = (k + 100, made(k + 100))
    idx = [rng.choice(ns, 64, replace=False).astype(np.uint32) for _ in nets]
    di = [ctx.to_device(i) for i in idx]
    losses = [m.train_step(df.ptr, dt.ptr, ns, d.ptr, 64, apply_adam=False)
              for (_, m), d in zip(nets, di)]
    for (seed, m), i, loss in zip(nets, idx, losses):
        _, ref = oracle.mlp_grad(he_params(seed), mean, std, feat, target, i, emulate_bf16=True)
        assert loss == pytest.approx(ref, rel=1e-3)
        m.close()
