"""GPU tests of the fused training step: batches that leave a workgroup half
empty, minibatches drawn by index, and query planes of other strides."""
import ctypes
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
import mlp as M  # noqa: E402

from openshadinglanguage_amd import check, lib  # noqa: E402
from openshadinglanguage_amd import surrogate as S  # noqa: E402
from openshadinglanguage_amd import workloads as W  # noqa: E402

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def data():
    check(lib().oslmi_init())
    q = torch.from_numpy(S.upper_hemisphere_queries(8192, seed=31)).to("cuda:0")
    t = torch.empty((4, 8192), device="cuda:0")
    m = W.layered_material()
    check(lib().oslmi_layered_eval_local(ctypes.byref(m), 8192, S._p(q), S._p(t), None))
    torch.cuda.synchronize()
    return q, t


def _surrogate(seed=7):
    s = S.Surrogate(max_batch=4096)
    s.set_params(S.init_params(seed))
    return s


@pytest.mark.parametrize("B", [64, 128, 192, 2048, 4032])
def test_gradients_of_partly_filled_workgroups(data, B):
    """Against the oracle at its bf16 rounding points: 2e-3 of a layer's
    largest gradient, the bar of the 1024-sample test (single bf16 roundings
    that fall the other way)."""
    q, t = data[0][:, :B].contiguous(), data[1][:, :B].contiguous()
    s = _surrogate()
    print("gradients, batch %d" % B, flush=True)
    g, loss = s.grads(q, t)
    p = M.unpack(S.init_params(7).astype(np.float64))
    x = (q.cpu().numpy() - np.float32(S.IN_OFFSET)[:, None]) * np.float32(S.IN_SCALE)[:, None]
    y = t.cpu().numpy()
    y = np.concatenate([np.log(np.maximum(y[:3], 1e-6)), np.log(np.maximum(y[3:], 1e-12))])
    rl, rg = M.loss_and_grads(p, x.T.astype(np.float64), y.T.astype(np.float64), bf=True)
    assert abs(loss - rl) <= 1e-4 * abs(rl)
    a, b = M.unpack(g.astype(np.float64)), M.unpack(M.pack(rg))
    for name, _ in M.SHAPES:
        assert np.abs(a[name] - b[name]).max() <= 2e-3 * np.abs(b[name]).max(), name


@pytest.mark.parametrize("B", [64, 192, 2048])
def test_indexed_step_equals_gathered_step(data, B):
    """The same minibatch by index (with repeats) and gathered: same bits."""
    q, t = data
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(B)
    a, b = _surrogate(), _surrogate()
    for step in (1, 2, 3):
        idx = torch.randint(0, q.shape[1], (B,), device="cuda:0", generator=gen)
        idx[1] = idx[0]
        qb, tb = q[:, idx].contiguous(), t[:, idx].contiguous()
        check(lib().oslmi_surrogate_train_step(a.h, B, S._p(qb), S._p(tb), 1e-3, 0.9, 0.999, 1e-8,
                                               step, None))
        check(lib().oslmi_surrogate_train_step_indexed(b.h, B, q.shape[1], S._p(q), S._p(t),
                                                       S._p(idx), 1e-3, 0.9, 0.999, 1e-8, step,
                                                       None))
        torch.cuda.synchronize()
    assert np.array_equal(a.get_params(), b.get_params())


def test_train_takes_strided_planes_and_refuses_others(data):
    q, t = data
    a, b = _surrogate(), _surrogate()
    a.train(q[:, :4096].contiguous(), t[:, :4096].contiguous(), 4, batch=256)
    b.train(q[:, :4096], t[:, :4096], 4, batch=256)  # rows 8192 apart
    assert np.array_equal(a.get_params(), b.get_params())
    # the copies that other strides need, on a stream of the caller's; t has
    # more columns than samples
    c = _surrogate()
    c.train(q[:, :4096], t, 4, batch=256, stream=torch.cuda.Stream())
    assert np.array_equal(a.get_params(), c.get_params())
    # planes beyond the 14 and 4 are not read
    d = _surrogate()
    d.train(torch.cat([q, q[:2]])[:, :4096], torch.cat([t, t[:1]]), 4, batch=256)
    assert np.array_equal(a.get_params(), d.get_params())
    for bad in ((q.double(), t), (q, t[:, :100]), (q[:13], t), (q.cpu(), t.cpu())):
        with pytest.raises(ValueError):
            a.train(*bad, 1, batch=256)


def test_activation_derivative_keeps_binary32_accuracy(data):
    """Layer 1 with zero weights: every sample has the biases as its
    pre-activations, and layer 2 weighs all units alike, so the units' bias
    gradients stand in the ratio of their SiLU derivatives (to 0.5, that of a
    unit at zero). Bound, relative: exp 1 ulp (2^-23), the sum, the quotient,
    four operations of the derivative and two inexact adds of 64 equal terms
    2^-24 each, the last factor for the reference unit: 12 * 2^-24. The
    biases are ones whose product with log2(e) rounds badly: an exponential
    of that product is off by 20 * 2^-24 there."""
    B = 64
    z = np.linspace(-30, -22.5, 100000).astype(np.float32)
    prod = (z * np.float32(1.4426950408889634)).astype(np.float64)
    z = z[np.argsort(-np.abs(prod - z.astype(np.float64) * 1.4426950408889634))[:63]]
    z = np.concatenate([[0.0], z]).astype(np.float32)
    p = M.unpack(S.init_params(7).astype(np.float64))
    p["W1"][:] = 0.0
    p["b1"][:] = z
    p["W2"][:] = p["W2"][:, :1]
    q = data[0][:, :B].contiguous()
    t = torch.full((4, B), 50.0, device="cuda:0")  # errors of one sign
    s = _surrogate()
    s.set_params(M.pack(p).astype(np.float32))
    print("bias gradients, batch %d" % B, flush=True)
    g, _ = s.grads(q, t)
    g = M.unpack(g.astype(np.float64))["b1"]
    sg = 1 / (1 + np.exp(-z.astype(np.float64)))
    want = sg * (1 + z.astype(np.float64) * (1 - sg))
    assert g[0] != 0
    assert np.abs(g / g[0] * 0.5 / want - 1).max() <= 12 * 2.0 ** -24
