"""The gradient kernels over batch sizes: fewer bricks than the weight
gradient has splits' worth, a partly filled last block of the loss head, and a
batch larger than the predictor's own (buffers of the call's).  The bound is
that of the oracle comparison elsewhere (dz2 rounded to bfloat16: 2e-2
relative L2), held here by each of the 27 taps on its own."""
import numpy as np
import pytest

from conftest import gpu_available, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


@pytest.mark.parametrize("n,batch", [(1, 1), (2, 4), (5, 2)])
def test_gpu_gradient_of_each_tap_over_batch_sizes(n, batch):
    from oracle import predictor as P
    from channel_flow_amd.solver import Predictor
    print(f"gradient of {n} crops, batch {batch}", flush=True)
    rng = np.random.default_rng(40 + n)
    p = P.init_params(5)
    p["W3"] = rng.standard_normal(P.SHAPES["W3"]) * 0.2
    p = {k: a.astype(np.float32).astype(np.float64) for k, a in p.items()}
    x = rng.standard_normal((n, 16, 16, 16, 16)).astype(np.float32)
    x[..., 15] = 1.0
    x[0, :, :2] = 0.0  # cells outside the domain
    t = rng.standard_normal((n, 14, 14, 14, 5)).astype(np.float32)
    with Predictor(dataset_crops=1, batch_crops=batch) as pr:
        pr.set_params(P.pack(p))
        g, loss = pr.gradient(x, t)
        again, loss2 = pr.gradient(x, t)
    np.testing.assert_array_equal(g, again)
    assert loss == loss2
    y, cache = P.forward(p, x.astype(np.float64), margin=1, bf=True)
    go = P.backward(p, cache, y, t.astype(np.float64))
    assert abs(loss - P.loss(y, t)) <= 1e-5 * P.loss(y, t)
    gg = P.unpack(g)
    for k in P.ORDER:
        if k == "W2":
            a, b = np.reshape(gg[k], (27, -1)), np.reshape(go[k], (27, -1))
            for tap in range(27):
                assert rel_l2(a[tap], b[tap]) <= 2e-2, tap
        else:
            assert rel_l2(gg[k], go[k]) <= 2e-2, k
