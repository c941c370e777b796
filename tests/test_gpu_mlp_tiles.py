"""GPU: the network's products at the edges of their tiles and launch groups against the numpy
oracle (tests/_mlp_oracle.py).

Batches of one row, one row more than a 128-row pad, and enough rows for 64 x 64 tiles on every
layer; widths that leave ragged columns; more layers than one grouped launch of the gradients
and of Adam takes (8).  Same bar as tests/test_gpu_membrane.py: BF16 operands are rounded where
the oracle rounds them and FP32 sums run in another order, 2e-3 in relative Frobenius norm.
"""
import numpy as np
import pytest

from _mlp_oracle import MLPOracle

pytestmark = pytest.mark.gpu
TOL = 2e-3


def rel(a, b):
    return np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b)


@pytest.mark.parametrize("din,width,nh,dout,batch", [
    (867, 512, 4, 1734, 1),
    (867, 512, 4, 1734, 129),
    (130, 512, 1, 577, 2048),   # 64 x 64 tiles (256 of them in the hidden layer), ragged output
    (65, 64, 9, 33, 100),       # ten layers: two grouped launches
])
def test_products_match_oracle(din, width, nh, dout, batch):
    import torch

    from suguru_amd.membrane import SurrogateMLP

    print(f"case: mlp {din}-{width}x{nh}-{dout}, batch {batch}", flush=True)
    rng = np.random.default_rng(din + batch)
    f = lambda *s: rng.normal(size=s).astype(np.float32)
    x, t, mean = f(batch, din), 3.0 * f(batch, dout), 0.1 * f(din)
    scale = rng.uniform(0.5, 2.0, din).astype(np.float32)
    omean, oscale = f(dout), rng.uniform(1.0, 3.0, dout).astype(np.float32)
    wt = rng.uniform(0.5, 1.5, dout).astype(np.float32)
    m = SurrogateMLP(din, width, nh, dout, max_batch=batch)
    m.init(11)
    m.set_norm(mean, scale, omean, oscale)
    layers = [m.get_layer(i) for i in range(m.nl)]
    ref = MLPOracle(layers, mean, scale, oscale, out_mean=omean)
    d = [torch.from_numpy(a).to("cuda:0") for a in (x, t, wt)]
    y = torch.full((batch + 1, dout), 7.0, dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    m.forward(d[0], y, batch=batch)
    torch.cuda.synchronize()
    assert rel(y[:batch].cpu().numpy(), ref.predict(x)) < TOL
    assert bool((y[batch] == 7.0).all())  # nothing past the last real row
    loss = m.grad_only(d[0], d[1], d[2])
    want, g = ref.grads(x, t, wt)
    assert abs(loss - want) < TOL * want
    for i in range(m.nl):
        gW, gb = m.get_grad(i)
        assert rel(gW, g[i][0]) < TOL and rel(gb, g[i][1]) < TOL, i
    # one Adam step from zero moments moves every weight by lr * g / (|g| + eps')
    m.train_step(d[0], d[1], 1e-3, d[2])
    for i in range(m.nl):
        W, b = m.get_layer(i)
        gW, gb = m.get_grad(i)
        for new, old, gr in ((W, layers[i][0], gW), (b, layers[i][1], gb)):
            step = 1e-3 * gr.astype(np.float64) / (np.abs(gr) + 1e-8)
            # (1 - b) and the bias correction cancel to a few FP32 roundings
            assert np.abs((new.astype(np.float64) - old) + step).max() < 1e-6 + 2e-7, i
    m.close()
