"""GPU: training with and without the loss read back (memb_mlp_train_step's loss may be NULL): the same
weights to the last bit, and the loss whichever call asks for it first.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_loss_is_read_only_where_asked():
    import torch

    from suguru_amd.membrane import SurrogateMLP, _ptr

    print("case: training steps without and with the loss", flush=True)
    rng = np.random.default_rng(5)
    x, t = (torch.from_numpy(rng.standard_normal((70, n)).astype(np.float32)).to("cuda:0") for n in (33, 50))
    nets = [SurrogateMLP(33, 96, 2, 50, 70) for _ in range(2)]
    try:
        for m in nets:
            m.init(9)
        torch.cuda.synchronize()
        a, b = nets
        losses = []
        for _ in range(3):
            a._check(a.lib.memb_mlp_train_step(a.h, 70, _ptr(x), _ptr(t), None, 1e-3, None))
            losses.append(b.train_step(x, t, 1e-3))
        assert a.grad_only(x, t) == b.grad_only(x, t)
        assert all(np.isfinite(losses)) and losses[2] < losses[0]
        for i in range(a.nl):
            for v, w in zip(a.get_layer(i), b.get_layer(i)):
                assert np.array_equal(v, w)
    finally:
        for m in nets:
            m.close()
