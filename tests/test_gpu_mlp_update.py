"""GPU: the training step's fused update (k_mlp_update) writes every
parameter's places in the operand image and reduces any number of
wavefront partials.  After training, the resident image must give the
outputs of a network built from the downloaded parameters, bit for bit
(the image holds the same bfloat16 roundings of the same FP32 values).  The
gradient is held to the oracle as in test_gpu_mlp.py (2e-3 in norm: a
bfloat16 rounding that FP32 and FP64 put on opposite sides of a tie moves an
element by 2^-8), from one sample up to more rounds of 32 than there are
wavefronts (768 on 256 CUs, 24576 samples)."""
import numpy as np
import pytest

import csparks as cs
import mlp_init
import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def _data(seed, n):
    rng = np.random.default_rng(seed)
    return rng.normal(0, 1, (n, cs.MLP_IN)).astype(np.float32), rng.normal(0, 1, n).astype(np.float32)


@pytest.mark.parametrize("n,batch,steps", [(32, 32, 1), (500, 33, 3), (3000, 999, 7), (70000, 40000, 4)])
def test_training_keeps_the_operand_image_in_step(n, batch, steps):
    print(f"case: n={n} batch={batch} steps={steps}", flush=True)
    x, t = _data(n, n)
    net = cs.Mlp(mlp_init.params(3))
    net.set_data(x, t, seed=2)
    before = net.params
    net.train(steps, batch, 2e-3)
    after = net.params
    assert np.count_nonzero(before != after) > 5000
    fresh = cs.Mlp(after)
    np.testing.assert_array_equal(net.forward(x[:777]), fresh.forward(x[:777]))
    net.close()
    fresh.close()


@pytest.mark.parametrize("n", [1, 511, 513, 24576, 24609])
def test_gradient_over_few_and_many_wavefronts(n):
    print(f"case: n={n}", flush=True)
    x, t = _data(7, n)
    p = mlp_init.params(1).astype(np.float32)
    net = cs.Mlp(p)
    g, loss = net.grad(x, t)
    net.close()
    want, lw = mo.grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), bf16_ops=True)
    assert np.linalg.norm(g - want) <= 2e-3 * np.linalg.norm(want)
    assert abs(loss - lw) <= 2e-3 * lw
