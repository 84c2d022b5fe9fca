"""The training kernels at the edges of their tiles: batches of one sample,
around the 16-sample workgroups and the 128-row chunks of the weights'
gradients, and one past the most chunks, against the float64 oracle
(oracle/mlp.py).  Bound: a term of a weight's gradient of up to 8,197 rows goes
through one product, at most 33 steps of four additions in its chunk (132 rows)
and at most 63 additions of chunks, 196 roundings of 6e-8.  Independent ones
leave sqrt(196) * 6e-8 = 8.4e-7 of the sums of magnitudes, which are up to 5
times the gradient's norm here: 4.2e-6; the tolerance leaves ten times that for
the activations' and the loss's own errors."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 15, 17, 127, 129, 131, 8192, 8197])
def test_gradient_matches_oracle(nb, fullchem):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    print("case: gradient of %d samples" % nb, flush=True)
    from gckpp_amd import hip, learned
    from oracle import mlp
    rng = np.random.default_rng(nb)
    net = hip.MLP(nb, *learned.inputs(fullchem))
    p = np.zeros(hip.MLP_NPARAM, np.float32)
    for (o, e), (a, b) in zip(mlp.OFFS, mlp.SHAPES):
        p[o:e] = rng.normal(0, np.sqrt(2.0 / a), a * b)
        p[e:e + b] = rng.normal(0, 0.1, b)
    net.set_params(p)
    X = rng.normal(0, 1, (nb, 48)).astype(np.float32)
    y = rng.normal(0, 1, nb).astype(np.float32)
    k = rng.integers(0, 4, nb).astype(np.int32)
    g, loss = net.grad(*[torch.from_numpy(v).cuda() for v in (X, y, k)], wh=0.7, wc=1.3)
    g, loss = g.cpu().numpy(), float(loss.item())
    L, ref = mlp.loss_grad(p, X, y, k, 0.7, 1.3)
    assert abs(loss - L) <= 4e-5 * abs(L)
    assert np.linalg.norm(g - ref) <= 4e-5 * np.linalg.norm(ref)
    out = net.forward(torch.from_numpy(X).cuda()).cpu().numpy()
    o = mlp.forward(p, X)[2]
    assert np.linalg.norm(out - o) <= 4e-5 * np.linalg.norm(o)
    net.close()
