"""The training kernels at the edges of their launches: networks whose
activations need the default LDS and more (from five hidden layers), one
block of 64 samples and several, and gradient sums over exactly a chunk of
128 blocks and one block more."""
import numpy as np
import pytest

from fjsph_amd import abi, surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n_hidden,batch", [(3, 1, 64), (2, 1, 128), (3, 5, 192), (2, 8, 64), (3, 8, 8256),
                                                (3, 4, 8192), (2, 5, 8256)])
def test_gradients(dim, n_hidden, batch):
    from fjsph_amd.engine import Engine
    from oracle import mlp_oracle as mo
    s = abi.default_settings(dim)
    s.particle_step = 1e-4
    eng = Engine(s)
    rng = np.random.default_rng(7 * dim + n_hidden)
    w, b = surrogate.init_params(dim, n_hidden, seed=dim)
    b = (b + rng.normal(0, 0.2, size=b.size)).astype(np.float32)
    xn = rng.uniform(-1, 1, size=(batch, dim)).astype(np.float32)
    tn = rng.normal(size=(batch, dim + 2)).astype(np.float32)
    print(f"[train blocks] dim={dim} n_hidden={n_hidden} batch={batch}", flush=True)
    dw, db, loss = eng.surrogate_grad(n_hidden, w, b, xn, tn)
    eng.close()
    rw, rb, rloss = mo.forward_backward(w, b, n_hidden, dim, xn.astype(np.float64), tn.astype(np.float64))
    assert abs(loss - rloss) <= 1e-3 * rloss
    # the oracle rounds activations and dZ to BF16 where the kernels do, but
    # from its own sums: a value that rounds the other way is off by 2^-8, in
    # the forward and the backward pass of each layer, of which at most a
    # third add up (2e-2 with four layers)
    tol = 2.0 ** -8 * 2 * max(n_hidden, 4) * 2 / 3
    for a, r in ((dw, rw), (db, rb)):
        assert np.max(np.abs(np.asarray(a, np.float64) - r)) <= tol * np.max(np.abs(r))
