"""Weight gradients at the edges of the reduction's stages of 32 rows and chunks
of 256: rings of n nodes (2 n edges) against the oracle network with BF16
operands.  An operand rounded the other way is off by 2^-8 at most, so the norms
agree within 2^-6."""
import numpy as np
import pytest

from oracle import mpnn_ref
from spherocyls_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 16, 31, 33, 128, 129, 520])
def test_gradients_of_rings(n):
    rng = np.random.default_rng(n)
    near = [sorted({(i - 1) % n, (i + 1) % n}) for i in range(n)]
    g = native.Graph(rng.normal(0, 1, (n, 4)), np.cumsum([0] + [len(s) for s in near]),
                     np.concatenate(near), rng.normal(0, 1, (sum(map(len, near)), 5)))
    p = rng.normal(0, 0.08, mpnn_ref.num_params())
    lay, _ = mpnn_ref.layout()
    o, K, N = lay["wo"]
    p[o:o + K * N].reshape(K, N)[:, 3:] = 0.0
    p = p.astype(np.float32)
    target = rng.normal(0, 1, (n, 3)).astype(np.float32)
    print("ring", n, flush=True)
    m = native.Mpnn(seed=1)
    try:
        m.set_params(p)
        m.load_graph(g)
        m.forward()
        m.backward(target)
        got = m.grads()
    finally:
        m.close()
    _, want = mpnn_ref.loss_and_grad(p.astype(np.float64), g.node_feat, g.offsets, g.src,
                                     g.edge_feat, target, bf16=True)
    for name, (o, K, N) in lay.items():
        a, b = got[o:o + K * N], want[o:o + K * N]
        assert np.linalg.norm(a - b) <= 2.0 ** -6 * np.linalg.norm(b), name
