"""The attention backward's scores against the forward's row statistics. P is rebuilt as e^(s - m) / l from m and l
that the forward formed from its own scores; if the backward formed them any other way, scores of hundreds would
differ by 2^-24 of the sums of magnitudes behind them, and P by as much (1e-5 and more here). Two sums show it: over
the keys, dV of a query whose dO is 1 (P's sum, 1), and dQ of a column in which K is constant and Q is 0 (dS's sum,
0). Every kernel that forms the scores: the key kernels of each head dim, and the query kernel, which head dims 32 and
64 take where the workspace does not hold dQ's partial sums; and each with an element of Q, K, V or dO outside the
split's range, whose blocks are computed again. The bounds are the exponentials' and sums' own roundings,
about 2^-24 for each of a few dozen blocks and steps."""
import numpy as np
import pytest

from staleynet_amd.gemm import Gpu, Shape

pytestmark = pytest.mark.gpu

HEADS, TIME = 8, 384


@pytest.mark.parametrize("tiny", [False, True])
@pytest.mark.parametrize("h,small_workspace", [(32, False), (64, False), (128, False), (32, True), (64, True)])
def test_probabilities_agree_with_the_statistics(gpu, h, small_workspace, tiny):
    print(f"h={h} small_workspace={small_workspace} tiny={tiny}", flush=True)
    rng = np.random.default_rng(h)
    q, k, v, d = (rng.standard_normal((HEADS, TIME, h)).astype(np.float32) for _ in range(4))
    q, k = 16 * q, 16 * k  # scores with a spread of 256
    q[..., 0], k[..., 0] = 0.0, 1.0
    if tiny:  # each in another head
        q[0, 40, 3] = k[1, 70, 5] = v[2, 100, 7] = d[3, 50, 2] = 2.0 ** -120
    ones = np.zeros_like(d)
    ones[:, TIME - 1] = 1.0
    records = HEADS * 3 * TIME * 4
    own = Gpu(0, workspace_bytes=records) if small_workspace else gpu
    n, scale = HEADS * TIME * h, h ** -0.5
    Q, K, V, D, E = (own.upload(Shape.vector(n), x.ravel()) for x in (q, k, v, d, ones))
    O, dQ, dK, dV = (own.zeros(Shape.vector(n)) for _ in range(4))
    stats = own.zeros(Shape.vector(2 * HEADS * TIME))
    own.causal_attention_with_stats(Q, K, V, O, stats, HEADS, TIME, TIME, h, scale, 0)
    own.causal_attention_backward(Q, K, V, O, E, stats, dQ, dK, dV, HEADS, TIME, TIME, h, scale, 0)
    sums = own.download(dV).reshape(HEADS, TIME, h).astype(np.float64).sum(axis=1)
    own.causal_attention_backward(Q, K, V, O, D, stats, dQ, dK, dV, HEADS, TIME, TIME, h, scale, 0)
    column = own.download(dQ).reshape(HEADS, TIME, h)[..., 0].astype(np.float64) / scale
    size = np.abs(np.einsum("nqh,nkh->nqk", d, v)).max()  # of dP, which dS's sum is relative to
    for t in (Q, K, V, D, E, O, dQ, dK, dV, stats):
        t.free()
    print(f"P's sums off by {np.abs(sums - 1).max():.1e}, dS's by {np.abs(column).max() / size:.1e}")
    assert np.abs(sums - 1).max() < 3e-6
    assert np.abs(column).max() / size < 3e-6
