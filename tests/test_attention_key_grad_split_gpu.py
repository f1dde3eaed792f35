"""The split key kernel of the attention backward (attention_key_grad_split.h) where it can go wrong: short
sequences, ragged stages (32 queries) and key blocks (128), the flush of its accumulators (every 2048 queries),
offsets; and operands outside the split's range or gradients too large for its scaled sums, whose blocks it
computes again with the fp32 instruction. Against the oracle's restatement of the reference's backward
(crates/staleynet-model/src/layers/attention.rs:220-260) at the reference's fp32 tolerance."""
import numpy as np
import pytest

from oracle import oracle
from staleynet_amd.gemm import Shape
from test_attention_backward_gpu import TOLERANCE, reference, run

pytestmark = pytest.mark.gpu

CASES = [
    (2, 127, 127, 64, 0), (2, 128, 129, 64, 1), (1, 161, 255, 64, 94), (1, 511, 511, 32, 0), (3, 512, 513, 32, 0),
    (1, 545, 130, 32, 0), (1, 512, 512, 64, 0), (1, 513, 385, 64, 0), (1, 544, 640, 64, 96), (1, 1061, 1061, 64, 0),
    (1, 1057, 700, 32, 3), (1, 2100, 130, 32, 0),
]


@pytest.mark.parametrize("heads,queries,keys,h,offset", CASES)
def test_edges_match_the_reference_calls(gpu, heads, queries, keys, h, offset):
    print(f"heads={heads} queries={queries} keys={keys} h={h} offset={offset}", flush=True)
    scale = h ** -0.5
    inputs, got = run(gpu, heads, queries, keys, h, scale, offset, seed=queries * keys + h)
    _, _, dq, dk, dv = reference(*inputs, heads, queries, keys, h, scale, offset)
    for name, expected in (("dq", dq), ("dk", dk), ("dv", dv)):
        assert np.all(np.isfinite(got[name])), name
        assert oracle.relative_error(expected, got[name]) < TOLERANCE, name


def exact(q, k, v, d_out, heads, queries, keys, h, scale, offset):
    q, k, v, d_out = (x.reshape(heads, -1, h).astype(np.float64) for x in (q, k, v, d_out))
    scale = np.float64(np.float32(scale))
    visible = np.arange(keys)[None, :] <= np.arange(queries)[:, None] + offset
    s = np.where(visible, scale * (q @ k.transpose(0, 2, 1)), -np.inf)
    p = np.exp(s - s.max(axis=2, keepdims=True))
    p /= p.sum(axis=2, keepdims=True)
    ds = p * (d_out @ v.transpose(0, 2, 1) - np.sum(d_out * (p @ v), axis=2, keepdims=True))
    return scale * (ds @ k), scale * (ds.transpose(0, 2, 1) @ q), p.transpose(0, 2, 1) @ d_out


def backward(gpu, q, k, v, d_out, heads, queries, keys, h, scale, offset=0):
    print(f"heads={heads} queries={queries} keys={keys} h={h} offset={offset}", flush=True)
    Q, K, V, dO = (gpu.upload(Shape.vector(x.size), x) for x in (q, k, v, d_out))
    O, dQ = (gpu.zeros(Shape.vector(heads * queries * h)) for _ in range(2))
    dK, dV = (gpu.zeros(Shape.vector(heads * keys * h)) for _ in range(2))
    stats = gpu.zeros(Shape.vector(2 * heads * queries))
    gpu.causal_attention_with_stats(Q, K, V, O, stats, heads, queries, keys, h, scale, offset)
    gpu.causal_attention_backward(Q, K, V, O, dO, stats, dQ, dK, dV, heads, queries, keys, h, scale, offset)
    got = [gpu.download(t) for t in (dQ, dK, dV)]
    for t in (Q, K, V, dO, O, stats, dQ, dK, dV):
        t.free()
    return got


@pytest.mark.parametrize("h", [32, 64])
def test_gradients_below_the_split_range(gpu, h):
    # dO of magnitude 2^-112: its lowest bits pass the smallest bf16. A power of two scales the reference exactly
    # (but for values that fall under the smallest normal number, 2^-14 of the largest here).
    heads, queries, scale = 2, 600, h ** -0.5
    rng = np.random.default_rng(h)
    q, k, v, d_out = (rng.normal(0, 1, heads * queries * h).astype(np.float32) for _ in range(4))
    _, _, *expected = reference(q, k, v, d_out, heads, queries, queries, h, scale, 0)
    got = backward(gpu, q, k, v, np.ldexp(d_out, -112).astype(np.float32), heads, queries, queries, h, scale)
    for name, e, g in zip(("dq", "dk", "dv"), expected, got):
        error = np.linalg.norm(np.ldexp(g.astype(np.float64), 112) - e) / np.linalg.norm(e.astype(np.float64))
        assert error < TOLERANCE, f"{name}: {error}"


@pytest.mark.parametrize("h", [32, 64])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_a_bad_query_reaches_what_it_sees_and_no_more(gpu, h, value):
    # One dO value of head 1 is not finite: neither are dQ of its query, and dV's column (dK whole) for every key
    # that query sees. Later key blocks, other queries and head 0 hold what they hold without that query.
    heads, queries, bad, scale = 2, 640, 200, h ** -0.5
    rng = np.random.default_rng(h + 1)
    q, k, v, d_out = (rng.normal(0, 1, heads * queries * h).astype(np.float32) for _ in range(4))
    without = d_out.reshape(heads, queries, h).copy()
    without[1, bad] = 0.0
    _, _, *expected = reference(q, k, v, without.ravel(), heads, queries, queries, h, scale, 0)
    d_out.reshape(heads, queries, h)[1, bad, 3] = value
    got = backward(gpu, q, k, v, d_out, heads, queries, queries, h, scale)
    dq, dk, dv = (x.reshape(heads, queries, h) for x in got)
    eq, ek, ev = (x.reshape(heads, queries, h) for x in expected)
    assert not np.any(np.isfinite(dq[1, bad])) and not np.any(np.isfinite(dk[1, :bad + 1]))
    assert not np.any(np.isfinite(dv[1, :bad + 1, 3]))
    block = (bad // 128 + 1) * 128  # the first key block that starts past the query
    others = np.arange(queries) != bad
    for name, e, g in (("dq", eq[1, others], dq[1, others]), ("dk", ek[1, block:], dk[1, block:]),
                       ("dv", ev[1, block:], dv[1, block:]), ("dq", eq[0], dq[0]), ("dk", ek[0], dk[0]),
                       ("dv", ev[0], dv[0])):
        assert np.all(np.isfinite(g)), name
        assert oracle.relative_error(e.ravel(), g.ravel()) < TOLERANCE, name


@pytest.mark.parametrize("h", [32, 64])
@pytest.mark.parametrize("heads,queries,keys,offset", [(2, 300, 300, 0), (1, 131, 257, 126), (1, 2100, 130, 0)])
@pytest.mark.parametrize("powers", [dict(q=-122, k=122), dict(q=122, k=-122), dict(v=-124), dict(d=-124),
                                    dict(v=-60, d=-62), dict(d=70), dict(v=65, d=-10)],
                         ids=lambda p: " ".join(f"{n} 2^{e}" for n, e in p.items()))
def test_operands_outside_the_range(gpu, h, heads, queries, keys, offset, powers):
    # Scores stay of ordinary size; the gradients are scaled by powers of two, so their norms are taken in float64.
    scale = h ** -0.5
    rng = np.random.default_rng(h + queries)
    sizes = dict(q=queries, k=keys, v=keys, d=queries)
    q, k, v, d = (np.ldexp(rng.standard_normal(heads * n * h).astype(np.float32), powers.get(name, 0))
                  for name, n in sizes.items())
    expected = exact(q, k, v, d, heads, queries, keys, h, scale, offset)
    got = backward(gpu, q, k, v, d, heads, queries, keys, h, scale, offset)
    for name, e, g in zip(("dq", "dk", "dv"), expected, got):
        assert np.all(np.isfinite(g)), name
        assert np.linalg.norm(g.astype(np.float64) - e.ravel()) / np.linalg.norm(e) < TOLERANCE, name


@pytest.mark.parametrize("h", [32, 64])
def test_peaked_scores_and_small_gradients(gpu, h):
    # Scores with gaps of 60 and more and dO of 2^-80: P dO of keys that hardly any query weighs is near the smallest
    # normal fp32. Each key's dV (sums without cancellation) relative to its own size, down to 2^-100; the weights'
    # own error is |s - m| 2^-24 and a few roundings, under 1e-5 for the gaps that matter there (100 2^-24).
    heads, queries, scale = 2, 400, h ** -0.5
    rng = np.random.default_rng(h + 9)
    q, k, v, d = (rng.standard_normal((heads, queries, h)).astype(np.float32) for _ in range(4))
    q, k, d = 3 * q, 3 * k, np.ldexp(np.abs(d), -80)
    *_, expected = exact(q, k, v, d, heads, queries, queries, h, scale, 0)
    *_, got = backward(gpu, *(x.ravel() for x in (q, k, v, d)), heads, queries, queries, h, scale)
    rows = np.linalg.norm(expected, axis=2)
    error = np.linalg.norm(got.reshape(expected.shape).astype(np.float64) - expected, axis=2)
    assert np.min(rows) < 2.0 ** -80 and np.max((error / rows)[rows > 2.0 ** -100]) < TOLERANCE
