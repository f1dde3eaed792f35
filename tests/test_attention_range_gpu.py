"""The fused attention forward (attention_forward.hip) where its operands leave the range of the split into three
bf16 parts, so that waves compute their queries again with the fp32 instruction: Q, K or V under 2^-110 (with
partners that bring the scores back to ordinary size), subnormal V, infinities and NaN, scores that overflow. Each
with and without the probabilities and with the keys split over workgroups (one head of queries against a cache),
at every head dim, against float64 at the reference's fp32 tolerance. And the merge of split keys at the edges of
its ranges: a ragged last range, ranges past some queries' horizon, queries over several blocks."""
import numpy as np
import pytest

from oracle import oracle
from staleynet_amd.gemm import Shape

pytestmark = pytest.mark.gpu

TOLERANCE = 1e-5  # kernels_match_reference.rs:12
# heads, queries, keys, offset, probabilities: whole sequences, then queries against a cache (split keys without
# probabilities: three ranges, the last one ragged)
FORMS = [(2, 200, 200, 0, False), (2, 200, 200, 0, True), (1, 100, 540, 400, False), (1, 100, 540, 400, True)]


def exact(q, k, v, heads, queries, keys, h, scale, offset):
    q, k, v = (x.reshape(heads, -1, h).astype(np.float64) for x in (q, k, v))
    s = q @ k.transpose(0, 2, 1) * np.float64(np.float32(scale))
    visible = np.arange(keys)[None, :] <= np.arange(queries)[:, None] + offset
    s = np.where(visible, s, -np.inf)
    p = np.exp(s - s.max(axis=2, keepdims=True))
    p /= p.sum(axis=2, keepdims=True)
    return p @ v, p


def run(gpu, q, k, v, heads, queries, keys, h, scale, offset, with_p):
    print(f"heads={heads} queries={queries} keys={keys} h={h} offset={offset} probabilities={with_p}", flush=True)
    tensors = [gpu.upload(Shape.vector(x.size), x.ravel()) for x in (q, k, v)]
    out = gpu.upload(Shape.vector(heads * queries * h), np.full(heads * queries * h, 7.0, np.float32))
    p = gpu.zeros(Shape.vector(heads * queries * keys)) if with_p else None
    gpu.causal_attention(*tensors, out, heads, queries, keys, h, scale, offset, probabilities=p)
    got = gpu.download(out).reshape(heads, queries, h)
    got_p = gpu.download(p).reshape(heads, queries, keys) if with_p else None
    for t in tensors + [out] + ([p] if with_p else []):
        t.free()
    return got, got_p


def inputs(heads, queries, keys, h, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((heads, n, h)).astype(np.float32) for n in (queries, keys, keys))


def close(expected, got):
    assert np.all(np.isfinite(got))
    assert oracle.relative_error(expected.ravel(), got.ravel()) < TOLERANCE


@pytest.mark.parametrize("h", [32, 64, 128])
@pytest.mark.parametrize("heads,queries,keys,offset,with_p", FORMS)
@pytest.mark.parametrize("down", ["q", "k", "v"])
def test_tiny_operands(gpu, h, heads, queries, keys, offset, with_p, down):
    q, k, v = inputs(heads, queries, keys, h, h + keys)
    if down == "v":
        v = np.ldexp(v, -124)
    else:  # 2^-125 against 2^125
        q, k = (np.ldexp(x, -125 if down == name else 125) for x, name in ((q, "q"), (k, "k")))
    scale = h ** -0.5
    eo, ep = exact(q, k, v, heads, queries, keys, h, scale, offset)
    go, gp = run(gpu, q, k, v, heads, queries, keys, h, scale, offset, with_p)
    # Scaled by a power of two, so that the norms do not underflow.
    close(eo * (2.0 ** 124 if down == "v" else 1), go.astype(np.float64) * (2.0 ** 124 if down == "v" else 1))
    if with_p:
        close(ep, gp)


@pytest.mark.parametrize("h", [32, 64, 128])
@pytest.mark.parametrize("heads,queries,keys,offset,with_p", FORMS)
def test_subnormal_values(gpu, h, heads, queries, keys, offset, with_p):
    # V of 2^-136: under the smallest bf16 part. A sum of `keys` products and a quotient, each rounded at 2^-149.
    q, k, v = inputs(heads, queries, keys, h, h + keys + 1)
    v = np.ldexp(v, -136)
    eo, _ = exact(q, k, v, heads, queries, keys, h, h ** -0.5, offset)
    go, _ = run(gpu, q, k, v, heads, queries, keys, h, h ** -0.5, offset, with_p)
    assert np.max(np.abs(go - eo)) <= (keys + 8) * 2.0 ** -149


@pytest.mark.parametrize("h", [32, 64, 128])
@pytest.mark.parametrize("heads,queries,keys,offset,with_p", FORMS)
@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("where", ["q", "k", "v"])
def test_values_that_are_not_finite(gpu, h, heads, queries, keys, offset, with_p, value, where):
    # One value of the last head: its query, or the queries that see its key, and no others.
    q, k, v = inputs(heads, queries, keys, h, h + keys + 2)
    eo, ep = exact(q, k, v, heads, queries, keys, h, h ** -0.5, offset)
    row = queries // 2 if where == "q" else queries // 2 + offset
    {"q": q, "k": k, "v": v}[where][-1, row, 3] = value
    go, gp = run(gpu, q, k, v, heads, queries, keys, h, h ** -0.5, offset, with_p)
    if where == "q":
        bad = np.arange(queries) == row
        clear = ~bad
    else:
        bad = np.arange(queries) + offset >= row
        clear = np.arange(queries) + offset < row
        if where == "v":  # times the weight 0 it is NaN too, in a block of 32 keys that a wave's 32 queries reach
            clear = np.arange(queries) // 32 * 32 + 31 + offset < row // 32 * 32
    if where == "v":
        assert not np.any(np.isfinite(go[-1, bad, 3]))
    elif value is np.nan or where == "q":
        assert not np.any(np.isfinite(go[-1, bad]))
    close(eo[-1, clear], go[-1, clear])
    close(eo[:-1], go[:-1]) if heads > 1 else None
    if with_p:
        close(ep[-1, clear], gp[-1, clear])


@pytest.mark.parametrize("heads,queries,keys,offset,with_p", FORMS)
def test_scores_beyond_the_largest_float(gpu, heads, queries, keys, offset, with_p):
    # Every score is -(2^64 - 2^54)^2, finite, where the first parts are 2^64 and their product is past the largest
    # float. All the same: the weights are equal.
    h = 64
    q, k, v = inputs(heads, queries, keys, h, 5)
    q[:], k[:] = 0.0, 0.0
    x = np.float32(2.0 ** 64 - 2.0 ** 54)
    q[..., 0], k[..., 0] = x, -x
    assert np.isfinite(np.float32(x) * np.float32(-x))
    eo, _ = exact(q, k, v, heads, queries, keys, h, 2.0 ** -100, offset)
    go, _ = run(gpu, q, k, v, heads, queries, keys, h, 2.0 ** -100, offset, with_p)
    close(eo, go)


@pytest.mark.parametrize("h", [32, 64, 128])
@pytest.mark.parametrize("heads,queries,keys,offset", [
    (1, 5, 2000, 1990),     # a range's last key past the cache's end for some queries
    (1, 300, 1000, 40),     # ranges the first queries do not see
    (2, 129, 1408, 1),      # two query blocks, keys far past every horizon
    (1, 128, 256, 128),     # two ranges of exactly 128 keys
    (3, 260, 900, 619),     # a last range of a few keys
    (12, 300, 1408, 468),
])
def test_keys_split_over_workgroups(gpu, h, heads, queries, keys, offset):
    q, k, v = inputs(heads, queries, keys, h, queries + keys)
    v[:, min(keys, queries + offset):] = np.nan  # never read
    k[:, min(keys, queries + offset):] = np.nan
    eo, _ = exact(q, np.nan_to_num(k), np.nan_to_num(v), heads, queries, keys, h, h ** -0.5, offset)
    go, _ = run(gpu, q, k, v, heads, queries, keys, h, h ** -0.5, offset, False)
    close(eo, go)
