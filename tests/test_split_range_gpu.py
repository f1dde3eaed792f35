"""The fp32 tile engine (gemm_f32.h) at the ends of its arithmetic: operands split into three bf16 parts.

Every layout and tile (128 x 128, 128 x 64, 64 x 64, persistent; 16-byte and 4-byte-aligned loads), at the edges
of its tiles, against the float64 product:
- wide spreads of magnitude, within the bound of an fp32 sum in any order, (K + 8) 2^-24 sum |a| |b|;
- operands the split does not hold (nonzero under 2^-110; the kernel computes such tiles again with the fp32
  instruction), of every size down to the subnormals, with ordinary and with huge partners, whatever the size of
  the outputs: the same bound plus K of the smallest subnormal;
- sums of one to four products, where the split's own error shows: one product is rounded once, and up to four are
  within the terms left out plus one rounding;
- infinities and NaN: the same outputs are NaN or infinite (with the same sign) as in the float64 product, the
  others within the bound."""
import numpy as np
import pytest

from staleynet_amd import gemm
from staleynet_amd.gemm import MatmulSpec, Shape

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24
SHAPES = [  # m, n, k and the tile it takes on 256 CUs (0: the register path's own)
    (128, 60, 96, (128, 64)),        # narrow
    (260, 132, 68, (64, 64)),        # small, ragged by 4
    (131, 197, 131, (64, 64)),       # small, unaligned
    (129, 67, 33, (128, 128)),       # square, unaligned, one step and one element
    (4096, 4096, 256, (128, 128)),   # persistent
    (2052, 4100, 132, (128, 128)),   # square, edges, a partial last step
]
IDS = [f"{m}x{n}x{k}" for m, n, k, _ in SHAPES]


def run(gpu, layout, m, n, k, a, b, tile):
    spec = MatmulSpec.new(m, n, k)
    left, right = a, b
    if layout[0] == "T":
        spec, left = spec.left_transposed(), a.T
    if layout[1] == "T":
        spec, right = spec.right_transposed(), b.T
    plan = gemm.plan(spec, cu_count=256)
    assert tile is None or (plan.tile_rows, plan.tile_cols) == tile, (plan.tile_rows, plan.tile_cols)
    print(f"{layout} {m}x{n}x{k} path {plan.path}", flush=True)
    lt = gpu.upload(Shape.vector(m * k), np.ascontiguousarray(left).ravel())
    rt = gpu.upload(Shape.vector(k * n), np.ascontiguousarray(right).ravel())
    out = gpu.zeros(Shape(m, n))
    gpu.matmul(spec, lt, rt, out)
    got = gpu.download(out).reshape(m, n)
    for t in (lt, rt, out):
        t.free()
    return got


def check(got, a, b, k):
    with np.errstate(invalid="ignore", over="ignore"):
        expected = a.astype(np.float64) @ b.astype(np.float64)
        bound = (k + 8) * EPS * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + k * 2.0 ** -149
    finite = np.isfinite(expected)
    assert np.array_equal(np.isnan(expected), np.isnan(got))
    assert np.array_equal(expected[np.isinf(expected)], got[np.isinf(expected)].astype(np.float64))
    excess = np.abs(got[finite] - expected[finite]) - bound[finite]
    assert excess.max(initial=-1.0) <= 0.0, f"{int((excess > 0).sum())} outputs past the bound"


@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,tile", SHAPES, ids=IDS)
def test_spread_and_tiny_operands(gpu, layout, m, n, k, tile):
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)) * np.exp(4.0 * rng.standard_normal((m, k)))
    b = rng.standard_normal((k, n)) * np.exp(4.0 * rng.standard_normal((k, n)))
    a, b = a.astype(np.float32), b.astype(np.float32)
    check(run(gpu, layout, m, n, k, a, b, tile), a, b, k)
    # Rows of magnitude 2^-115 .. 2^-126, whose lowest bits no bf16 holds, and subnormal ones.
    tiny = np.ldexp(a, -110 - (np.arange(m) % 30)[:, None]).astype(np.float32)
    check(run(gpu, layout, m, n, k, tiny, b, tile), tiny, b, k)


@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,tile", SHAPES, ids=IDS)
def test_tiny_operands_with_huge_partners(gpu, layout, m, n, k, tile):
    rng = np.random.default_rng(m * k + n)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    for down, up in ((-112, 30), (-120, 60), (-136, 118), (-140, 0)):
        x, y = np.ldexp(a, down), np.ldexp(b, up)
        check(run(gpu, layout, m, n, k, x, y, tile), x, y, k)
        check(run(gpu, layout, m, n, k, np.ldexp(a, up), np.ldexp(b, down), tile), np.ldexp(a, up), np.ldexp(b, down), k)
    # One tiny column, the only one of some rows, with a huge partner row; the last k and row of ragged tiles too.
    for column, row in ((k // 2, 0), (k - 1, m - 1)):
        x, y = a.copy(), b.copy()
        x[:, column] = np.ldexp(a[:, column], -125)
        y[column] = np.ldexp(b[column], 110)
        for r in {row, m // 2}:
            x[r, :column] = 0.0
            x[r, column + 1:] = 0.0
        check(run(gpu, layout, m, n, k, x, y, tile), x, y, k)


@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,tile", SHAPES, ids=IDS)
def test_infinities_nan_and_the_largest_values(gpu, layout, m, n, k, tile):
    rng = np.random.default_rng(m * n + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    a[:, 0], a[:, k - 1] = 0.25, -0.25  # the partners of the largest values below
    a[m // 2, k - 1] = np.inf
    a[m - 1, 0] = -np.inf
    a[0, k // 2] = np.nan
    b[k // 3, n - 1] = np.inf
    b[k - 1, 0] = np.float32(3.4e38)  # the largest values have no bf16 above them
    b[0, n // 2] = np.float32(-3e38)
    a[1, :] = np.ldexp(a[1, :], -20)
    b[:, 1] = 0.0  # infinity times zero
    check(run(gpu, layout, m, n, k, a, b, tile), a, b, k)


@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("m,n", [(128, 60), (260, 132), (2052, 4100)])  # every tile, by the alignment of k too
@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_sums_of_few_products(gpu, layout, m, n, k):
    # Values with the largest rests a split by truncation leaves among mantissas of every kind. Past K = 1: the terms
    # left out are under 2^-24 of each product, the last addition rounds by 2^-24 of the sum, the five before it
    # (2^-8 of it and less) are within 2^-6 of that.
    rng = np.random.default_rng(m + k)
    a = (rng.uniform(1, 2, (m, k)) * rng.choice([-1, 1], (m, k))).astype(np.float32)
    b = rng.uniform(1, 2, (k, n)).astype(np.float32)
    worst = np.array([0x3f80ff80], np.uint32).view(np.float32)[0]
    a[::3], b[:, ::2] = worst, worst
    got = run(gpu, layout, m, n, k, a, b, None)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    if k == 1:
        assert np.array_equal(got, exact.astype(np.float32))
    bound = (2 + 2.0 ** -6) * EPS * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert np.max(np.abs(got - exact) / bound) <= 1.0
