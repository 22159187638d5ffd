"""The fp32 products (ar_gemm_f32.hip): three-term bf16 splits on the bf16
matrix cores, against fp64, at the edges of every block tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    from autoresearch_amd import ops
    import gpu_util as gu
    return torch, ops, gu


def _products(torch, ops, gu, M, N, K, x, w, dy, dw0):
    y, dx, dw = gu.empty(M, N), gu.empty(M, K), dw0.clone()
    ops.linear_fwd(y, x, w, M, N, K)
    ops.linear_bwd_dx(dx, dy, w, M, N, K)
    ops.linear_bwd_dw(dw, dy, x, M, N, K)
    torch.cuda.synchronize()
    return y, dx, dw


# one block and one past it in each direction for the 32, 64, 128 and 256 wide
# tiles, reductions of whole and partial k-tiles, extents 8 and 9, and sizes
# that choose the large tiles and a split reduction
SHAPES = [(8, 8, 8), (9, 9, 9), (32, 32, 128), (33, 31, 129), (64, 64, 64), (65, 63, 71), (1, 40, 24), (128, 128, 32),
          (129, 257, 33), (515, 130, 1999), (2048, 513, 520), (4100, 1031, 96), (8192, 2048, 64), (30, 77, 5001),
          (7, 300, 5), (4097, 3, 12),
          # short reductions of large outputs: fwd over K, dW over M, one k-tile, a part of one, three
          (1024, 1031, 8), (1100, 1024, 48), (1030, 1021, 33), (16, 1024, 1024), (9, 1030, 1027), (33, 2050, 1000),
          (96, 1999, 1030)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp32_products_vs_fp64(env, M, N, K):
    """Each value is split exactly, the dropped terms are below 2^-25 of the
    product, and every accumulation rounds once per matrix instruction (six per
    16 k-values, plus the group, split and epilogue adds): elementwise |error| <=
    2^-24 (6 R / 16 + 8) sum |a b| with R the reduction length, and norm-wise no
    more than one random fp32 rounding per term, 2^-24 sqrt(R + 8)."""
    torch, ops, gu = env
    r = gu.rng(M * 7 + N * 3 + K)
    x, w, dy, dw0 = (gu.dev(gu.randn(r, *s)) for s in ((M, K), (N, K), (M, N), (N, K)))
    y, dx, dw = _products(torch, ops, gu, M, N, K, x, w, dy, dw0)
    X, W, DY = x.double(), w.double(), dy.double()
    for got, a, b, c in ((y, X, W.T, None), (dx, DY, W, None), (dw, DY.T, X, dw0.double())):
        ref, mass = a @ b, a.abs() @ b.abs()
        if c is not None:
            ref, mass = ref + c, mass + c.abs()
        R = a.shape[1]
        err = (got.double() - ref).abs()
        assert bool((err <= 2.0 ** -24 * (6 * R / 16 + 8) * mass).all())
        assert float(err.norm() / ref.norm()) <= 2.0 ** -24 * np.sqrt(R + 8)


@pytest.mark.parametrize("M,N,K", [(40, 48, 56), (300, 130, 256), (2048, 512, 64)])
def test_fp32_products_non_finite_and_extreme(env, M, N, K):
    """Infinities, NaN and values that bf16 rounds to infinity give what fp32
    products give (the affected outputs are formed on the fp32 matrix cores),
    and leave every other output alone."""
    torch, ops, gu = env
    r = gu.rng(M + N + K)
    x, w, dy, dw0 = (gu.randn(r, *s) for s in ((M, K), (N, K), (M, N), (N, K)))
    x[3, 5], x[7, 2], dy[1, 9], dy[5, 4] = np.inf, np.nan, -np.inf, np.float32(3.4e38)
    w[:, 11] = np.abs(w[:, 11]) + 0.5
    x[9, :] = 0.0
    x[9, 11] = np.float32(3.3999e38)  # finite in fp32, rounds to infinity in bf16
    w[2, :] = 0.0
    w[2, 11] = 1.0
    dev = [gu.dev(a) for a in (x, w, dy, dw0)]
    y, dx, dw = _products(torch, ops, gu, M, N, K, *dev)
    with np.errstate(all="ignore"):
        for got, a, b, c in ((y, x, w.T, 0.0), (dx, dy, w, 0.0), (dw, dy.T, x, dw0)):
            ref = (a.astype(np.float64) @ b.astype(np.float64) + c)
            big = np.abs(ref) > 3.4028235e38
            ref32 = np.where(big, np.copysign(np.inf, ref), ref)
            g = gu.host(got).astype(np.float64)
            fine = np.isfinite(ref32)
            # |sum| close to the fp32 limit may overflow in one order and not another
            edge = np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64)) > 3.0e38
            edge |= ~np.isfinite(np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64)))
            plain = fine & ~edge
            assert np.isfinite(g[plain]).all()
            assert np.linalg.norm(g[plain] - ref32[plain]) <= 1e-6 * np.linalg.norm(ref32[plain])
            assert np.array_equal(np.isnan(g[~fine & ~big]), np.isnan(ref32[~fine & ~big]))
            inf = np.isinf(ref32) & ~big
            assert np.array_equal(g[inf], ref32[inf])
    assert float(y[9, 2]) == np.float32(3.3999e38)


# GEMM-space sizes that choose each block tile, ragged ones, and a split reduction
@pytest.mark.parametrize("m,n,r", [(40, 48, 72), (33, 57, 131), (1024, 1000, 64), (1040, 1030, 33), (2050, 1999, 40), (8192, 2048, 64),
                                   (64, 72, 20000)])
@pytest.mark.parametrize("exp,up", [(-109, 100), (-111, 100), (-111, 20), (-118, 20), (-125, 100), (-140, 20), (-140, 100)])
@pytest.mark.parametrize("mixed", [False, True])
def test_fp32_products_of_small_values(env, m, n, r, exp, up, mixed):
    """Operands near 2^exp (below 2^-110 bf16 has no bits for their low terms):
    as whole rows of one operand, or beside larger values of the same row that
    meet zeros.  The other operand is scaled by 2^up, to ordinary and to small
    outputs, and has a row of zeros.  Products and sums are of the same kind as
    in test_fp32_products_vs_fp64, and so is the bound (the least output, 2^-120,
    still has all its bits).  Either operand is the small one, in all three layouts."""
    torch, ops, gu = env
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + r + up - exp)
    small = torch.randn(m if m < n else n, r, generator=g, device="cuda")
    other = torch.randn(max(m, n), r, generator=g, device="cuda") * 2.0 ** up
    other[5] = 0.0
    if mixed:
        small[:, 1::2] *= 2.0 ** exp
        other[:, 0::2] = 0.0
    else:
        small[::3] *= 2.0 ** exp
    for first in (False, True):
        A, B = (small, other) if first else (other, small)
        M, N = A.shape[0], B.shape[0]
        At, Bt = A.T.contiguous(), B.T.contiguous()
        y, dx, dw = gu.empty(M, N), gu.empty(M, N), torch.zeros(M, N, device="cuda")
        ops.linear_fwd(y, A, B, M, N, r)
        ops.linear_bwd_dx(dx, A, Bt, M, r, N)
        ops.linear_bwd_dw(dw, At, Bt, r, M, N)
        ref, mass = A.double() @ Bt.double(), A.double().abs() @ Bt.double().abs()
        for got in (y, dx, dw):
            assert bool(((got.double() - ref).abs() <= 2.0 ** -24 * (6 * r / 16 + 8) * mass).all())
            # one random rounding per term: row by row, whatever the rows' magnitudes
            rows = 1 if first else 0
            err = (got.double() - ref).norm(dim=rows) / ref.norm(dim=rows).clamp_min(1e-300)
            assert float(err.max()) <= 2.0 ** -24 * 2 * np.sqrt(r + 8)
