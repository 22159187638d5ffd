"""Row kernels of ar_reduce.hip (softmax, cross entropy) at the edges of their
register-held lengths, and softcap's tanh, against fp64."""
import math

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    from autoresearch_amd import ops
    return torch, ops


# one value, partial 4-value chunks, both sides of each register-held length, rows read twice
@pytest.mark.parametrize("V", [1, 3, 4, 5, 257, 511, 512, 513, 2047, 2048, 2050, 8191, 8192, 8196, 16384, 16387, 40001])
def test_rows_of_exponentials_vs_fp64(env, V):
    torch, ops = env
    n, scale = 37, 0.37
    g = torch.Generator(device="cuda")
    g.manual_seed(V)
    x = torch.randn(n, V, generator=g, device="cuda") * 4
    tg = torch.randint(0, V, (n,), generator=g, device="cuda")
    tg[3], tg[5], tg[0], tg[1] = -1, V, V - 1, 0  # two ignored rows, the ends of a row
    if V > 2:
        x[7, : V - 1] = -math.inf  # whole chunks and waves without a finite value
        tg[7] = V - 1
        x[8, V // 2:] = -math.inf
        tg[8] = 0
    x[9, V // 2] = math.nan
    x[10, 0] = math.inf
    p, gr = (torch.full_like(x, 7.0) for _ in range(2))
    loss = torch.full((n,), 7.0, device="cuda")
    ops.softmax_fwd(p, x, n, V)
    ops.cross_entropy_fwd(loss, x, tg, n, V)
    ops.cross_entropy_softcap_bwd(gr, x, tg, 15.0, n, V, scale)
    inplace = x.clone()
    ops.cross_entropy_softcap_bwd(inplace, inplace, tg, 15.0, n, V, scale)
    torch.cuda.synchronize()
    torch.testing.assert_close(inplace, gr, rtol=0, atol=0, equal_nan=True)
    ok = (tg >= 0) & (tg < V)
    assert (loss[~ok] == 0).all() and (gr[~ok] == 0).all()
    for t in (p, gr):
        assert t[9:11].isnan().all()
    assert loss[9:11].isnan().all()
    live = ok.clone()
    live[9:11] = False
    X = x.double()
    P = torch.softmax(X, 1)
    # an exponential of x - m: the difference's and its product with log2 e's
    # rounding (2^-24 of up to 40 each, times ln 2), 2 ulp of the exponential;
    # the sum and the quotient a few more
    rel = (2 * 40 + 8) * 2.0 ** -24
    keep = torch.arange(n, device="cuda")
    keep = keep[(keep != 9) & (keep != 10)]
    assert ((p[keep] - P[keep]).abs() <= rel * P[keep] + 2.0 ** -126).all()
    G = P.clone()
    G[live] -= torch.nn.functional.one_hot(tg[live], V)
    assert ((gr[live] - scale * G[live]).abs() <= scale * (rel * P[live] + 2.0 ** -23 * G[live].abs()) + 2.0 ** -126).all()
    L = torch.logsumexp(X, 1) - X.gather(1, tg.clamp(0, V - 1)[:, None])[:, 0]
    assert ((loss[live] - L[live]).abs() <= rel + 2.0 ** -23 * (L[live].abs() + 40)).all()


@pytest.mark.parametrize("n,off", [(1, 0), (5, 0), (4096, 0), (4096, 1), (100003, 0)])
@pytest.mark.parametrize("cap", [15.0, 0.3])
def test_softcap_vs_fp64(env, n, off, cap):
    torch, ops = env
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    buf = torch.randn(n + off, generator=g, device="cuda") * cap * 10.0 ** (torch.rand(n + off, generator=g, device="cuda") * 6 - 5)
    out = torch.full((n + off + 1,), 7.0, device="cuda")
    x = buf[off:off + n]
    ops.softcap_fwd(out[off:off + n], x, cap, n)
    torch.cuda.synchronize()
    assert (out[off + n:] == 7).all() and (out[:off] == 7).all()
    ref = cap * torch.tanh(x.double() / cap)
    # x / cap, tanh (0.9 ulp) and the product: under 4 ulp
    assert ((out[off:off + n] - ref).abs() <= 4 * 2.0 ** -23 * ref.abs() + 2.0 ** -126).all()


def test_softcap_limits(env):
    torch, ops = env
    x = torch.tensor([0.0, -0.0, math.inf, -math.inf, math.nan, 1e30, -1e30, 3e-39], device="cuda")
    y = torch.empty_like(x)
    ops.softcap_fwd(y, x, 15.0, 8)
    got = y.tolist()
    assert got[:4] == [0.0, 0.0, 15.0, -15.0] and math.copysign(1, got[1]) == -1
    assert math.isnan(got[4]) and got[5:7] == [15.0, -15.0] and abs(got[7] - 3e-39) < 1e-43


# vectors of 4 in batches of 4 per thread of a 512 x 256 grid: one value, a
# remainder alone, both sides of a whole round of the grid, an odd batch count
@pytest.mark.parametrize("n", [1, 3, 4, 7, 1025, 524288, 2097151, 2097152, 2097157, 6815749])
@pytest.mark.parametrize("shift", [0, 1])
def test_fixed_sums_vs_fp64(env, n, shift):
    torch, ops = env
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    a, b = (torch.randn(n + 1, generator=g, device="cuda")[shift:shift + n] for _ in range(2))
    dot, mean = torch.full((3,), 2.0, device="cuda"), torch.zeros(1, device="cuda")
    ops.scalar_grad_reduce(dot, a, b, 1, n)
    ops.mean_reduce(mean, a, n)
    a64, b64 = a.double(), b.double()
    # a value passes fewer than 64 roundings: its thread's sum, then the
    # trees of a block and of the blocks
    eps = 64 * 2.0 ** -24
    assert abs(dot[1].item() - 2.0 - (a64 * b64).sum().item()) <= eps * ((a64 * b64).abs().sum().item() + 2.0)
    assert abs(mean.item() - a64.mean().item()) <= eps * a64.abs().mean().item()
    assert dot[0].item() == 2.0 and dot[2].item() == 2.0
