"""fp32 attention (ar_attn_f32.hip) against fp64 at the edges of its 32-row
tiles, and with values that its bf16 splits cannot hold."""
import math

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    from autoresearch_amd import ops
    return torch, ops


def _inputs(torch, B, T, H, hd, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    q, k, v, do = (torch.randn(B, T, H, hd, generator=g, device="cuda") for _ in range(4))
    q, k = (t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5) for t in (q, k))
    return q.contiguous(), k.contiguous(), v, do


def _run(torch, ops, q, k, v, do, window):
    B, T, H, hd = q.shape
    a = (B, T, H, hd)
    o, dq, dk, dv = (torch.full_like(q, math.nan) for _ in range(4))
    lse, d = (torch.full((B, T, H), math.nan, device="cuda") for _ in range(2))
    ops.flash_attn_fwd(o, lse, q, k, v, *a, window)
    ops.flash_attn_bwd_precompute_d(d, o, do, *a)
    ops.flash_attn_bwd_dq(dq, q, k, v, do, lse, d, *a, window)
    ops.flash_attn_bwd_dkv(dk, dv, q, k, v, do, lse, d, *a, window)
    torch.cuda.synchronize()
    return o, lse, dq, dk, dv


def _exact(torch, q, k, v, do, window):
    T, hd = q.shape[1], q.shape[3]
    Q, K, V, DO = (t.double().permute(0, 2, 1, 3).contiguous() for t in (q, k, v, do))
    i = torch.arange(T, device="cuda")
    ok = i[None, :] <= i[:, None]
    if window > 0:
        ok &= i[None, :] >= i[:, None] - window
    s = (Q @ K.transpose(2, 3).contiguous() / math.sqrt(hd)).masked_fill(~ok, -math.inf)
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse[..., None])
    o = p @ V
    ds = p * (DO @ V.transpose(2, 3).contiguous() - (o * DO).sum(-1, keepdim=True)) / math.sqrt(hd)
    back = lambda t: t.permute(0, 2, 1, 3)  # noqa: E731
    return (back(o), lse.permute(0, 2, 1), back(ds @ K), back(ds.transpose(2, 3).contiguous() @ Q),
            back(p.transpose(2, 3).contiguous() @ DO))


# one row, below / at / past one tile, partial last tiles, more tiles than waves,
# windows around the tile size, and a grid past the dK / dV dispatch's 512 workgroups
@pytest.mark.parametrize("B,T,H,hd,window", [
    (1, 1, 1, 128, 0), (2, 31, 3, 64, 0), (1, 32, 2, 128, 1), (2, 33, 1, 32, 0), (1, 63, 2, 128, 31), (1, 65, 8, 64, 32),
    (2, 100, 3, 128, 33), (1, 255, 2, 32, 0), (1, 513, 2, 128, 200), (3, 1001, 6, 128, 500), (2, 300, 16, 64, 300)])
def test_fp32_attention_vs_fp64(env, B, T, H, hd, window):
    """Norm-wise: scores carry at most hd + 6 fp32 roundings of N(0, 1)-size
    terms, softmax a few more, and the sums over T keys one per matrix
    instruction (2 per 32 keys and one per tile): 1e-6 is above any of them."""
    torch, ops = env
    x = _inputs(torch, B, T, H, hd, B * 1000 + T + hd)
    got, ref = _run(torch, ops, *x, window), _exact(torch, *x, window)
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), got, ref):
        assert bool(torch.isfinite(a).all()), name
        if T == 1 and name in ("dq", "dk", "lse"):  # one key: dS is 0, and LSE the score itself
            assert float((a.double() - b).abs().max()) <= 2e-6
        else:
            assert float((a.double() - b).norm() / b.norm()) <= 1e-6, name


@pytest.mark.parametrize("T", [40, 130])
def test_fp32_attention_non_finite_and_tiny(env, T):
    """An infinite value reaches its own output column, where every query that
    sees it gets +inf as in fp32; a sequence of values near 1e-36 keeps fp32's
    relative accuracy; everything else is untouched."""
    torch, ops = env
    q, k, v, do = _inputs(torch, 3, T, 2, 128, T)
    v[0, 20, 1, 5] = math.inf
    v[1] *= 1e-36
    o, lse, dq, dk, dv = _run(torch, ops, q, k, v, do, 0)
    v0 = v.clone()
    v0[0, 20, 1, 5] = 0.0
    ref = _exact(torch, q, k, v0, do, 0)
    assert bool(torch.isposinf(o[0, 20:, 1, 5]).all())
    o[0, :, 1, 5] = ref[0][0, :, 1, 5].float()  # (queries before it: 0 x inf, as the reference's sum has it)
    for b in range(3):
        assert float((o[b].double() - ref[0][b]).norm() / ref[0][b].norm()) <= 1e-6
    assert float((lse.double() - ref[1]).norm() / ref[1].norm()) <= 1e-6
    for a, b in zip((dq, dk, dv), ref[2:]):
        for i, h in ((2, slice(None)), (1, slice(None)), (0, slice(0, 1))):  # untouched, tiny, the infinity's neighbour
            x, y = a[i, :, h].double(), b[i, :, h]
            assert float((x - y).norm() / y.norm()) <= 1e-6


def _close(torch, got, ref, tol, dim):
    err, size = (got.double() - ref).norm(dim=dim), ref.norm(dim=dim)
    assert bool(torch.isfinite(got).all())
    assert bool((err <= tol * size).all()), float((err / size.clamp_min(1e-300)).max())


# powers of two on q, k, v, dO: values below 2^-110 of one operand behind
# ordinary results (the other operand large), small results of ordinary
# products, and the second pass of every kernel
@pytest.mark.parametrize("sq,sk,sv,sdo", [(112, -112, 0, 0), (-112, 112, 0, 0), (0, 0, -116, 116), (0, 0, 100, -118),
                                          (100, -100, 108, -112), (-100, 100, -116, 120), (-60, 60, -50, 60),
                                          (0, 0, -112, 40), (0, 0, -109, 109), (0, 0, 0, -111)])
@pytest.mark.parametrize("T,hd,window", [(40, 128, 0), (130, 64, 50), (257, 32, 0)])
def test_fp32_attention_of_small_values(env, sq, sk, sv, sdo, T, hd, window):
    """Scaling by powers of two is exact, so the results' relative errors are
    those of test_fp32_attention_vs_fp64 (the terms of every result are 2^-118 or
    more in size, so fp32's own subnormal roundings, 2^-149 each, do not show)."""
    torch, ops = env
    q, k, v, do = _inputs(torch, 2, T, 2, hd, T + hd)
    q, k, v, do = q * 2.0 ** sq, k * 2.0 ** sk, v * 2.0 ** sv, do * 2.0 ** sdo
    got, ref = _run(torch, ops, q, k, v, do, window), _exact(torch, q, k, v, do, window)
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), got, ref):
        _close(torch, a, b, 2e-6, (1, 3) if name != "lse" else 1)


@pytest.mark.parametrize("T", [40, 130])
def test_fp32_attention_of_small_values_beside_large(env, T):
    """Single columns below 2^-110 beside ordinary ones: every column of O, dK,
    dV and dQ keeps fp32's accuracy by itself (column 3 of V and column 2 of Q,
    K and dO are small, with dO's column 3 and one of q and k large)."""
    torch, ops = env
    q, k, v, do = _inputs(torch, 1, T, 2, 64, T)
    v[..., 3] *= 2.0 ** -116
    do[..., 3] *= 2.0 ** 20
    k[..., 2] *= 2.0 ** -118
    q[..., 2] *= 2.0 ** 30
    do[..., 2] *= 2.0 ** -114
    got, ref = _run(torch, ops, q, k, v, do, 0), _exact(torch, q, k, v, do, 0)
    for a, b in zip((got[0],) + got[2:], (ref[0],) + ref[2:]):
        _close(torch, a, b, 4e-6, 1)


@pytest.mark.parametrize("T", [40, 130])
def test_fp32_attention_second_pass_is_finite(env, T):
    """A finite value that bf16 rounds to infinity has the blocks it reaches
    formed again: their results, and those of the rows beside it, as fp64 has
    them (dO's large value meets a column of V, and so of O, that is zero)."""
    torch, ops = env
    q, k, v, do = _inputs(torch, 2, T, 2, 128, T)
    v[0, :, 1, 5] = 0.0
    do[0, 20, 1, 5] = 3.3999e38
    got, ref = _run(torch, ops, q, k, v, do, 0), _exact(torch, q, k, v, do, 0)
    for a, b in zip(got[2:4], ref[2:4]):
        _close(torch, a, b, 1e-6, (1, 3))
    a, b = got[4], ref[4]
    _close(torch, a[0, :, 1, 5][None, :21], b[0, :, 1, 5][None, :21], 1e-6, 1)
    a[0, :, 1, 5] = b[0, :, 1, 5].float()  # (the keys after query 20 have the other queries' ordinary sums)
    _close(torch, a, b, 1e-6, (1, 3))
    v[0, 20, 1, 5] = 3.3999e38
    o, lse = _run(torch, ops, q, k, v, do, 0)[:2]
    _close(torch, o, _exact(torch, q, k, v, do, 0)[0], 1e-6, 1)
