"""bf16 products on fp32 tensors (ar_flash.hip) at every kind of head_dim,
against fp64 on the rounded operands."""
import math

import pytest

pytestmark = pytest.mark.gpu


# the tiled sizes, below / between them, rows only 4- and 8-byte aligned, one
# column; T below, at and past the 32-, 64- and 128-row blocks; windows
@pytest.mark.parametrize("B,T,H,hd,window", [
    (1, 33, 2, 32, 0), (2, 129, 3, 64, 0), (1, 300, 2, 128, 70), (1, 64, 2, 1, 0), (1, 65, 3, 5, 16), (2, 127, 1, 30, 0),
    (1, 128, 2, 33, 0), (1, 200, 2, 50, 64), (2, 257, 2, 63, 0), (1, 161, 3, 80, 100), (2, 31, 1, 97, 0),
    (1, 260, 2, 126, 0), (1, 5, 1, 127, 2), (1, 1, 1, 48, 0),
    # one 128-row block of a tiled size: every operand is rounded
    (2, 128, 3, 128, 0), (3, 100, 2, 64, 40), (2, 1, 2, 32, 0)])
def test_bf16_attention_of_fp32_tensors_vs_fp64(B, T, H, hd, window):
    import torch
    from autoresearch_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(T * 131 + hd)
    q, k, v, do = (torch.randn(B, T, H, hd, generator=g, device="cuda") for _ in range(4))
    q, k = (t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5) for t in (q, k))
    q, k = q.contiguous(), k.contiguous()
    a = (B, T, H, hd)
    guard = torch.full((B * T * H * hd + 64,), 7.0, device="cuda")
    outs = [guard.clone() for _ in range(4)]
    o, dq, dk, dv = (t[:q.numel()].view_as(q) for t in outs)
    lse, d = (torch.full((B, T, H), math.nan, device="cuda") for _ in range(2))
    ops.flash_attn_fwd(o, lse, q, k, v, *a, window, bf16=True)
    ops.flash_attn_bwd_precompute_d(d, o, do, *a, bf16=True)
    ops.flash_attn_bwd_dq(dq, q, k, v, do, lse, d, *a, window, bf16=True)
    ops.flash_attn_bwd_dkv(dk, dv, q, k, v, do, lse, d, *a, window, bf16=True)
    alias = q.clone()  # a result may take the place of an operand that only its own rows read
    ops.flash_attn_bwd_dq(alias, alias, k, v, do, lse, d, *a, window, bf16=True)
    torch.cuda.synchronize()
    assert torch.equal(alias, dq)
    for t in outs:
        assert (t[q.numel():] == 7).all()
    Q, K, V, DO = (t.bfloat16().double().permute(0, 2, 1, 3).contiguous() for t in (q, k, v, do))
    i = torch.arange(T, device="cuda")
    ok = i[None, :] <= i[:, None]
    if window > 0:
        ok &= i[None, :] >= i[:, None] - window
    tr = lambda t: t.transpose(2, 3).contiguous()  # noqa: E731
    sc = 1 / math.sqrt(hd)
    s = (Q @ tr(K) * sc).masked_fill(~ok, -math.inf)
    L = torch.logsumexp(s, -1)
    P = torch.exp(s - L[..., None])
    O = P @ V
    dP = DO @ tr(V)
    D = (O * DO).sum(-1, keepdim=True)
    dS = P * (dP - D)
    # P and dS enter their products rounded to bf16 (2^-9 relative, twice for
    # the sums' own roundings); D carries O's error, 2^-9 of P's row times |V|
    u = 2.0 ** -8
    eO = u * (P @ V.abs()) + 1e-5
    eS = u * dS.abs() + P * ((eO * DO.abs()).sum(-1, keepdim=True) + 1e-4)
    bounds = (eO, sc * (eS @ K.abs()) + 1e-5, sc * (tr(eS) @ Q.abs()) + 1e-5, u * (tr(P) @ DO.abs()) + 1e-5)
    want = (O, sc * (dS @ K), sc * (tr(dS) @ Q), tr(P) @ DO)
    for name, got, w, e in zip(("o", "dq", "dk", "dv"), (o, dq, dk, dv), want, bounds):
        bad = ((got.double().permute(0, 2, 1, 3) - w).abs() > e)
        assert not bad.any(), (name, int(bad.sum()))
    assert (lse.double().permute(0, 2, 1) - L).abs().max() < 1e-4
