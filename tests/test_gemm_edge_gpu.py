"""The persistent bf16-storage GEMM with edge tiles (rows and columns that are
multiples of 8 but not of 256) against fp64, all layouts, output types,
accumulation, reduction splits and fused epilogues."""
import math

import pytest

pytestmark = pytest.mark.gpu


# last tile of 8, of 128 and of 248 rows / columns, several items per
# workgroup (two rounds), tiles that only the row or only the column cuts
@pytest.mark.parametrize("M,N,K", [(13320, 2560, 640), (16384, 640, 2560), (16384, 2560, 640), (16320, 1016, 128),
                                   (8192, 2048 + 248, 64), (40960, 456, 192), (4032, 4032, 4032), (8192, 1528, 1016)])
@pytest.mark.parametrize("layout,c_bf16,acc", [(0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 0, 0), (1, 1, 1), (2, 0, 0), (2, 1, 1)])
def test_edge_tiles_vs_fp64(M, N, K, layout, c_bf16, acc):
    import torch
    from autoresearch_amd import _lib
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    bf = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    x, w, dy = bf(M, K), bf(N, K), bf(M, N)
    a, b, shape = ((x, w, (M, N)), (dy, w, (M, K)), (dy, x, (N, K)))[layout]
    t = torch.bfloat16 if c_bf16 else torch.float32
    buf = torch.full((shape[0] * shape[1] + 4096,), 3.0, device="cuda", dtype=t)  # the tail must stay
    c = buf[:shape[0] * shape[1]].view(shape)
    c0 = torch.randn(shape, generator=g, device="cuda").to(t) if acc else torch.zeros(shape, device="cuda", dtype=t)
    c.copy_(c0)
    _lib.check(_lib.load().ar_gemm_mixed(torch.cuda.current_stream().cuda_stream, layout, c.data_ptr(), c_bf16,
                                         a.data_ptr(), 1, b.data_ptr(), 1, M, N, K, acc), "gemm_mixed")
    torch.cuda.synchronize()
    assert (buf[shape[0] * shape[1]:] == 3).all()
    A, B = a.double(), b.double()
    if layout == 0:
        want, mag, red = A @ B.T.contiguous(), A.abs() @ B.T.contiguous().abs(), K
    elif layout == 1:
        want, mag, red = A @ B, A.abs() @ B.abs(), N
    else:
        want, mag, red = A.T.contiguous() @ B, A.T.contiguous().abs() @ B.abs(), M
    want += c0.double()
    # fp32 accumulation of exact products: roundings of 2^-24 of partial sums,
    # which for random signs stay far below mag; then the output's rounding
    tol = 8 * 2.0 ** -24 * mag + 1e-6 + (2.0 ** -8 if c_bf16 else 2.0 ** -23) * want.abs()
    assert not ((c.double() - want).abs() > tol).any()


def test_edge_tile_epilogues_in_a_training_step():
    """A model 640 wide (no multiple of 256): its residual, ReLU^2 and ReLU^2
    gradient products run on edge tiles at 16384 tokens and on gemm_k at 2048,
    with the same products in the same order: the losses of 32 sequences
    together are those of 4 at a time."""
    import torch
    from autoresearch_amd.model import BF16, GPT, GPTConfig
    T, V = 512, 512
    cfg = GPTConfig(T, V, 2, 5, 5, 640, 128, 640)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.randint(0, V, (32, T), generator=g, device="cuda")
    y = torch.randint(0, V, (32, T), generator=g, device="cuda")

    def run(B, xs, ys):
        m = GPT(cfg, B, T, precision=BF16, rope_period=T)
        m.init_weights(42)
        p = m.params()
        r = torch.Generator(device="cuda")
        r.manual_seed(5)
        p += 0.02 * torch.randn(p.numel(), generator=r, device="cuda")
        m.zero_grads()
        m.forward(xs, ys)
        m.backward(xs, ys)
        torch.cuda.synchronize()
        out = m.token_loss().clone().reshape(-1), m.grads().clone()
        m.close()
        return out

    loss, grads = run(32, x, y)
    parts = [run(4, x[i:i + 4].contiguous(), y[i:i + 4].contiguous()) for i in range(0, 32, 4)]
    torch.testing.assert_close(loss, torch.cat([p[0] for p in parts]), rtol=1e-5, atol=1e-5)
    # the gradient is that of the summed token losses, so the parts' add up, in
    # another order and from bf16 gradients of other roundings
    want = torch.stack([p[1] for p in parts]).double().sum(0)
    err = (grads.double() - want).norm() / want.norm()
    assert err < 2.0 ** -8, float(err)
