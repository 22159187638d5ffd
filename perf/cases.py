"""Measured cases: what a user of this library has it do, through its public
entry points, and what each call has to return.

`listed()` are the cases that are timed by name and `draw()` gives more of the
same ranges.  `prepare()` makes what a program holds before the call, `run()`
is one pass, `work()` the bytes and operations such a pass cannot do without,
`tolerance()` how far another correct implementation at the same precision may
be off, and `exact()` the same outputs from plain torch in 64 bits.

Kinds of case:
  train      the whole training step (zero_grads, forward, backward, AdamW and
             Muon) of a model of the configured depth rule, at 8192 tokens of
             vocabulary, as the training driver and the benchmark run it
  linear     one linear layer: forward, input gradient, weight gradient.
             mode "fp32" and "bf16" take fp32 buffers, "stored" takes bf16 ones
  attention  one attention layer: forward, D, dQ, dK and dV
  rows       everything of a layer that is no matrix product (embedding, norms,
             RoPE, ReLU^2, value-embedding gate) and the softcapped loss, each
             forward and backward, in fp32
  optimizer  one layer's six matrices through Muon and one embedding through AdamW
"""
import math

import torch

from autoresearch_amd import _lib, ops
from autoresearch_amd.model import BF16, FP32, GPT, GPTConfig

GATE = 32        # gate channels of the value embedding
CAP = 15.0       # logit softcap
VOCAB = 8192
D = torch.float64
POLAR = [(8.156554524902461, -22.48329292557795, 15.878769915207462),
         (4.042929935166739, -2.808917465908714, 0.5000178451051316),
         (3.8916678022926607, -2.772484153217685, 0.5060648178503393),
         (3.285753657755655, -2.3681294933425376, 0.46449024233003106),
         (2.3465413258596377, -1.7097828382687081, 0.42323551169305323)]


def listed():
    return [
        # the benchmark's training step: depth 8, d512, T 2048, B 32, bf16 compute
        {"name": "train_full_bf16", "kind": "train", "depth": 8, "B": 32, "T": 2048, "precision": "bf16"},
        # the training driver as shipped: its default batch, the reference's fp32
        {"name": "train_driver_fp32", "kind": "train", "depth": 8, "B": 4, "T": 512, "precision": "fp32"},
        # the tiny test model's layer: latency and launches
        {"name": "linear_small_fp32", "kind": "linear", "M": 128, "N": 512, "K": 128, "mode": "fp32"},
        # an MLP layer of the depth-8 model at four sequences, the reference's precision
        {"name": "linear_fp32", "kind": "linear", "M": 8192, "N": 2048, "K": 512, "mode": "fp32"},
        # sizes that are no multiple of anything
        {"name": "linear_fp32_ragged", "kind": "linear", "M": 1999, "N": 1030, "K": 515, "mode": "fp32"},
        # the fused q | k | v product at B 16, T 2048: fp32 buffers, bf16 compute
        {"name": "linear_bf16", "kind": "linear", "M": 32768, "N": 1536, "K": 512, "mode": "bf16"},
        # an MLP layer of the depth-10 model (d640) on bf16 storage
        {"name": "linear_stored", "kind": "linear", "M": 16384, "N": 2560, "K": 640, "mode": "stored"},
        # an attention layer of the driver's batch, half-length window
        {"name": "attention_fp32", "kind": "attention", "B": 4, "T": 512, "H": 4, "hd": 128, "window": 256,
         "precision": "fp32"},
        # the isolated attention benchmark: B 16, H 4, T 2048, causal
        {"name": "attention_bf16", "kind": "attention", "B": 16, "T": 2048, "H": 4, "hd": 128, "window": 0,
         "precision": "bf16"},
        # a head size between the tiled ones, a length that fills no tile
        {"name": "attention_bf16_ragged", "kind": "attention", "B": 3, "T": 1001, "H": 6, "hd": 96, "window": 500,
         "precision": "bf16"},
        # the row passes of the depth-8 model at four sequences
        {"name": "rows", "kind": "rows", "M": 8192, "C": 512, "H": 4, "V": VOCAB},
        # one depth-8 layer and its embedding
        {"name": "optimizer", "kind": "optimizer", "C": 512, "V": VOCAB, "precision": "fp32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "linear", "linear", "linear", "attention", "attention", "rows", "optimizer"])
    if kind == "train":
        prec = rng.choice(["bf16", "fp32"])
        depth = rng.randint(2, 8)
        T = 8 * _log(rng, 8, 256)
        most = 65536 if prec == "bf16" else 4096
        return {"kind": kind, "depth": depth, "B": max(1, _log(rng, 1, max(1, most // T))), "T": T,
                "precision": prec}
    if kind == "linear":
        mode = rng.choice(["fp32", "bf16", "stored"])
        while True:
            M, N, K = _log(rng, 16, 65536), _log(rng, 32, 8192), _log(rng, 32, 4096)
            if rng.random() < 0.6 or mode == "stored":  # bf16 storage takes multiples of 8
                M, N, K = [(x + 7) // 8 * 8 for x in (M, N, K)]
            if M * N * K < 3.4e10 and max(M * N, M * K, N * K) < 1.4e8:
                return {"kind": kind, "M": M, "N": N, "K": K, "mode": mode}
    if kind == "attention":
        prec = rng.choice(["bf16", "fp32"])
        while True:
            B, T, H = _log(rng, 1, 32), _log(rng, 33, 2048), rng.randint(1, 8)
            hd = rng.choice([32, 64, 128, 128, 48, 80, 96])
            if B * T * T * H * hd < (3.5e10 if prec == "bf16" else 4e9):
                return {"kind": kind, "B": B, "T": T, "H": H, "hd": hd,
                        "window": rng.choice([0, T, T // 2, T // 2, rng.randint(1, T)]), "precision": prec}
    if kind == "rows":
        C = 128 * rng.randint(1, 6)
        return {"kind": kind, "M": _log(rng, 64, 16384), "C": C, "H": C // 128, "V": 8 * _log(rng, 64, 1024)}
    return {"kind": kind, "C": 128 * rng.randint(1, 8), "V": 8 * _log(rng, 64, 1024),
            "precision": rng.choice(["bf16", "fp32"])}


# ---------------------------------------------------------------- inputs

_scratch = None


def _workspace():
    """One workspace for the process, bound to its stream, as a program makes it once."""
    global _scratch
    if _scratch is None:
        _scratch = ops.Workspace(2 << 30).bind()


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(scale)


def _zipf(g, n, V):
    """Token ids with the long tail that text has: p_k ~ 1 / (k + 1)^1.1."""
    p = 1.0 / torch.arange(1, V + 1, dtype=D, device="cuda") ** 1.1
    cdf = torch.cumsum(p / p.sum(), 0)
    u = torch.rand(n, generator=g, device="cuda", dtype=D)
    return torch.searchsorted(cdf, u).clamp_(max=V - 1).to(torch.int64)


def _f(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _config(c):
    return GPTConfig.default(VOCAB, c["depth"])


def _period(c):
    """RoPE rows as the driver sets them: the flat token up to its 2048-row table, else per sequence."""
    return 0 if c["B"] * c["T"] <= 2048 else c["T"]


def _train_inputs(c, seed):
    """Token ids and a state some way into training: every tensor non-zero."""
    cfg = _config(c)
    cfg.sequence_len = c["T"]
    g = _gen(seed)
    n = c["B"] * c["T"]
    toks = _zipf(g, n + 1, VOCAB)
    L, C = cfg.n_layer, cfg.n_embd
    shapes = {"wte": (VOCAB, C), "lm_head": (VOCAB, C), "resid_lambdas": (L,), "x0_lambdas": (L,)}
    for i in range(L):
        p = "h%d." % i
        shapes.update({p + "c_q": (C, C), p + "c_k": (C, C), p + "c_v": (C, C), p + "c_proj": (C, C),
                       p + "c_fc": (4 * C, C), p + "mlp_proj": (C, 4 * C)})
        if cfg.has_ve(i):
            shapes.update({p + "value_embeds": (VOCAB, C), p + "ve_gate": (cfg.n_head, GATE)})
    W = {}
    for name, sh in shapes.items():
        s = {"wte": 1.0, "lm_head": 0.1, "resid_lambdas": 0.05, "x0_lambdas": 0.05}.get(name)
        if s is None:
            s = 0.3 if name.endswith("ve_gate") else 0.5 if name.endswith("value_embeds") else \
                0.2 / math.sqrt(C) if name.endswith("proj") else 0.8 / math.sqrt(C)
        W[name] = _randn(g, *sh, scale=s)
    W["resid_lambdas"] += 1.0
    W["x0_lambdas"] += 0.1
    return cfg, W, toks[:-1].contiguous(), toks[1:].contiguous()


def _linear_inputs(c, seed):
    g = _gen(seed)
    M, N, K = c["M"], c["N"], c["K"]
    x, w = _randn(g, M, K), _randn(g, N, K, scale=K ** -0.5)
    dy = _randn(g, M, N, scale=0.01)
    if c["mode"] == "stored":
        x, w, dy = [t.to(torch.bfloat16) for t in (x, w, dy)]
    return x, w, dy


def _attention_inputs(c, seed):
    g = _gen(seed)
    n = c["B"] * c["T"] * c["H"]
    q, k, v, do = [_randn(g, n, c["hd"]) for _ in range(4)]
    for t in (q, k):  # the model normalises q and k per head
        t /= torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5)
    return q, k, v, do.mul_(0.1)


def _rows_inputs(c, seed):
    g = _gen(seed)
    M, C, H, V = c["M"], c["C"], c["H"], c["V"]
    hd = C // H
    ang = torch.arange(M, dtype=D, device="cuda")[:, None] % 2048 / \
        10000.0 ** (torch.arange(0, hd, 2, dtype=D, device="cuda") / hd)
    return dict(idx=_zipf(g, M, V), tgt=_zipf(g, M, V), wte=_randn(g, V, C), ve_w=_randn(g, V, C, scale=0.5),
                xin=_randn(g, M, C), sa=1 + _randn(g, 4, scale=0.05), sb=0.1 + _randn(g, 4, scale=0.05),
                gate_w=_randn(g, H, GATE, scale=0.3), qin=_randn(g, M, C), h=_randn(g, M, 4 * C),
                logits=_randn(g, M, V, scale=3.0), cos=ang.cos().float(), sin=ang.sin().float(),
                gact=_randn(g, M, 4 * C, scale=0.01), gxn=_randn(g, M, C, scale=0.01), gq=_randn(g, M, C, scale=0.01),
                gv=_randn(g, M, C, scale=0.01), res=_randn(g, M, C))


def _optimizer_inputs(c, seed):
    g = _gen(seed)
    C, V = c["C"], c["V"]
    mats = []
    for r, k in ((C, C), (C, C), (C, C), (C, C), (4 * C, C), (C, 4 * C)):
        mats.append((_randn(g, r, k, scale=0.8 / math.sqrt(k)), _randn(g, r, k, scale=0.02), _randn(g, r, k, scale=0.02)))
    emb = (_randn(g, V, C), _randn(g, V, C, scale=0.01), _randn(g, V, C, scale=0.01),
           _randn(g, V, C, scale=0.01).square_().add_(1e-6))
    return mats, emb


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "train":
        cfg, W, x, y = _train_inputs(c, seed)
        m = GPT(cfg, c["B"], c["T"], precision=BF16 if c["precision"] == "bf16" else FP32, rope_period=_period(c))
        m.init_weights(42)
        p = m.params()
        for name, off, size in m.tensors():
            p[off:off + size] = W[name].reshape(-1)
        out = (m.token_loss(), m.grads(), p)
        for t in out:  # views of the model's own memory: a result keeps its model alive
            t.model = m
        return {"c": c, "m": m, "x": x, "y": y, "out": out}
    _workspace()
    if kind == "linear":
        x, w, dy = _linear_inputs(c, seed)
        t = torch.bfloat16 if c["mode"] == "stored" else torch.float32
        y = torch.empty(c["M"], c["N"], dtype=t, device="cuda")
        dx = torch.empty(c["M"], c["K"], dtype=t, device="cuda")
        return {"c": c, "x": x, "w": w, "dy": dy, "y": y, "dx": dx, "dw": _f(c["N"], c["K"]), "lib": _lib.load()}
    if kind == "attention":
        q, k, v, do = _attention_inputs(c, seed)
        n = q.shape[0]
        return {"c": c, "q": q, "k": k, "v": v, "do": do, "o": torch.empty_like(q), "lse": _f(n), "d": _f(n),
                "dq": torch.empty_like(q), "dk": torch.empty_like(q), "dv": torch.empty_like(q)}
    if kind == "rows":
        s = _rows_inputs(c, seed)
        M, C, H, V = c["M"], c["C"], c["H"], c["V"]
        s.update(c=c, e=_f(M, C), rms0=_f(M), x0=_f(M, C), x=_f(M, C), xn=_f(M, C), rms=_f(M), gate=_f(M, H),
                 ve=_f(M, C), q=_f(M, C), qn=_f(M, C), rmsq=_f(M * H), act=_f(M, 4 * C), xr=_f(M, C),
                 capped=_f(M, V), loss=_f(M), mean=_f(1), glogits=_f(M, V), gh=_f(M, 4 * C), gx=_f(M, C),
                 gqin=_f(M, C), gve=_f(M, C), ggate=_f(M, H), ggw=_f(H, GATE), gsc=_f(4), gwte=_f(V, C))
        return s
    mats, emb = _optimizer_inputs(c, seed)
    return {"c": c, "mats": mats, "emb": emb}


# ---------------------------------------------------------------- one pass

def _gemm_mixed(lib, layout, C, X, W, M, N, K, accumulate):
    # the bf16-storage product of the C interface
    _lib.check(lib.ar_gemm_mixed(torch.cuda.current_stream().cuda_stream, layout, C.data_ptr(),
                                 int(C.dtype == torch.bfloat16), X.data_ptr(), 1, W.data_ptr(), 1, M, N, K,
                                 accumulate), "gemm_mixed")


def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "train":
        # near the end of the schedule: the whole optimizer runs and the weights stay close to where they were
        s["m"].train_step(s["x"], s["y"], progress=0.999, sync_loss=False)
        return dict(zip(("token_loss", "grads", "params"), s["out"]))
    if kind == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        if c["mode"] == "stored":
            _gemm_mixed(s["lib"], 0, s["y"], s["x"], s["w"], M, N, K, 0)
            _gemm_mixed(s["lib"], 1, s["dx"], s["dy"], s["w"], M, N, K, 0)
            _gemm_mixed(s["lib"], 2, s["dw"], s["dy"], s["x"], M, N, K, 0)
        else:
            bf = c["mode"] == "bf16"
            ops.linear_fwd(s["y"], s["x"], s["w"], M, N, K, bf16=bf)
            ops.linear_bwd_dx(s["dx"], s["dy"], s["w"], M, N, K, bf16=bf)
            ops.zero_buffer(s["dw"], N * K)  # the weight gradient accumulates
            ops.linear_bwd_dw(s["dw"], s["dy"], s["x"], M, N, K, bf16=bf)
        return {"y": s["y"], "dx": s["dx"], "dw": s["dw"]}
    if kind == "attention":
        a = (c["B"], c["T"], c["H"], c["hd"])
        w, bf = c["window"], c["precision"] == "bf16"
        ops.flash_attn_fwd(s["o"], s["lse"], s["q"], s["k"], s["v"], *a, w, bf16=bf)
        ops.flash_attn_bwd_precompute_d(s["d"], s["o"], s["do"], *a, bf16=bf)
        ops.flash_attn_bwd_dq(s["dq"], s["q"], s["k"], s["v"], s["do"], s["lse"], s["d"], *a, w, bf16=bf)
        ops.flash_attn_bwd_dkv(s["dk"], s["dv"], s["q"], s["k"], s["v"], s["do"], s["lse"], s["d"], *a, w, bf16=bf)
        return {n: s[n] for n in ("o", "lse", "d", "dq", "dk", "dv")}
    if kind == "rows":
        M, C, H, V = c["M"], c["C"], c["H"], c["V"]
        hd = C // H
        ops.embedding_fwd(s["e"], s["wte"], s["idx"], M, C)
        ops.rmsnorm_fwd(s["x0"], s["rms0"], s["e"], M, C)
        ops.scaled_add_fwd(s["x"], s["xin"], s["x0"], s["sa"], s["sb"], 2, M * C)
        ops.rmsnorm_fwd(s["xn"], s["rms"], s["x"], M, C)
        ops.embedding_fwd(s["ve"], s["ve_w"], s["idx"], M, C)
        ops.ve_gate_fwd(s["gate"], s["xn"], s["gate_w"], M, H, GATE, C)
        ops.rope_fwd(s["q"], s["qin"], s["cos"], s["sin"], M, H, hd)
        ops.rmsnorm_fwd(s["qn"], s["rmsq"], s["q"], M * H, hd)
        ops.relu_squared_fwd(s["act"], s["h"], M * 4 * C)
        ops.add_residual_fwd(s["xr"], s["x"], s["res"], M * C)
        ops.softcap_fwd(s["capped"], s["logits"], CAP, M * V)
        ops.cross_entropy_fwd(s["loss"], s["capped"], s["tgt"], M, V)
        ops.mean_reduce(s["mean"], s["loss"], M)
        ops.cross_entropy_softcap_bwd(s["glogits"], s["capped"], s["tgt"], CAP, M, V, 1.0)
        ops.relu_squared_bwd(s["gh"], s["gact"], s["h"], M * 4 * C)
        ops.rmsnorm_bwd(s["gx"], s["gxn"], s["x"], s["rms"], M, C)
        ops.rope_bwd(s["gqin"], s["gq"], s["cos"], s["sin"], M, H, hd)
        ops.ve_apply_bwd(s["gve"], s["ggate"], s["gv"], s["gate"], s["ve"], M, H, hd)
        for n in ("ggw", "gsc", "gwte"):  # these accumulate
            ops.zero_buffer(s[n], s[n].numel())
        ops.ve_gate_bwd(s["gx"], s["ggw"], s["ggate"], s["gate"], s["xn"], s["gate_w"], M, H, GATE, C)
        ops.scalar_grad_reduce(s["gsc"], s["gx"], s["x"], 2, M * C)
        ops.embedding_bwd(s["gwte"], s["gx"], s["idx"], M, C)
        return {n: s[n] for n in ROWS_OUT}
    for p, g, b in s["mats"]:
        ops.muon_step(p, g, b, p.shape[0], p.shape[1], 0.02, 0.5, 0.95, 0.1, bf16=c["precision"] == "bf16")
    p, g, m, v = s["emb"]
    ops.adamw_step_group(p, g, m, v, p.numel(), 0.3, 0.8, 0.95, 1e-10, 0.0, 0.1, 100)
    return {"params": [x[0] for x in s["mats"]], "momenta": [x[2] for x in s["mats"]], "emb": [p, m, v]}


ROWS_OUT = ("x0", "xn", "rms", "gate", "qn", "act", "xr", "capped", "loss", "mean", "glogits", "gh", "gx", "gqin",
            "gve", "ggate", "ggw", "gsc", "gwte")


# ---------------------------------------------------------------- work

def _keys(T, window):
    """Visible (query, key) pairs of one head."""
    if window <= 0 or window >= T:
        return T * (T + 1) / 2
    return (window + 1) * T - window * (window + 1) / 2


def work(case):
    c, kind = case, case["kind"]
    if kind == "train":
        cfg = _config(c)
        cfg.sequence_len = c["T"]
        L, C, M = cfg.n_layer, cfg.n_embd, c["B"] * c["T"]
        fl = 72.0 * L * M * C * C + 6.0 * M * C * VOCAB
        for i in range(L):
            fl += 14.0 * c["B"] * C * _keys(c["T"], cfg.window_size(i))
        fl += 5.0 * L * (4 * (4 * C ** 3 + 2 * C ** 3) + 2 * (16 * C ** 3 + 2 * C ** 3))
        n = 12.0 * L * C * C + 2 * VOCAB * C + sum(VOCAB * C for i in range(L) if cfg.has_ve(i))
        # weights, gradients and two moments (one for Muon's) read and written; tokens and losses
        return {"bytes": 4.0 * n * 7 + 20.0 * M, "flops": fl}
    if kind == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        e = 2.0 if c["mode"] == "stored" else 4.0
        return {"bytes": 2 * e * (M * K + M * N) + e * N * K + 4.0 * N * K, "flops": 6.0 * M * N * K}
    if kind == "attention":
        n = c["B"] * c["T"] * c["H"]
        fl = 14.0 * c["B"] * c["H"] * c["hd"] * _keys(c["T"], c["window"])
        return {"bytes": 4.0 * n * (8 * c["hd"] + 2), "flops": fl}
    if kind == "rows":
        M, C, H, V = c["M"], c["C"], c["H"], c["V"]
        values = 3.0 * M * V + 14.0 * M * C + 16.0 * M * C + M * C + 3.0 * V * C + M * (8 + 2 * H)
        return {"bytes": 4.0 * values, "flops": 10.0 * M * (V + C)}
    C, V = c["C"], c["V"]
    return {"bytes": 4.0 * (12 * C * C * 5 + 7 * V * C), "flops": 5.0 * (4 * 6 * C ** 3 + 2 * 18 * C ** 3)}


def tolerance(case):
    """About four times what the library shows against exact(), or against itself
    with its fused kernels off (training, bf16): gradients 2.4e-3 and 9e-4 there."""
    c = case
    bf = c.get("precision") == "bf16" or c.get("mode") in ("bf16", "stored")
    if c["kind"] == "train":
        # AdamW's early steps are close to sign(g): a gradient entry near zero moves its weight by up to 2 lr
        return {"rel": 1e-2} if bf else {"rel": 1e-5, "max": 0.05}
    if c["kind"] == "linear":
        return {"rel": 1e-2 if bf else 1e-5}
    if c["kind"] == "attention":
        return {"rel": 1.6e-2 if bf else 1e-5}
    if c["kind"] == "rows":
        return {"rel": 1e-5}
    # Muon's cautious decay takes one of two branches where the update is near zero
    return {"rel": 2e-3} if bf else {"rel": 1e-5, "max": 0.01}


# ---------------------------------------------------------------- the same in 64 bits

def _rms(x):
    return torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)


def _mask(T, window):
    i = torch.arange(T, device="cuda")
    ok = i[None, :] <= i[:, None]
    if window > 0:
        ok &= i[None, :] >= i[:, None] - window
    return ok


def _attention_rows(q, k, v, do, ok, scale):
    """Heads of one sequence [H, T, hd] in 64 bits: o, lse and, with do, d, dq, dk, dv."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    s.masked_fill_(~ok, -math.inf)
    lse = torch.logsumexp(s, -1)
    p = s.sub_(lse[..., None]).exp_()
    o = torch.matmul(p, v)
    if do is None:
        return o, lse
    d = (o * do).sum(-1)
    ds = torch.matmul(do, v.transpose(1, 2).contiguous()).sub_(d[..., None]).mul_(p).mul_(scale)
    return (o, lse, d, torch.matmul(ds, k), torch.matmul(ds.transpose(1, 2).contiguous(), q),
            torch.matmul(p.transpose(1, 2).contiguous(), do))


def _exact_attention(q, k, v, do, B, T, H, hd, window):
    """q, k, v, do: [B T H, hd]; every output laid out the same."""
    ok, scale = _mask(T, window), hd ** -0.5
    got = []
    for b in range(B):
        heads = [None if t is None else t.view(B, T, H, hd)[b].to(D).transpose(0, 1).contiguous()
                 for t in (q, k, v, do)]
        got.append([x.transpose(0, 1).reshape(T * H, -1) for x in _attention_rows(*heads, ok, scale)])
    out = [torch.cat(x) for x in zip(*got)]
    return [x if x.shape[1] == hd and i != 1 and i != 2 else x.reshape(-1) for i, x in enumerate(out)]


class _Attention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, dims):
        ctx.save_for_backward(q, k, v)
        ctx.dims = dims
        return _exact_attention(q, k, v, None, *dims)[0]

    @staticmethod
    def backward(ctx, g):
        q, k, v = ctx.saved_tensors
        return (*_exact_attention(q, k, v, g.contiguous(), *ctx.dims)[3:], None)


class _ScaledAdd(torch.autograd.Function):
    """x = a[i] x_in + b[i] x0; the gradients of the scalars take the scaled x,
    and the value that reaches x0 this way goes no further (the model's own rules)."""
    @staticmethod
    def forward(ctx, x, x0, sa, sb, i):
        out = sa[i] * x + sb[i] * x0
        ctx.save_for_backward(out, x0, sa)
        ctx.i = i
        return out

    @staticmethod
    def backward(ctx, g):
        out, x0, sa = ctx.saved_tensors
        ga, gb = torch.zeros_like(sa), torch.zeros_like(sa)
        ga[ctx.i] = (g * out).sum()
        gb[ctx.i] = (g * x0).sum()
        return sa[ctx.i] * g, None, ga, gb, None


class _MlpNorm(torch.autograd.Function):
    """The MLP's norm, whose backward takes the layer's input x in place of the mid-layer one."""
    @staticmethod
    def forward(ctx, x, x_saved):
        r = _rms(x)
        ctx.save_for_backward(x_saved, r)
        return x / r

    @staticmethod
    def backward(ctx, g):
        x, r = ctx.saved_tensors
        return (g - x * (g * x).sum(-1, keepdim=True) / (x.shape[-1] * r * r)) / r, None


def _through(x, y):
    """y forward, the gradient of x itself backward."""
    return x + (y - x).detach()


def _turn(x, cos, sin):
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos + b * sin, b * cos - a * sin], -1)


def _exact_train(c, seed):
    cfg, W, ids, tgt = _train_inputs(c, seed)
    B, T, L, C, H = c["B"], c["T"], cfg.n_layer, cfg.n_embd, cfg.n_head
    hd, n = C // H, c["B"] * c["T"]
    P = {k: t.to(D).requires_grad_() for k, t in W.items()}
    pos = torch.arange(n, dtype=D, device="cuda") % (_period(c) or n)
    ang = (pos[:, None] / 10000.0 ** (torch.arange(0, hd, 2, dtype=D, device="cuda") / hd))[:, None, :]
    cos, sin = ang.cos().float().to(D), ang.sin().float().to(D)
    e = P["wte"][ids]
    x0 = _through(e, e / _rms(e))
    x = x0
    for i in range(L):
        p = "h%d." % i
        x = _ScaledAdd.apply(x, x0.detach(), P["resid_lambdas"], P["x0_lambdas"], i)
        top, xn = x, x / _rms(x)
        q, k, v = [(xn @ P[p + w].T).view(n, H, hd) for w in ("c_q", "c_k", "c_v")]
        if cfg.has_ve(i):
            gate = 2.0 * torch.sigmoid(xn[:, :GATE] @ P[p + "ve_gate"].T)
            v = v + gate[:, :, None] * P[p + "value_embeds"][ids].view(n, H, hd)
        q, k = [_turn(t, cos, sin) for t in (q, k)]
        q, k = [_through(t, t / _rms(t)).reshape(n * H, hd) for t in (q, k)]
        a = _Attention.apply(q, k, v.reshape(n * H, hd), (B, T, H, hd, cfg.window_size(i)))
        x = x + a.view(n, C) @ P[p + "c_proj"].T
        x = x + torch.relu(_MlpNorm.apply(x, top) @ P[p + "c_fc"].T) ** 2 @ P[p + "mlp_proj"].T
    z = (x / _rms(x)) @ P["lm_head"].T
    z = _through(z, CAP * torch.tanh(z / CAP))
    loss = torch.logsumexp(z, -1) - z.gather(1, tgt[:, None])[:, 0]
    loss.sum().backward()
    # the gradient arena: tensors in registration order, each padded to 64 values
    flat = []
    for name in W:
        gt = P[name].grad.reshape(-1)
        flat += [gt, gt.new_zeros(-gt.numel() % 64)]
    return {"token_loss": loss.detach(), "grads": torch.cat(flat), "params": None}


def _exact_rows(c, seed):
    s = _rows_inputs(c, seed)
    M, C, H = c["M"], c["C"], c["H"]
    hd, idx, tgt = C // H, s.pop("idx"), s.pop("tgt")
    s = {k: t.to(D) for k, t in s.items()}
    o = {}
    e = s["wte"][idx]
    o["x0"] = e / _rms(e)
    x = s["sa"][2] * s["xin"] + s["sb"][2] * o["x0"]
    r = _rms(x)
    o["xn"], o["rms"] = x / r, r[:, 0]
    ve = s["ve_w"][idx].view(M, H, hd)
    o["gate"] = 2.0 * torch.sigmoid(o["xn"][:, :GATE] @ s["gate_w"].T)
    cos, sin = s["cos"][:, None, :], s["sin"][:, None, :]
    q = _turn(s["qin"].view(M, H, hd), cos, sin)
    o["qn"] = (q / _rms(q)).view(M, C)
    o["act"] = torch.relu(s["h"]) ** 2
    o["xr"] = x + s["res"]
    o["capped"] = CAP * torch.tanh(s["logits"] / CAP)
    lse = torch.logsumexp(o["capped"], -1, keepdim=True)
    o["loss"] = (lse - o["capped"].gather(1, tgt[:, None]))[:, 0]
    o["mean"] = o["loss"].mean().reshape(1)
    o["glogits"] = (o["capped"] - lse).exp()
    o["glogits"][torch.arange(M, device="cuda"), tgt] -= 1.0
    o["gh"] = 2.0 * torch.relu(s["h"]) * s["gact"]
    gx = (s["gxn"] - x * (s["gxn"] * x).sum(-1, keepdim=True) / (C * r * r)) / r
    o["gqin"] = _turn(s["gq"].view(M, H, hd), cos, -sin).reshape(M, C)
    gv = s["gv"].view(M, H, hd)
    o["gve"] = (o["gate"][:, :, None] * gv).view(M, C)
    o["ggate"] = (ve * gv).sum(-1)
    dz = o["ggate"] * o["gate"] * (1.0 - o["gate"] / 2.0)
    o["ggw"] = dz.T @ o["xn"][:, :GATE]
    gx[:, :GATE] += dz @ s["gate_w"]
    o["gx"] = gx
    o["gsc"] = torch.zeros(4, dtype=D, device="cuda")
    o["gsc"][2] = (gx * x).sum()
    o["gwte"] = torch.zeros_like(s["wte"]).index_add_(0, idx, gx)
    return {n: o[n] for n in ROWS_OUT}


def _exact_optimizer(c, seed):
    mats, emb = _optimizer_inputs(c, seed)
    ps, bs = [], []
    for p, g, b in mats:
        p, g, b = p.to(D), g.to(D), b.to(D)
        b = 0.95 * b + 0.05 * g
        x = 0.05 * g + 0.95 * b
        x /= x.norm() * 1.02 + 1e-6
        tall = p.shape[0] >= p.shape[1]
        for a, bb, cc in POLAR:
            xt = x.T.contiguous()
            A = xt @ x if tall else x @ xt
            B = bb * A + cc * (A @ A)
            x = a * x + (x @ B if tall else B @ x)
        lr = 0.02 * 0.5 * math.sqrt(max(1.0, p.shape[0] / p.shape[1]))
        ps.append(p - lr * (x + 0.1 * p * (x * p >= 0)))
        bs.append(b)
    p, g, m, v = [t.to(D) for t in emb]
    m = 0.8 * m + 0.2 * g
    v = 0.95 * v + 0.05 * g * g
    p = p - 0.3 * 0.1 * (m / (1 - 0.8 ** 100)) / (torch.sqrt(v / (1 - 0.95 ** 100)) + 1e-10)
    return {"params": ps, "momenta": bs, "emb": [p, m, v]}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "train":
        return _exact_train(c, seed)
    if kind == "linear":
        x, w, dy = [t.to(D) for t in _linear_inputs(c, seed)]
        return {"y": x @ w.T, "dx": dy @ w, "dw": dy.T @ x}
    if kind == "attention":
        q, k, v, do = _attention_inputs(c, seed)
        o = _exact_attention(q, k, v, do, c["B"], c["T"], c["H"], c["hd"], c["window"])
        return dict(zip(("o", "lse", "d", "dq", "dk", "dv"), o))
    if kind == "rows":
        return _exact_rows(c, seed)
    return _exact_optimizer(c, seed)
