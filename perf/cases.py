"""Performance cases of the GDN library: the calls that a serving program makes, through the
package's public entry points, over the sizes it makes them at.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the inputs, weights, states and workspaces a program holds before the call
    run(state)          one pass; returns every output and every state the call updates
    work(case)          bytes and operations that one pass cannot do without
    tolerance(case)     how far another correct implementation's results may be
    exact(case, seed)   run's results in 64-bit arithmetic, from plain torch and numpy

A case is a dict of plain values. "kind" picks the path:

    legacy    one token through the five drop-in launchers (conv, L2 norms, beta, step, norm)
    decode    one token for B sequences of a layer, with or without the gated output norm
    window    verify K drafted tokens for B sequences, then commit the accepted prefixes
    in_proj   the layer's input projection for B token rows (decode batches and prompts)
    gemv      the single-token bf16 projection pair
    q8_0      activations quantised to q8_1, then the Q8_0 product for ncols columns
    prefill   packed prompts, with or without the gated output norm
"""
import math
import random

import numpy as np
import torch

import baloon_amd as bx

D = 128                       # head dimension of the fused kernels
LN16 = math.log(16.0)


# ---------------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------------
# Layer options: "plain" is the reference's semantics (modulo head pairing, no activation after
# the conv, unscaled queries); "next" is the Qwen3-Next layer (contiguous head groups, SiLU after
# the conv, queries scaled by 1/sqrt(128)).

def listed():
    return [
        # One token of one sequence through the drop-in launchers, at the reference test's shape:
        # a host program that swapped the library in and calls it operator by operator.
        dict(name="legacy_token", kind="legacy", h_k=16, h_v=48, S=128, d_conv=4),
        # A single interactive user: one token, one sequence. Latency and launches.
        dict(name="decode_1", kind="decode", B=1, h_k=16, h_v=32, opts="plain", gated=False),
        # The serving batch: 64 sequences, one token each.
        dict(name="decode_64", kind="decode", B=64, h_k=16, h_v=32, opts="plain", gated=False),
        # A batch as it stands between arrivals and departures, with the layer's output norm
        # fused in and bf16 activations out.
        dict(name="decode_gated_37", kind="decode", B=37, h_k=16, h_v=32, opts="next", gated=True),
        # Speculative decoding: four drafted tokens per sequence verified on the matrix cores, then
        # a part of them committed.
        dict(name="window_64x4", kind="window", B=64, K=4, h_k=16, h_v=32, opts="plain"),
        # The projection ahead of a decode step: 64 rows against all the weights.
        dict(name="in_proj_64", kind="in_proj", B=64, hidden=2048, h_k=16, h_v=32),
        # The projection ahead of a prefill: a 4,096-token prompt.
        dict(name="in_proj_4096", kind="in_proj", B=4096, hidden=2048, h_k=16, h_v=32),
        # A single user's projection as two matrix-vector products sharing the activations
        # (mixed q|k|v channels, then the gate logits).
        dict(name="gemv_pair", kind="gemv", n_in=2560, n_out1=8192, n_out2=4096),
        # A quantised model's projection for a small batch: activations to q8_1, then Q8_0 weights.
        dict(name="q8_0_4", kind="q8_0", n_in=4096, n_out=6144, ncols=4),
        # A short question: one prompt of a few hundred tokens, output norm fused.
        dict(name="prefill_300", kind="prefill", n_seq=1, T=300, h_k=16, h_v=32, opts="next", gated=True),
        # One long prompt.
        dict(name="prefill_4096", kind="prefill", n_seq=1, T=4096, h_k=16, h_v=32, opts="plain", gated=False),
        # A prefill batch: 32 prompts of 1 to 2,048 tokens, packed, output norm fused.
        dict(name="prefill_varlen_32", kind="prefill", n_seq=32, lo=1, hi=2048, lens_seed=4, h_k=16, h_v=32,
             opts="next", gated=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    # Head layouts: the Qwen3-Next layer, the reference test's, and tensor-parallel shares of them.
    h_k, h_v = rng.choice([(16, 32), (16, 32), (16, 48), (16, 16), (8, 16), (4, 8)])
    opts = rng.choice(["plain", "next"])
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "window", "window", "in_proj",
                       "in_proj", "gemv", "q8_0", "legacy"])
    if kind == "legacy":
        return dict(kind=kind, h_k=h_k, h_v=h_v, S=rng.choice([128, 128, 64, 96]), d_conv=rng.choice([4, 4, 3, 2]))
    if kind == "decode":
        return dict(kind=kind, B=_log_int(rng, 1, 256), h_k=h_k, h_v=h_v, opts=opts, gated=rng.random() < 0.5)
    if kind == "window":
        return dict(kind=kind, B=_log_int(rng, 1, 64), K=rng.randint(2, 8), h_k=h_k, h_v=h_v, opts=opts)
    if kind == "in_proj":
        if h_v > 32:
            h_v = 32
        return dict(kind=kind, B=_log_int(rng, 1, 4096), hidden=rng.choice([1024, 1536, 2048]), h_k=h_k, h_v=h_v)
    if kind == "gemv":
        return dict(kind=kind, n_in=8 * _log_int(rng, 64, 640), n_out1=_log_int(rng, 64, 8192),
                    n_out2=_log_int(rng, 64, 8192))
    if kind == "q8_0":
        return dict(kind=kind, n_in=32 * _log_int(rng, 16, 128), n_out=_log_int(rng, 512, 12352),
                    ncols=rng.randint(1, 8))
    # prefill: one prompt, or a batch of them
    gated = rng.random() < 0.5
    if rng.random() < 0.5:
        return dict(kind=kind, n_seq=1, T=_log_int(rng, 2, 8192), h_k=h_k, h_v=h_v, opts=opts, gated=gated)
    return dict(kind=kind, n_seq=rng.randint(2, 16), lo=1, hi=_log_int(rng, 64, 2048),
                lens_seed=rng.randrange(1 << 16), h_k=h_k, h_v=h_v, opts=opts, gated=gated)


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------

def _cfg(case):
    o = case["opts"]
    if o == "next":
        return bx.make_cfg(h_k=case["h_k"], h_v=case["h_v"], head_map=bx.HEAD_DIV, conv_act=bx.ACT_SILU,
                           q_scale=D ** -0.5)
    return bx.make_cfg(h_k=case["h_k"], h_v=case["h_v"])


def _lens(case):
    if case["n_seq"] == 1:
        return [case["T"]]
    r = random.Random(case["lens_seed"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["n_seq"])]


class _Gen:
    """Seeded normal and uniform tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        t = torch.empty(*shape, dtype=dtype, device="cuda")
        return t.normal_(0.0, std, generator=self.g)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.empty(*shape, dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=self.g)

    def integers(self, lo, hi, *shape, dtype=torch.int32):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=dtype)


def _layer_inputs(case, seed, n, rows):
    """Layer parameters, the states of n sequences and the inputs of the token rows."""
    g = _Gen(seed)
    hk, hv = case["h_k"], case["h_v"]
    C = (2 * hk + hv) * D
    return dict(
        conv_w=g.normal(C, 4, std=0.1), A_log=g.uniform(hv, hi=LN16), dt_bias=g.normal(hv, std=0.1, dtype=torch.float32),
        ssm_norm=1.0 + g.normal(D, std=0.1, dtype=torch.float32),
        state=g.normal(n, hv, D, D, std=0.02, dtype=torch.float32), conv_state=g.normal(n, C, 3),
        x=g.normal(*rows, C), a=g.normal(*rows, hv), b=g.normal(*rows, hv),
        z=g.normal(*rows, hv, D) if case.get("gated") else None, gen=g)


def _legacy_inputs(case, seed):
    g = _Gen(seed)
    hk, hv, S, dc = case["h_k"], case["h_v"], case["S"], case["d_conv"]
    C = (2 * hk + hv) * S
    f32 = torch.float32
    return dict(conv_state=g.normal(C, dc - 1, dtype=f32), x=g.normal(C, dtype=f32), kW=g.normal(C, dc, std=0.1, dtype=f32),
                beta=g.normal(hv, dtype=f32), gate=-g.uniform(hv, lo=0.01, hi=2.0),
                state=g.normal(S, hv, S, std=0.02, dtype=f32), z=g.normal(hv, S, dtype=f32),
                ssm_norm=1.0 + g.normal(S, std=0.1, dtype=f32))


def _in_proj_inputs(case, seed):
    g = _Gen(seed)
    N = (2 * case["h_k"] + 2 * case["h_v"]) * D + 2 * case["h_v"]
    return dict(h=g.normal(case["B"], case["hidden"]), w=g.normal(N, case["hidden"], std=0.05))


def _gemv_inputs(case, seed):
    g = _Gen(seed)
    n = case["n_in"]
    return dict(x=g.normal(n), w1=g.normal(case["n_out1"], n, std=0.05), w2=g.normal(case["n_out2"], n, std=0.05))


def _q8_inputs(case, seed):
    g = _Gen(seed)
    nb, n_out = case["n_in"] // 32, case["n_out"]
    qs = g.integers(-127, 128, n_out, nb, 32, dtype=torch.int8)
    d = (0.05 / 127.0 * g.uniform(n_out, nb, lo=0.5, hi=2.0)).to(torch.float16)
    w = torch.empty(n_out, nb, 34, dtype=torch.uint8, device="cuda")      # blocks: fp16 scale, 32 codes
    w[..., :2] = d.unsqueeze(-1).view(torch.uint8)
    w[..., 2:] = qs.view(torch.uint8)
    return dict(x=g.normal(case["ncols"], case["n_in"], dtype=torch.float32), w=w)


# ---------------------------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------------------------

def _layer(case, d, n):
    layer = bx.GdnLayer(n, _cfg(case))
    layer.conv_w, layer.A_log, layer.dt_bias, layer.ssm_norm = d["conv_w"], d["A_log"], d["dt_bias"], d["ssm_norm"]
    layer.state, layer.conv_state = d["state"], d["conv_state"]
    return layer


def prepare(case, seed):
    kind = case["kind"]
    out = dict(case=case)
    if kind == "legacy":
        d = _legacy_inputs(case, seed)
        out.update(d, conv=torch.empty_like(d["x"]), o=torch.empty(case["h_v"], case["S"], device="cuda"),
                   y=torch.empty(case["h_v"], case["S"], device="cuda"))
    elif kind == "decode":
        B, hv = case["B"], case["h_v"]
        d = _layer_inputs(case, seed, B, (B,))
        out.update(layer=_layer(case, d, B), x=d["x"], a=d["a"], b=d["b"], z=d["z"],
                   o=torch.empty(B, hv, D, dtype=torch.bfloat16, device="cuda"))
    elif kind == "window":
        B, K, hv = case["B"], case["K"], case["h_v"]
        d = _layer_inputs(case, seed, B, (B, K))
        cfg = _cfg(case)
        out.update(d, cfg=cfg, accepted=d["gen"].integers(0, K + 1, B),
                   o=torch.empty(B, K, hv, D, device="cuda"),
                   record=torch.empty(bx.ix_gdn_window_record_size(cfg, B, K), dtype=torch.uint8, device="cuda"))
    elif kind == "in_proj":
        B, hv, C = case["B"], case["h_v"], (2 * case["h_k"] + case["h_v"]) * D
        bf = dict(dtype=torch.bfloat16, device="cuda")
        out.update(_in_proj_inputs(case, seed), cfg=bx.make_cfg(h_k=case["h_k"], h_v=hv), x=torch.empty(B, C, **bf),
                   z=torch.empty(B, hv, D, **bf), a=torch.empty(B, hv, **bf), b=torch.empty(B, hv, **bf))
    elif kind == "gemv":
        out.update(_gemv_inputs(case, seed), y1=torch.empty(case["n_out1"], device="cuda"),
                   y2=torch.empty(case["n_out2"], device="cuda"))
    elif kind == "q8_0":
        n = case["ncols"] * case["n_in"]
        out.update(_q8_inputs(case, seed), xq=torch.empty(n // 32 * 36, dtype=torch.uint8, device="cuda"),
                   y=torch.empty(case["ncols"], case["n_out"], device="cuda"))
    else:
        lens = _lens(case)
        T, n, hv = sum(lens), case["n_seq"], case["h_v"]
        d = _layer_inputs(case, seed, n, (T,))
        cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32).cuda()
        if case["gated"]:
            o = torch.empty(T, hv, D, dtype=torch.bfloat16, device="cuda")
        else:
            o = torch.empty(T, hv, D, device="cuda")
        out.update(layer=_layer(case, d, n), cu=cu, x=d["x"], a=d["a"], b=d["b"], z=d["z"], o=o)
    return out


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode":
        layer = st["layer"]
        if case["gated"]:
            layer.decode(st["x"], st["a"], st["b"], z=st["z"], y_bf16=st["o"])
        else:
            layer.decode(st["x"], st["a"], st["b"], o_bf16=st["o"])
        return dict(o=st["o"], state=layer.state, conv_state=layer.conv_state)
    if kind == "prefill":
        layer = st["layer"]
        if case["gated"]:
            layer.prefill(st["cu"], st["x"], st["a"], st["b"], z=st["z"], y_bf16=st["o"])
        else:
            layer.prefill(st["cu"], st["x"], st["a"], st["b"], o=st["o"])
        return dict(o=st["o"], state=layer.state, conv_state=layer.conv_state)
    if kind == "window":
        cfg, B, K = st["cfg"], case["B"], case["K"]
        bx.check("verify", bx.ix_gdn_decode_window_mfma(cfg, B, K, st["x"], st["conv_state"], st["conv_w"], st["a"],
                                                        st["b"], st["A_log"], st["dt_bias"], st["state"], st["o"],
                                                        None, st["record"]))
        bx.check("commit", bx.ix_gdn_commit_window(cfg, B, K, st["accepted"], st["x"], st["record"],
                                                   st["conv_state"], st["state"]))
        return dict(o=st["o"], state=st["state"], conv_state=st["conv_state"])
    if kind == "in_proj":
        bx.check("in_proj", bx.ix_gdn_in_proj(st["cfg"], case["B"], case["hidden"], st["h"], st["w"], st["x"], st["z"],
                                              st["a"], st["b"]))
        return dict(x=st["x"], z=st["z"], a=st["a"], b=st["b"])
    if kind == "gemv":
        bx.check("gemv", bx.ix_bf16_gemv_pair(st["x"], st["w1"], st["y1"], case["n_out1"], st["w2"], st["y2"],
                                              case["n_out2"], case["n_in"]))
        return dict(y1=st["y1"], y2=st["y2"])
    if kind == "q8_0":
        n_in, ncols = case["n_in"], case["ncols"]
        bx.check("quantize", bx.ix_q8_1_quantize(st["x"], st["xq"], ncols * n_in))
        bx.check("q8_0", bx.ix_mmvq_q8_0(st["w"], st["xq"], st["y"], n_in, case["n_out"], ncols))
        return dict(y=st["y"], xq=st["xq"])
    hk, hv, S, dc = case["h_k"], case["h_v"], case["S"], case["d_conv"]
    conv = st["conv"]
    q, k, v = conv[:hk * S], conv[hk * S:2 * hk * S], conv[2 * hk * S:]
    bx.check("conv", bx.ix_gdn_conv_step(st["conv_state"], st["x"], st["kW"], conv, conv.numel(), dc))
    bx.check("l2", bx.ix_gdn_l2_norm(conv, 2 * hk, S, 1e-6))               # q rows, then k rows
    bx.check("beta", bx.ix_gdn_beta_gate(st["beta"], hv))
    bx.check("step", bx.ix_gdn_step(st["state"], q, k, v, st["gate"], st["beta"], st["o"], S, hk, hv))
    bx.check("norm", bx.ix_gdn_out_norm(st["o"], st["z"], st["ssm_norm"], st["y"], hv, S, 1e-6))
    return dict(y=st["y"], state=st["state"], conv_state=st["conv_state"], beta=st["beta"])


# ---------------------------------------------------------------------------------------------
# Costs and tolerances
# ---------------------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "legacy":
        hk, hv, S, dc = case["h_k"], case["h_v"], case["S"], case["d_conv"]
        C = (2 * hk + hv) * S
        return dict(bytes=4 * (2 * hv * S * S + C * (dc + 2 * (dc - 1) + 1) + 2 * hv * S + S + 3 * hv),
                    flops=6 * hv * S * S + 2 * C * dc)
    if kind == "in_proj":
        N = (2 * case["h_k"] + 2 * case["h_v"]) * D + 2 * case["h_v"]
        B, K = case["B"], case["hidden"]
        return dict(bytes=2 * (B * K + N * K + B * N), flops=2 * B * N * K)
    if kind == "gemv":
        n, m = case["n_in"], case["n_out1"] + case["n_out2"]
        return dict(bytes=2 * n + 2 * n * m + 4 * m, flops=2 * n * m)
    if kind == "q8_0":
        n, m, c = case["n_in"], case["n_out"], case["ncols"]
        return dict(bytes=n // 32 * 34 * m + 4 * c * n + n // 32 * 36 * c + 4 * c * m, flops=2 * n * m * c)
    hk, hv = case["h_k"], case["h_v"]
    C = (2 * hk + hv) * D
    params = 8 * C + 8 * hv
    state, conv = 4 * hv * D * D, 6 * C                                    # one sequence's
    row = 2 * C + 4 * hv                                                   # one token's x, a, b
    per_token = 6 * hv * D * D + 8 * C                                     # S^T k, S^T q, rank-1 update; conv
    if kind == "decode":
        B = case["B"]
        out = hv * D * (4 if case["gated"] else 2)                         # bf16 out (and z in)
        return dict(bytes=params + B * (2 * state + 2 * conv + row + out), flops=B * per_token)
    if kind == "window":
        # verify: states in, outputs out; commit: states in and out again (the acceptance
        # decides between the two, so the state is read twice)
        B, K = case["B"], case["K"]
        return dict(bytes=params + B * (3 * state + 3 * conv + K * (row + 4 * hv * D)), flops=B * K * per_token)
    lens = _lens(case)
    T, n = sum(lens), case["n_seq"]
    return dict(bytes=params + n * (2 * state + 2 * conv) + T * (row + 4 * hv * D), flops=T * per_token)


def tolerance(case):
    kind = case["kind"]
    # About four times the measured distance to exact().
    if kind in ("legacy", "gemv", "q8_0"):
        return {"rel": 1e-6, "differ": 1e-4}                               # 32-bit sums; ties of the q8_1 codes
    if kind == "window":
        return {"rel": 2e-5}                                               # split-bf16 products, K tokens
    if kind == "prefill" and not case["gated"]:
        return {"rel": 6e-5}                                               # the same over chunks of 64 tokens
    return {"rel": 7e-3, "max": 2e-2}                                      # bf16 outputs


# ---------------------------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------------------------

def _silu(v):
    return v * torch.sigmoid(v)


def _recurrence(case, d, rows, n_of, keep=None):
    """Conv, norms, gates and the delta rule in float64. rows[s] are the indices of sequence s's
    token rows (in x, a, b flattened to rows); n_of[s] how many of them. Returns the outputs of
    every row, the states and the conv histories after n_of[s] tokens, or after keep[s] of them
    where keep is given."""
    hk, hv = case["h_k"], case["h_v"]
    f = torch.float64
    C = (2 * hk + hv) * D
    x, a, b = d["x"].reshape(-1, C).to(f), d["a"].reshape(-1, hv).to(f), d["b"].reshape(-1, hv).to(f)
    w = d["conv_w"].to(f)
    y = torch.empty_like(x)
    conv_state = torch.empty_like(d["conv_state"])
    for s, (r0, n) in enumerate(zip(rows, n_of)):
        ext = torch.cat([d["conv_state"][s].to(f).t(), x[r0:r0 + n]])      # [3 + n][C]
        y[r0:r0 + n] = sum(ext[i:i + n] * w[:, i] for i in range(4))
        m = n if keep is None else keep[s]
        conv_state[s] = ext[m:m + 3].t().to(conv_state.dtype)
    if case["opts"] == "next":
        y = _silu(y)
        src = [h // (hv // hk) for h in range(hv)]
        q_scale = float(np.float32(D ** -0.5))
    else:
        src = [h % hk for h in range(hv)]
        q_scale = 1.0
    src = torch.tensor(src, device="cuda")
    q, k, v = (t.reshape(-1, h, D) for t, h in zip(y.split([hk * D, hk * D, hv * D], 1), (hk, hk, hv)))
    eps = float(np.float32(1e-6))
    q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + eps) * q_scale
    k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + eps)
    t = a + d["dt_bias"].to(f)
    g = torch.exp(-torch.exp(d["A_log"].to(f)) * torch.nn.functional.softplus(t, threshold=20.0))
    beta = torch.sigmoid(b)
    S = d["state"].to(f)                                                   # [n][hv][d_v][d_k]
    final = S.clone()
    o = torch.empty(x.shape[0], hv, D, dtype=f, device="cuda")
    order = sorted(range(len(rows)), key=lambda s: -n_of[s])               # longest first
    S = S[order]
    r0 = torch.tensor([rows[s] for s in order], device="cuda")
    for step in range(max(n_of)):
        live = sum(1 for s in order if n_of[s] > step)
        at = r0[:live] + step
        kt, qt = k[at][:, src], q[at][:, src]
        Sl = S[:live]
        Sl *= g[at][:, :, None, None]
        delta = beta[at][:, :, None] * (v[at] - (Sl * kt[:, :, None, :]).sum(-1))
        Sl += delta[:, :, :, None] * kt[:, :, None, :]
        o[at] = (Sl * qt[:, :, None, :]).sum(-1)
        for i in range(live):
            if step + 1 == (n_of[order[i]] if keep is None else keep[order[i]]):
                final[order[i]] = S[i]
    return o, final, conv_state


def _gate_norm(o, d):
    f = torch.float64
    y = o / torch.sqrt((o * o).mean(-1, keepdim=True) + float(np.float32(1e-6)))
    return y * d["ssm_norm"].to(f) * torch.sigmoid(d["z"].reshape(o.shape).to(f))


def exact(case, seed):
    kind = case["kind"]
    f = torch.float64
    if kind == "decode":
        B = case["B"]
        d = _layer_inputs(case, seed, B, (B,))
        o, st, cs = _recurrence(case, d, list(range(B)), [1] * B)
        return dict(o=_gate_norm(o, d) if case["gated"] else o, state=st, conv_state=cs)
    if kind == "prefill":
        lens = _lens(case)
        d = _layer_inputs(case, seed, case["n_seq"], (sum(lens),))
        o, st, cs = _recurrence(case, d, [int(v) for v in np.concatenate([[0], np.cumsum(lens)[:-1]])], lens)
        return dict(o=_gate_norm(o, d) if case["gated"] else o, state=st, conv_state=cs)
    if kind == "window":
        B, K = case["B"], case["K"]
        d = _layer_inputs(case, seed, B, (B, K))
        acc = d["gen"].integers(0, K + 1, B).tolist()
        o, st, cs = _recurrence(case, d, [b * K for b in range(B)], [K] * B, keep=acc)
        return dict(o=o.reshape(B, K, case["h_v"], D), state=st, conv_state=cs)
    if kind == "in_proj":
        d = _in_proj_inputs(case, seed)
        B, hv, C = case["B"], case["h_v"], (2 * case["h_k"] + case["h_v"]) * D
        y = d["h"].to(f) @ d["w"].to(f).t()
        x, z, a, b = y.split([C, hv * D, hv, hv], 1)
        return dict(x=x, z=z.reshape(B, hv, D), a=a, b=b)
    if kind == "gemv":
        d = _gemv_inputs(case, seed)
        return dict(y1=d["w1"].to(f) @ d["x"].to(f), y2=d["w2"].to(f) @ d["x"].to(f))
    if kind == "q8_0":
        # The quantiser's rounding is part of its definition: d = max|x| / 127 in fp32, codes
        # rounded half away from zero, d stored in fp16.
        d = _q8_inputs(case, seed)
        n_out, nc, nb = case["n_out"], case["ncols"], case["n_in"] // 32
        x = d["x"].cpu().numpy().reshape(nc, nb, 32)
        dx = (np.abs(x).max(-1) / np.float32(127.0)).astype(np.float32)
        r = (x / dx[..., None]).astype(np.float32).astype(np.float64)
        codes = np.clip(np.sign(r) * np.floor(np.abs(r) + 0.5), -127, 127)
        xd = torch.from_numpy(codes * dx.astype(np.float16).astype(np.float64)[..., None]).cuda().reshape(nc, -1)
        wd = d["w"][..., :2].contiguous().view(torch.float16).to(f) * d["w"][..., 2:].contiguous().view(torch.int8).to(f)
        return dict(y=xd @ wd.reshape(n_out, -1).t(), xq=None)
    d = _legacy_inputs(case, seed)
    hk, hv, S, dc = case["h_k"], case["h_v"], case["S"], case["d_conv"]
    ext = torch.cat([d["conv_state"], d["x"][:, None]], 1).to(f)           # [C][dc]
    conv = (ext * d["kW"].to(f)).sum(1)
    q, k, v = (t.reshape(-1, S) for t in conv.split([hk * S, hk * S, hv * S]))
    eps = float(np.float32(1e-6))
    q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + eps) for t in (q, k))
    src = torch.arange(hv, device="cuda") % hk
    q, k = q[src], k[src]
    beta = torch.sigmoid(d["beta"].to(f))
    st = d["state"].to(f).permute(1, 0, 2) * torch.exp(d["gate"].to(f))[:, None, None]     # [hv][i][j]
    delta = beta[:, None] * (v - (st * k[:, :, None]).sum(1))
    st = st + k[:, :, None] * delta[:, None, :]
    o = (st * q[:, :, None]).sum(1)
    y = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * d["ssm_norm"].to(f) * torch.sigmoid(d["z"].to(f))
    return dict(y=y, state=st.permute(1, 0, 2).contiguous(), conv_state=ext[:, 1:].contiguous(), beta=beta)
