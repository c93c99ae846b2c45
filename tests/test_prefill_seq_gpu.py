"""Prefill batches with many sequences (gdn_prefill_seq.hip): one workgroup per sequence and one or
two v heads, against the oracle, with lengths around the chunk's and its tiles' edges.

Tolerances as in test_prefill_gpu.py (outputs 1e-3 absolute, state max|d|/max|ref| 1e-4, conv state
and bf16 rounding exact); y against the norm of the double outputs 1e-4 (test_gated_gpu.py's
end-to-end bound); q8_1 bytes equal the separate quantiser's.
"""
import random

import numpy as np
import pytest

import baloon_amd as bx
import oracle
from oracle import bf16, inputs
from tests.common import (NT, TOL_O_ABS, TOL_STATE_REL, dev, extreme_gates, extreme_params, host, state_from_dev,
                          state_to_dev, tabled_chunks)

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 2, 3, 4, 15, 16, 17, 31, 33, 48, 63, 64, 65, 66, 67, 80, 127, 128, 129, 130]


def run(cfg, cu, tok, p, st, gate=None, window=None, tabled=None, with_o=False):
    """tabled: how many chunks the plan has to send through the windows. with_o: the gated call writes o too."""
    import torch
    n, T = len(cu) - 1, tok["x"].shape[0]
    size = bx.ix_gdn_prefill_workspace_size if gate is None else bx.ix_gdn_prefill_gated_workspace_size
    need = size(cfg, n, T) if window is None else bx.ix_gdn_prefill_window_workspace_size(cfg, n, T, window,
                                                                                          gate is not None)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    d_cs, d_st = dev(st["conv_state"]), state_to_dev(st["state"])
    o = torch.full((T, cfg.h_v, cfg.d_v), float("nan"), device="cuda")
    ob = torch.zeros(T, cfg.h_v, cfg.d_v, dtype=torch.bfloat16, device="cuda")
    args = (cfg, n, T, dev(np.asarray(cu, np.int32)), dev(tok["x"]), d_cs, dev(p["w"]), dev(tok["a"]), dev(tok["b"]),
            dev(p["A_log"]), dev(p["dt_bias"]), d_st)
    if gate is None:
        assert bx.ix_gdn_prefill(*args, o=o, o_bf16=ob, workspace=ws, workspace_bytes=need) == 0
        torch.cuda.synchronize()
        assert tabled is None or tabled_chunks(ws, n) == tabled
        return host(d_cs), state_from_dev(d_st), host(o), host(ob)
    y = torch.full((T, cfg.h_v, cfg.d_v), float("nan"), device="cuda")
    yb = torch.zeros(T, cfg.h_v, cfg.d_v, dtype=torch.bfloat16, device="cuda")
    yq = torch.zeros(T * cfg.h_v * cfg.d_v // 32 * 36, dtype=torch.uint8, device="cuda")
    z, nrm = dev(gate["z"]), dev(gate["nrm"])                  # held: the gate holds addresses alone
    og = bx.out_gate(z, nrm, 1e-6, y, yb, yq)
    assert bx.ix_gdn_prefill_gated(*args, o=o if with_o else None, gate=og, workspace=ws, workspace_bytes=need) == 0
    torch.cuda.synchronize()
    assert tabled is None or tabled_chunks(ws, n) == tabled
    q = torch.zeros_like(yq)
    assert bx.ix_q8_1_quantize(y, q, y.numel()) == 0
    torch.cuda.synchronize()
    np.testing.assert_array_equal(host(yq), host(q))
    return host(d_cs), state_from_dev(d_st), host(y), host(yb)


@pytest.mark.parametrize("kw,n", [
    (dict(h_k=4, h_v=8), 45),                                  # two heads a workgroup
    (dict(h_k=2, h_v=6, head_map=1, conv_act=1), 45),          # an odd count: the last half repeats a head
    (dict(h_k=3, h_v=3, conv_act=1), 60),                      # one head a workgroup
    (dict(h_k=2, h_v=5, d_conv=3), 60),                        # modulo pairing, uneven: 3 and 2 heads
    (dict(h_k=4, h_v=2, d_conv=2), 45),                        # q/k heads without v heads
    (dict(h_k=4, h_v=8, head_map=1, conv_act=1, q_scale=128 ** -0.5), 45),
])
@pytest.mark.parametrize("longest", [130, 1500])
def test_many_sequences(kw, n, longest):
    # Few heads make the windows cheap: the plan leaves most of these batches' chunks to them, and a
    # sequence of 1500 tokens in every case. test_by_sequence has the batches it does not.
    cfg = bx.make_cfg(**kw)
    lens = (EDGES * 3)[:n]
    lens[7] = longest
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, seed = int(cu[-1]), inputs.seed_for(4) + 301 + n + longest
    p, tok = inputs.layer_params(cfg, seed), inputs.token_inputs(cfg, seed, T)
    st, g = inputs.initial_states(cfg, seed, n), inputs.out_gate_inputs(cfg, seed, T)
    rcs, rs, ro = oracle.prefill(cfg, cu, tok["x"], st["conv_state"], p["w"], tok["a"], tok["b"], p["A_log"],
                                 p["dt_bias"], st["state"], nthreads=NT)
    cs, s, o, ob = run(cfg, cu, tok, p, st)
    np.testing.assert_array_equal(cs, rcs)
    assert oracle.rel_err(s, rs) <= TOL_STATE_REL
    assert float(np.max(np.abs(o - ro))) <= TOL_O_ABS
    np.testing.assert_array_equal(ob, bf16.from_f32(o))
    gcs, gs, y, yb = run(cfg, cu, tok, p, st, g)
    np.testing.assert_array_equal(gcs, cs)
    np.testing.assert_array_equal(gs, s)                       # the norm changes no state
    assert oracle.rel_err(y, oracle.gated_out(ro, g["z"], g["nrm"], 1e-6)) <= 1e-4
    np.testing.assert_array_equal(yb, bf16.from_f32(y))
    for a, b in zip((gcs, gs, y, yb), run(cfg, cu, tok, p, st, g, window=2)):
        np.testing.assert_array_equal(a, b)                    # whatever the workspace


def chunks(lens):
    return sum((v + 63) // 64 for v in lens)


@pytest.mark.parametrize("kw,n", [
    (dict(h_k=4, h_v=8), 180),                                 # two heads a workgroup
    (dict(h_k=2, h_v=6, head_map=1, conv_act=1), 220),         # an odd count: the last half repeats a head
    (dict(h_k=3, h_v=3, conv_act=1), 300),                     # one head a workgroup
    (dict(h_k=2, h_v=5, d_conv=3, conv_act=1), 260),           # modulo pairing, uneven: 3 and 2 heads
    (dict(h_k=4, h_v=3, d_conv=2), 300),                       # a q/k head without v heads, one head a workgroup
    (dict(h_k=3, h_v=6, d_conv=2, conv_act=1), 300),
    (dict(h_k=4, h_v=8, head_map=1, conv_act=1, q_scale=128 ** -0.5), 180),
])
@pytest.mark.parametrize("longest,gates", [(200, "drawn"), (1500, "drawn"), (200, "extreme")])
def test_by_sequence(kw, n, longest, gates):
    """Batches whose sequences all run in workgroups of their own, but for one of 1500 tokens (too long a
    walk beside the others) that the windows take, gated too with and without the caller's o."""
    cfg = bx.make_cfg(**kw)
    lens = (EDGES * 15)[:n]
    lens[7] = longest
    tabled = chunks([1500]) if longest == 1500 else 0
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, seed = int(cu[-1]), inputs.seed_for(4) + 501 + n + longest
    p, tok = inputs.layer_params(cfg, seed), inputs.token_inputs(cfg, seed, T)
    if gates == "extreme":                                     # decays of 0 next to decays of 1 (tests/common.py)
        p, tok = extreme_params(p), extreme_gates(cfg, tok, seed)
    st, g = inputs.initial_states(cfg, seed, n), inputs.out_gate_inputs(cfg, seed, T)
    rcs, rs, ro = oracle.prefill(cfg, cu, tok["x"], st["conv_state"], p["w"], tok["a"], tok["b"], p["A_log"],
                                 p["dt_bias"], st["state"], nthreads=NT)
    cs, s, o, ob = run(cfg, cu, tok, p, st, tabled=tabled)
    np.testing.assert_array_equal(cs, rcs)
    # Extreme gates: a chunk's cumulative log decay reaches -8,192, where each of the scan's 6 steps rounds
    # by up to 2^-12; a factor exp(G_t - G_s) takes both ends' errors. (The windows are no closer.)
    assert oracle.rel_err(s, rs) <= (TOL_STATE_REL if gates == "drawn" else 12 * 2.0 ** -12)
    assert float(np.max(np.abs(o - ro))) <= TOL_O_ABS
    np.testing.assert_array_equal(ob, bf16.from_f32(o))
    gated = run(cfg, cu, tok, p, st, g, tabled=tabled)
    np.testing.assert_array_equal(gated[0], cs)
    np.testing.assert_array_equal(gated[1], s)                 # the norm changes no state
    own = oracle.gated_out(o.astype(np.float64), g["z"], g["nrm"], 1e-6)
    assert oracle.rel_err(gated[2], own) <= 1e-5               # test_gated_gpu.py's bound on the call's own outputs
    np.testing.assert_array_equal(gated[3], bf16.from_f32(gated[2]))
    for kwargs in (dict(with_o=True), dict(window=2)):
        for u, v in zip(gated, run(cfg, cu, tok, p, st, g, tabled=tabled, **kwargs)):
            np.testing.assert_array_equal(u, v)


@pytest.mark.parametrize("beta_logit", [None, 30.0])
def test_no_decay_by_sequence(beta_logit):
    """Decays of 1 (and beta = 1): the blocks of (I + A)^-1 as large as they get, over several chunks."""
    cfg, n = bx.make_cfg(h_k=4, h_v=8), 100
    lens = [200 - s % 70 for s in range(n)]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, seed = int(cu[-1]), inputs.seed_for(3) + 43
    p, tok, st = inputs.layer_params(cfg, seed), dict(inputs.token_inputs(cfg, seed, T)), inputs.initial_states(cfg, seed, n)
    tok["a"] = bf16.from_f32(np.full(tok["a"].shape, -30.0, np.float32))
    if beta_logit is not None:
        tok["b"] = bf16.from_f32(np.full(tok["b"].shape, beta_logit, np.float32))
    rcs, rs, ro = oracle.prefill(cfg, cu, tok["x"], st["conv_state"], p["w"], tok["a"], tok["b"], p["A_log"],
                                 p["dt_bias"], st["state"], nthreads=NT)
    cs, s, o, ob = run(cfg, cu, tok, p, st, tabled=0)
    np.testing.assert_array_equal(cs, rcs)
    assert oracle.rel_err(s, rs) <= TOL_STATE_REL
    assert float(np.max(np.abs(o - ro))) <= TOL_O_ABS


@pytest.mark.parametrize("at", ["o", "o_bf16", "z", "y", "y_bf16", None])
def test_alignment(at):
    """Outputs and gate inputs off the vector accesses' alignment send the batch through the windows."""
    import torch
    cfg, n = bx.make_cfg(h_k=4, h_v=8), 64
    lens = [1 + s for s in range(n)]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, seed = int(cu[-1]), inputs.seed_for(4) + 77
    p, tok, st = inputs.layer_params(cfg, seed), inputs.token_inputs(cfg, seed, T), inputs.initial_states(cfg, seed, n)
    g = inputs.out_gate_inputs(cfg, seed, T)

    def buf(name, dtype):
        v = torch.zeros(T * 8 * 128 + 8, dtype=dtype, device="cuda")
        return v[1 if name == at else 0:][:T * 8 * 128]

    bufs = {name: buf(name, torch.bfloat16 if name in ("o_bf16", "z", "y_bf16") else torch.float32)
            for name in ("o", "o_bf16", "z", "y", "y_bf16")}
    bufs["z"].copy_(dev(g["z"]).view(-1))
    need = bx.ix_gdn_prefill_gated_workspace_size(cfg, n, T)
    ws, d_st, d_cs = torch.empty(need, dtype=torch.uint8, device="cuda"), state_to_dev(st["state"]), dev(st["conv_state"])
    nrm = dev(g["nrm"])                                        # held: the gate holds addresses alone
    og = bx.out_gate(bufs["z"], nrm, 1e-6, bufs["y"], bufs["y_bf16"])
    assert bx.ix_gdn_prefill_gated(cfg, n, T, dev(cu), dev(tok["x"]), d_cs, dev(p["w"]), dev(tok["a"]), dev(tok["b"]),
                                   dev(p["A_log"]), dev(p["dt_bias"]), d_st, o=bufs["o"], o_bf16=bufs["o_bf16"], gate=og,
                                   workspace=ws, workspace_bytes=need) == 0
    torch.cuda.synchronize()
    assert tabled_chunks(ws, n) == (0 if at is None else n)
    rcs, rs, ro = oracle.prefill(cfg, cu, tok["x"], st["conv_state"], p["w"], tok["a"], tok["b"], p["A_log"],
                                 p["dt_bias"], st["state"], nthreads=NT)
    o, y = (host(bufs[k]).reshape(T, 8, 128) for k in ("o", "y"))
    np.testing.assert_array_equal(host(d_cs), rcs)
    assert oracle.rel_err(state_from_dev(d_st), rs) <= TOL_STATE_REL
    assert float(np.max(np.abs(o - ro))) <= TOL_O_ABS
    assert oracle.rel_err(y, oracle.gated_out(o.astype(np.float64), g["z"], g["nrm"], 1e-6)) <= 1e-5
    np.testing.assert_array_equal(host(bufs["o_bf16"]), bf16.from_f32(o).reshape(-1))
    np.testing.assert_array_equal(host(bufs["y_bf16"]), bf16.from_f32(y).reshape(-1))


@pytest.mark.parametrize("n", [1, 3, 64])
def test_output_over_the_gate_inputs(n):
    """y_bf16 may overwrite z, row by row, whatever else is written: on one sequence, in windows, by sequence."""
    import torch
    cfg = bx.make_cfg(h_k=4, h_v=8)
    lens = [1 + (37 * s) % 100 for s in range(n)]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, seed = int(cu[-1]), inputs.seed_for(4) + 78 + n
    p, tok, st = inputs.layer_params(cfg, seed), inputs.token_inputs(cfg, seed, T), inputs.initial_states(cfg, seed, n)
    g = inputs.out_gate_inputs(cfg, seed, T)
    need = bx.ix_gdn_prefill_gated_workspace_size(cfg, n, T)

    def call(over):
        z, ws = dev(g["z"]), torch.empty(need, dtype=torch.uint8, device="cuda")
        y, yb = torch.zeros(T, 8, 128, device="cuda"), z if over else torch.zeros_like(z)
        yq, nrm = torch.zeros(T * 8 * 4 * 36, dtype=torch.uint8, device="cuda"), dev(g["nrm"])
        assert bx.ix_gdn_prefill_gated(cfg, n, T, dev(cu), dev(tok["x"]), dev(st["conv_state"]), dev(p["w"]), dev(tok["a"]),
                                       dev(tok["b"]), dev(p["A_log"]), dev(p["dt_bias"]), state_to_dev(st["state"]),
                                       gate=bx.out_gate(z, nrm, 1e-6, y, yb, yq), workspace=ws,
                                       workspace_bytes=need) == 0
        torch.cuda.synchronize()
        assert n == 1 or tabled_chunks(ws, n) == (0 if n == 64 else chunks(lens))
        return host(y), host(yb), host(yq)

    for u, v in zip(call(False), call(True)):
        np.testing.assert_array_equal(u, v)


def test_plan_prices_long_sequences():
    """A walk is as long as its longest sequence, also past the lengths the plan tells apart: one of
    3,000 chunks among short ones goes through the windows (19 ms against 50 in a workgroup of its own), the
    others do not. (Zero inputs: the plan sees the lengths alone.)"""
    import torch
    cfg = bx.make_cfg(h_k=16, h_v=96)
    lens = [3000 * 64] + [100] * 40
    n, T, C = len(lens), sum(lens), cfg.channels
    bf = dict(dtype=torch.bfloat16, device="cuda")
    x, a = torch.zeros(T, C, **bf), torch.zeros(T, 96, **bf)
    cu = dev(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
    need = bx.ix_gdn_prefill_workspace_size(cfg, n, T)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    assert bx.ix_gdn_prefill(cfg, n, T, cu, x, torch.zeros(n, C, 3, **bf), torch.zeros(C, 4, **bf), a, a,
                             torch.zeros(96, device="cuda"), torch.zeros(96, device="cuda"),
                             torch.zeros(n, 96, 128, 128, device="cuda"), workspace=ws, workspace_bytes=need) == 0
    torch.cuda.synchronize()
    assert tabled_chunks(ws, n) == 3000


@pytest.mark.parametrize("n,gated,tabled", [(12, True, True), (14, False, True), (32, False, False), (32, True, False)])
def test_plan_routes(n, gated, tabled):
    """U[1, 2048] tokens, 16 q/k and 32 v heads: 12 sequences are not priced, 14 fill too few CUs and are faster in
    windows, 32 are faster by sequence (measured at by_sequence, gdn_prefill.hip). Zero inputs: the plan sees the
    lengths alone."""
    import torch
    cfg = bx.make_cfg(conv_act=int(gated))
    rng = random.Random(4)
    lens = [rng.randint(1, 2048) for _ in range(n)]
    T, bf = sum(lens), dict(dtype=torch.bfloat16, device="cuda")
    x, a = torch.zeros(T, cfg.channels, **bf), torch.zeros(T, 32, **bf)
    z, yb, nrm = torch.zeros(T, 32, 128, **bf), torch.empty(T, 32, 128, **bf), torch.ones(128, device="cuda")
    need = bx.ix_gdn_prefill_gated_workspace_size(cfg, n, T)
    ws, zero = torch.empty(need, dtype=torch.uint8, device="cuda"), torch.zeros(32, device="cuda")
    args = (cfg, n, T, dev(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)), x, torch.zeros(n, cfg.channels, 3, **bf),
            torch.zeros(cfg.channels, 4, **bf), a, a, zero, zero, torch.zeros(n, 32, 128, 128, device="cuda"))
    if gated:
        assert bx.ix_gdn_prefill_gated(*args, gate=bx.out_gate(z, nrm, 1e-6, None, yb), workspace=ws, workspace_bytes=need) == 0
    else:
        assert bx.ix_gdn_prefill(*args, o_bf16=yb, workspace=ws, workspace_bytes=need) == 0
    torch.cuda.synchronize()
    assert tabled_chunks(ws, n) == (chunks(lens) if tabled else 0)


def test_more_workgroups_than_a_launch_takes():
    """2,048 sequences with 4,096 q/k heads would be 2^32 threads by sequence: they stay in the windows. (One v
    head, so that the states fit; inputs of one token each, of which k and q are zero.)"""
    import torch
    if torch.cuda.mem_get_info()[0] < 60e9:
        pytest.skip("needs 40 GB of device memory")
    cfg, n = bx.make_cfg(h_k=4096, h_v=1), 2048
    C, bf = cfg.channels, dict(dtype=torch.bfloat16, device="cuda")
    x = torch.zeros(n, C, **bf)
    x[:, -128:] = 1.0
    a, cs, zero = torch.zeros(n, 1, **bf), torch.zeros(n, C, 3, **bf), torch.zeros(1, device="cuda")
    need = bx.ix_gdn_prefill_window_workspace_size(cfg, n, n, 16, False)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    assert bx.ix_gdn_prefill(cfg, n, n, torch.arange(n + 1, dtype=torch.int32, device="cuda"), x, cs, torch.zeros(C, 4, **bf),
                             a, a, zero, zero, torch.zeros(n, 1, 128, 128, device="cuda"), workspace=ws,
                             workspace_bytes=need) == 0
    torch.cuda.synchronize()
    assert tabled_chunks(ws, n) == n
    assert bool((cs[:, -128:, 2] == 1).all())


def test_graph_replays():
    """A captured call (the plan, walks, windows and the norm over the table's chunks) replays like eager calls,
    each from the states the one before left, with eager work in between."""
    import torch
    cfg, lens = bx.make_cfg(h_k=4, h_v=8, conv_act=1), [1500] + [1 + (53 * s) % 190 for s in range(120)]
    n, T = len(lens), sum(lens)
    seed = inputs.seed_for(4) + 91
    p, tok, st = inputs.layer_params(cfg, seed), inputs.token_inputs(cfg, seed, T), inputs.initial_states(cfg, seed, n)
    g = inputs.out_gate_inputs(cfg, seed, T)
    cu = dev(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
    x, a, b, w, A, dt, z, nrm = (dev(v) for v in (tok["x"], tok["a"], tok["b"], p["w"], p["A_log"], p["dt_bias"], g["z"], g["nrm"]))
    need = bx.ix_gdn_prefill_gated_workspace_size(cfg, n, T)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")

    def buffers():
        return (dev(st["conv_state"]), state_to_dev(st["state"]), torch.zeros(T, 8, 128, device="cuda"),
                torch.zeros(T, 8, 128, device="cuda"))

    def call(cs, state, o, y):
        assert bx.ix_gdn_prefill_gated(cfg, n, T, cu, x, cs, w, a, b, A, dt, state, o=o, gate=bx.out_gate(z, nrm, 1e-6, y),
                                       workspace=ws, workspace_bytes=need) == 0

    eager, graphed = buffers(), buffers()
    call(*buffers())                                           # outside the capture once
    torch.cuda.synchronize()
    assert tabled_chunks(ws, n) == chunks([1500])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(*graphed)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        call(*eager)
        torch.cuda.synchronize()
        for u, v in zip(graphed, eager):
            np.testing.assert_array_equal(host(u), host(v))
