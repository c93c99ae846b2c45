"""How exactly the prefill evaluates its transcendental steps (SiLU, decay, output gate), in the
windows and one workgroup per sequence: inputs chosen so that a result shows one such value.

The matrix products split an fp32 operand into two bf16 (16 bits of it), so a value that goes
through them is compared with the split of the correctly rounded value: the two differ where the
rounding of the lower part falls the other way, by up to 2^-17 relative. Emulated for SiLU over [-64, -16],
that shifts 1.1% of the values by more than 1e-6 for an exponential and a division exact to an ulp
(relative error below 2.2e-7), and 20% for an exponential of a rounded argument (up to 3.3e-6).
"""
import numpy as np
import pytest

import baloon_amd as bx
from oracle import bf16, inputs
from tests.common import dev, host, state_from_dev, state_to_dev, tabled_chunks

pytestmark = pytest.mark.gpu
N = 64                                                         # sequences of the batches
DIFFER = 0.05


def split(v):
    """The two-bf16 split of values, as float64."""
    v = np.asarray(v, np.float32)
    hi = bf16.round_f32(v)
    return hi.astype(np.float64) + bf16.round_f32(v - hi)


def differing(got, ref):
    return float(np.mean(np.abs(got - ref) > 1e-6 * np.abs(ref)))


def prefill(route, cfg, lens, x, a, b, state, gate=None):
    """One call on the sequences (lens[s] tokens each), taps (0, .., 0, 1), A_log = dt_bias = 0; returns the
    state, o and, with gate = (z, nrm), y."""
    import torch
    n, T, C = len(lens), sum(lens), cfg.channels
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    w = np.zeros((C, cfg.d_conv), np.float32)
    w[:, -1] = 1.0
    d_st = state_to_dev(state)
    o = torch.full((T, cfg.h_v, 128), float("nan"), device="cuda")
    # The windows take an o_bf16 at any address, a workgroup per sequence only 8-byte aligned ones.
    ob = torch.zeros(T * cfg.h_v * 128 + 1, dtype=torch.bfloat16, device="cuda")[1:] if route == "windows" else None
    need = bx.ix_gdn_prefill_gated_workspace_size(cfg, n, T)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    zero = torch.zeros(cfg.h_v, device="cuda")
    args = (cfg, n, T, dev(cu), dev(bf16.from_f32(x)), torch.zeros(n, C, cfg.d_conv - 1, dtype=torch.bfloat16, device="cuda"),
            dev(bf16.from_f32(w)), dev(bf16.from_f32(a)), dev(bf16.from_f32(b)), zero, zero, d_st)
    y = None
    if gate is None:
        assert bx.ix_gdn_prefill(*args, o=o, o_bf16=ob, workspace=ws, workspace_bytes=need) == 0
    else:
        y = torch.full_like(o, float("nan"))
        z, nrm = dev(bf16.from_f32(gate[0])), dev(gate[1])     # held: the gate holds their addresses alone
        og = bx.out_gate(z, nrm, 1e-6, y)
        assert bx.ix_gdn_prefill_gated(*args, o=o, o_bf16=ob, gate=og, workspace=ws, workspace_bytes=need) == 0
    torch.cuda.synchronize()
    if n > 1:
        assert tabled_chunks(ws, n) == (0 if route == "seq" else sum((v + 63) // 64 for v in lens))
    return state_from_dev(d_st), host(o), None if y is None else host(y)


def drawn(rng, *shape):
    return bf16.round_f32(rng.uniform(-64.0, -16.0, shape))


@pytest.mark.parametrize("route", ["seq", "windows", "single"])
def test_silu(route):
    """One token per sequence; channel 0 of a head is 50 (SiLU 50, norm 50), the others show their own SiLU."""
    cfg = bx.make_cfg(h_k=4, h_v=8, conv_act=1)
    n = 1 if route == "single" else N
    rng = np.random.default_rng(1)
    silu = lambda v: (v.astype(np.float64) / (1.0 + np.exp(-v.astype(np.float64)))).astype(np.float32)  # noqa: E731
    head = np.zeros((4, 128), np.float32)
    head[:, 0] = 50.0
    drawn_k, drawn_v = drawn(rng, n, 4, 128), drawn(rng, n, 8, 128)
    drawn_k[..., 0] = drawn_v[..., 0] = 50.0
    full = lambda v: np.full((n, 8), v, np.float32)  # noqa: E731
    src = np.arange(8) % 4
    # S = 0, beta = 1: S' = k v^T; row 0 (k = 1) shows v, column 0 (v = 50) shows k.
    x = np.concatenate([np.broadcast_to(head.reshape(-1), (n, 512)), drawn_k.reshape(n, -1), drawn_v.reshape(n, -1)], 1)
    s, o, _ = prefill(route, cfg, [1] * n, x, full(0), full(30.0), np.zeros((n, 8, 128, 128), np.float32))
    k = split(silu(drawn_k) * np.float32(0.02))
    assert differing(s[:, :, 0, 1:], split(silu(drawn_v))[..., 1:]) <= DIFFER
    assert differing(s[:, :, 1:, 0], 50.0 * k[:, src, 1:]) <= DIFFER
    assert differing(o[..., 1:], split(silu(drawn_v))[..., 1:]) <= DIFFER
    # S = 1, beta = 0, no decay: o = q.
    x = np.concatenate([drawn_k.reshape(n, -1), np.broadcast_to(head.reshape(-1), (n, 512)), drawn_v.reshape(n, -1)], 1)
    s, o, _ = prefill(route, cfg, [1] * n, x, full(-100.0), full(-200.0),
                      np.broadcast_to(np.eye(128, dtype=np.float32), (n, 8, 128, 128)))
    assert differing(o[..., 1:], k[:, src, 1:]) <= DIFFER


@pytest.mark.parametrize("route", ["seq", "windows"])
def test_decay(route):
    """Whole gate logits above softplus's threshold: the log decay is minus the logit, exactly."""
    cfg = bx.make_cfg(h_k=4, h_v=8)
    rng = np.random.default_rng(2)
    a = (21 + np.arange(N * 8) % 40).reshape(N, 8).astype(np.float32)
    x = np.zeros((N, 16, 128), np.float32)
    x[:, :8, 0] = 50.0                                         # q = k = the first unit vector
    x[:, 8:] = bf16.round_f32(rng.standard_normal((N, 8, 128)))
    state = bf16.round_f32(rng.standard_normal((N, 8, 128, 128)))
    # beta = 0: S' = exp(-a) S, to the exponential's and the product's rounding; o = its row 0, times
    # q's factor (a square root and two products) twice rounded.
    s, o, _ = prefill(route, cfg, [1] * N, x.reshape(N, -1), a, np.full((N, 8), -200.0), state)
    want = np.exp(-a.astype(np.float64))[:, :, None, None] * state
    assert float(np.max(np.abs(s / want - 1.0))) <= 1.5 * 2.0 ** -23
    assert float(np.max(np.abs(o / want[:, :, 0] - 1.0))) <= 4.5 * 2.0 ** -23
    # Two tokens, S = 0, beta = 1 and then 0: S' = exp(-a_1) k v_0^T.
    two = lambda u, v: np.stack([u, v], 1).reshape(2 * N, -1)  # noqa: E731
    s, _, _ = prefill(route, cfg, [2] * N, two(x.reshape(N, -1), x.reshape(N, -1)), two(a, a),
                      two(np.full((N, 8), 30.0), np.full((N, 8), -200.0)), np.zeros_like(state))
    assert differing(s[:, :, 0], split(np.exp(-a.astype(np.float64))[..., None] * x[:, 8:])) <= DIFFER


@pytest.mark.parametrize("route", ["seq", "windows"])
def test_output_gate(route):
    """y from the call's own fp32 o: the sum of 128 squares (at most 9 roundings, halved by the root), its
    scaling, root and reciprocal, three products and the sigmoid (an ulp), each half an ulp."""
    cfg = bx.make_cfg(h_k=4, h_v=8)
    rng = np.random.default_rng(3)
    x, z = rng.standard_normal((N, 16 * 128)), bf16.round_f32(rng.uniform(-80.0, 80.0, (N, 8, 128)))
    nrm = (1.0 + 0.1 * rng.standard_normal(128)).astype(np.float32)
    _, o, y = prefill(route, cfg, [1] * N, x, rng.standard_normal((N, 8)), rng.standard_normal((N, 8)),
                      0.02 * rng.standard_normal((N, 8, 128, 128)), (z, nrm))
    o = o.astype(np.float64)
    want = o / np.sqrt((o * o).mean(-1, keepdims=True) + 1e-6) * nrm / (1.0 + np.exp(-z.astype(np.float64)))
    err = float(np.max(np.abs(y / want - 1.0)))
    assert err <= (4.5 + 1.0 + 3 * 1.0 + 1.5 + 2.0) * 2.0 ** -24, err
