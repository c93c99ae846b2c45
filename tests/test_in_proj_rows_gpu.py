"""The input projection at prompt sizes (in_proj_tile_kernel) against a double product: row counts
around the tiles' edges, each tile size, and the columns past the last whole tile. bf16 pieces within
half a bf16 ulp plus the GEMV tolerance 2e-5 x sum|h w| (test_proj_gpu.py); a call that also asks for
the fp32 result runs on small tiles and must agree to the same bound.
"""
import pytest

import baloon_amd as bx

pytestmark = pytest.mark.gpu


# Each row's comment: the tiles that the library's prices choose there.
@pytest.mark.parametrize("kw,B,hidden", [
    ({}, 8200, 64),                            # 256 x 256, one k stage
    ({}, 4097, 128),                           # 256 x 256, two stages, a row past the last whole tile
    ({}, 4095, 192),                           # 256 x 256, three
    ({}, 1025, 512),                           # 256 x 256
    (dict(h_k=2, h_v=5), 9001, 256),           # 128 x 128 (an odd number of them across x), four stages
    ({}, 385, 1024),                           # 128 x 128
])
def test_in_proj_rows(kw, B, hidden):
    import torch
    cfg = bx.make_cfg(**kw)
    N = bx.ix_gdn_in_proj_width(cfg)
    gen = torch.Generator(device="cuda").manual_seed(B + hidden)
    h = torch.randn(B, hidden, device="cuda", generator=gen).bfloat16()
    w = (0.05 * torch.randn(N, hidden, device="cuda", generator=gen)).bfloat16()
    ref, mag = h.double() @ w.double().t(), h.double().abs() @ w.double().abs().t()
    bf = dict(dtype=torch.bfloat16, device="cuda")

    def pieces():
        return [torch.full((B, cfg.channels), float("nan"), **bf), torch.full((B, cfg.h_v, cfg.d_v), float("nan"), **bf),
                torch.full((B, cfg.h_v), float("nan"), **bf), torch.full((B, cfg.h_v), float("nan"), **bf)]

    for out_y in (None, torch.empty(B, N, device="cuda")):
        out = pieces()
        assert bx.ix_gdn_in_proj(cfg, B, hidden, h, w, *out, out_y) == 0
        torch.cuda.synchronize()
        got = torch.cat([v.reshape(B, -1) for v in out], 1).double()
        # half a bf16 ulp is at most 2^-8 of the value
        assert bool(((got - ref).abs() <= 2e-5 * mag + (ref.abs() + 2e-5 * mag) * 2.0 ** -8).all())
