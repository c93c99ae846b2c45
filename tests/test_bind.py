"""The Python mirror's argument conversion (csrc/bind.cpp): what it refuses before any launch, on
the CPU, and on the GPU the streams and tensors it accepts."""
import ctypes

import pytest
import torch

import baloon_amd as bx


def test_refusals():
    cfg = bx.make_cfg()
    with pytest.raises(ValueError, match="must be on the GPU"):
        bx.ix_gdn_beta_gate(torch.zeros(4), 4, 0)
    with pytest.raises(ValueError, match="must be on the GPU"):        # the first of several
        bx.ix_gdn_decode(cfg, 1, *[torch.zeros(2)] * 8, s=0)
    with pytest.raises(AttributeError):
        bx.ix_gdn_beta_gate([1.0], 4, 0)
    for call in (lambda: bx.ix_gdn_beta_gate(None, 4.5, 0), lambda: bx.ix_gdn_l2_norm(None, 1, 1, "a", 0),
                 lambda: bx.ix_gdn_decode(None, 1, *[None] * 8, s=0),
                 lambda: bx.ix_gdn_decode_gated(cfg, 1, *[None] * 8, gate=cfg, s=0)):
        with pytest.raises(TypeError):
            call()
    # valid conversions, refused by the library before any launch
    assert bx.ix_gdn_beta_gate(None, 4, 0) == bx.HIP_ERROR_INVALID_VALUE
    assert bx.ix_gdn_beta_gate(None, 4, ctypes.c_void_p(0)) == bx.HIP_ERROR_INVALID_VALUE
    assert bx.ix_gdn_decode(cfg, 1, *[None] * 8, s=0) == bx.HIP_ERROR_INVALID_VALUE


def test_descriptions_of_other_types():
    """A program's own ctypes mirror of the C structures is read like the package's."""
    import oracle
    args = [None] * 8
    assert type(oracle.Cfg()) is not bx.Cfg
    assert bx.ix_gdn_decode(oracle.Cfg(), 1, *args, s=0) == bx.HIP_ERROR_INVALID_VALUE

    class Gate(ctypes.Structure):
        _fields_ = bx.OutGate._fields_

    assert bx.ix_gdn_decode_gated(bx.make_cfg(), 1, *args, gate=Gate(), s=0) == bx.HIP_ERROR_INVALID_VALUE
    with pytest.raises(TypeError):
        bx.ix_gdn_decode(ctypes.c_int(1), 1, *args, s=0)


@pytest.mark.gpu
def test_streams_and_tensors():
    x = torch.randn(6, 128, device="cuda")
    want = x / torch.sqrt((x.double() ** 2).sum(1, keepdim=True) + 1e-6).float()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for how in ("current", "object", "address"):
        y = torch.nn.Parameter(x.clone(), requires_grad=False)
        side.wait_stream(torch.cuda.current_stream())
        if how == "current":
            with torch.cuda.stream(side):
                assert bx.ix_gdn_l2_norm(y, 6, 128, 1e-6) == 0
        else:
            assert bx.ix_gdn_l2_norm(y, 6, 128, 1e-6, side if how == "object" else side.cuda_stream) == 0
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        assert float((y - want).abs().max()) <= 1e-6
    with pytest.raises(ValueError, match="contiguous"):
        bx.ix_gdn_l2_norm(x.t(), 128, 6, 1e-6)
