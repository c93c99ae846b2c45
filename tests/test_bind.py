"""The Python mirror's argument conversion (csrc/bind.cpp, and ctypes for what that leaves to it): what it
takes and refuses before any launch, on the CPU, and on the GPU the streams and tensors it accepts."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import baloon_amd as bx
from baloon_amd import build


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


class Stream:
    def __init__(self, cuda_stream):
        self.cuda_stream = cuda_stream


def test_arguments_left_to_ctypes():
    """What ctypes converts is taken as ctypes takes it, and what it refuses is its ArgumentError."""
    for ints in ((0, 1), (ctypes.c_int(0), ctypes.c_int(1)), (np.int64(0), np.int32(1)), (False, 1), (2 ** 40, 1)):   # no rows
        for eps in (1e-6, 1, ctypes.c_float(1e-6), np.float32(1e-6)):
            for s in (0, Stream(0), Stream(None), ctypes.c_void_p(0), ctypes.c_void_p(), 2 ** 64, -1):
                assert bx.ix_gdn_l2_norm(None, *ints, eps, s) == bx.HIP_ERROR_INVALID_VALUE
    assert bx.ix_bf16_gemv(None, None, None, ctypes.c_longlong(0), 0, 0) == bx.HIP_ERROR_INVALID_VALUE
    for args in ((4.5, 1, 1e-6, 0), (4, "a", 1e-6, 0), (4, 1, "a", 0), (4, 1, 10 ** 400, 0), (4, 1, 1e-6, np.int64(0)),
                 (4, 1, 1e-6, 0.0), (ctypes.c_longlong(4), ctypes.c_float(1), 1e-6, 0)):
        with pytest.raises(ctypes.ArgumentError):
            bx.ix_gdn_l2_norm(None, *args)


def test_library_without_the_extension():
    """Where _bind.so does not load, the library's symbols are there, and the calls go through ctypes, with a
    warning."""
    code = """
import sys, warnings
sys.modules["baloon_amd._bind"] = None
import baloon_amd as bx
assert bx.version().startswith("ixgdn") and bx.ix_gdn_in_proj_width(bx.make_cfg()) > 0
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    for _ in range(2):
        assert bx.ix_gdn_beta_gate(None, 4, 0) == bx.HIP_ERROR_INVALID_VALUE
assert len(seen) == 1 and "_bind.so" in str(seen[0].message), seen
"""
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300,
                   cwd=os.path.dirname(os.path.dirname(os.path.abspath(bx.__file__))))


@pytest.mark.parametrize("torch_there", [False, True])
def test_library_is_linked_without_the_extension(monkeypatch, tmp_path, torch_there):
    """Without torch the library alone is built; where the extension's build fails, the library is linked first."""
    for name in ("BUILD", "LIB", "BIND", "RESOURCE_REPORT"):
        monkeypatch.setattr(build, name, str(tmp_path / name))
    if not torch_there:
        monkeypatch.setitem(sys.modules, "torch", None)
    monkeypatch.setattr(build, "_compile", lambda src: (src + ".o", ""))

    def run(cmd, **_):
        if "-ltorch_python" in cmd:
            return subprocess.CompletedProcess(cmd, 1, "", "refused")
        open(cmd[cmd.index("-o") + 1], "w").close()
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(build.subprocess, "run", run)
    if torch_there:
        with pytest.raises(RuntimeError, match="refused"):
            build.build()
    else:
        build.build()
    assert os.path.exists(build.LIB) and not os.path.exists(build.BIND)


@pytest.mark.gpu
def test_streams_and_tensors():
    x = torch.randn(6, 128, device="cuda")
    want = x / torch.sqrt((x.double() ** 2).sum(1, keepdim=True) + 1e-6).float()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for how in ("current", "object", "address", "c_void_p"):
        y = torch.nn.Parameter(x.clone(), requires_grad=False)
        side.wait_stream(torch.cuda.current_stream())
        if how == "current":
            with torch.cuda.stream(side):
                assert bx.ix_gdn_l2_norm(y, 6, 128, 1e-6) == 0
        else:
            s = side if how == "object" else side.cuda_stream
            assert bx.ix_gdn_l2_norm(y, 6, 128, 1e-6, ctypes.c_void_p(s) if how == "c_void_p" else s) == 0
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        assert float((y - want).abs().max()) <= 1e-6
    with pytest.raises(ValueError, match="contiguous"):
        bx.ix_gdn_l2_norm(x.t(), 128, 6, 1e-6)
