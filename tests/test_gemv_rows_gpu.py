"""The bf16 products with few rows (loads of several steps ahead) against the double reference of
oracle/proj.py and, bit for bit, against the kernels that take more rows: row lengths around the
batches of 4, 2 and 1 steps of 512 values, and row counts on both sides of the lines between the
kernels. Tolerance 2e-5 x sum|x w|, as in test_proj_gpu.py.
"""
import numpy as np
import pytest

import baloon_amd as bx
from oracle import proj
from tests.common import host

pytestmark = pytest.mark.gpu


def _bf16(t):
    import torch
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("n_in", [8, 504, 512, 520, 1024, 1032, 1544, 2048, 2056, 2568, 3072, 3592, 4104])
def test_gemv_few_rows(n_in):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(0x6D4E0B00 + n_in)
    n, n2 = 4097, 4096
    x = torch.randn(n_in, device="cuda", generator=g).bfloat16()
    w = torch.randn(n, n_in, device="cuda", generator=g).bfloat16()
    w2 = torch.randn(n2, n_in, device="cuda", generator=g).bfloat16()

    def single(m, k):
        y = torch.full((k + 1,), float("nan"), device="cuda")
        assert bx.ix_bf16_gemv(x, m, y, n_in, k) == 0
        assert bool(torch.isnan(y[k]))
        return host(y[:k])

    many = single(w, n)                                        # one row past the line
    rows = np.r_[0:3, n - 3:n]
    ref, mag = proj.gemv_ref(_bf16(x), _bf16(w)[rows])
    assert float((np.abs(many[rows].astype(np.float64) - ref) / mag).max()) <= 2e-5
    for k in (1, 3, 4, 1000, n - 1):
        np.testing.assert_array_equal(single(w, k), many[:k])
    y2_all = single(w2, n2)
    for k1, k2 in ((1, 1), (3, 6), (70, 1001), (n - 1, n2), (n, n2), (5, 0), (0, 7)):
        y1, y2 = (torch.full((k + 1,), float("nan"), device="cuda") for k in (k1, k2))
        assert bx.ix_bf16_gemv_pair(x, w, y1, k1, w2, y2, k2, n_in) == 0
        np.testing.assert_array_equal(host(y1[:k1]), many[:k1])
        np.testing.assert_array_equal(host(y2[:k2]), y2_all[:k2])
        assert bool(torch.isnan(y1[k1])) and bool(torch.isnan(y2[k2]))
