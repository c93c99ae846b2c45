"""The Q8_0 product with many rows (activations in LDS) against the double reference of
oracle/proj.py: block counts around a wave's 64, row counts around the workgroups' 8 waves, the
longest rows it takes and the first ones it leaves. Tolerance 1e-5 x sum|d_w d_x| 32 127^2 and column
results independent of the number of columns, as in test_proj_gpu.py.
"""
import numpy as np
import pytest

import baloon_amd as bx
from oracle import proj
from tests.common import dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,n_out", [(32, 1024), (2016, 1025), (2048, 1031), (2080, 1023), (4128, 1024),
                                        (7264, 1030), (7296, 1030), (64, 9001)])
def test_q8_0_many_rows(n_in, n_out):
    import torch
    nb = n_in // 32
    seed = 0x6D4E0A00 + n_in + n_out
    wd, wq = proj.q8_blocks(seed, 1, n_out, nb)
    xd, xq = proj.q8_blocks(seed, 5, 8, nb)
    ref, sc = proj.q8_0_ref(wd, wq, xd, xq)
    w, x = dev(proj.pack_q8_0(wd, wq)), dev(proj.pack_q8_1(xd, xq))
    outs = {}
    for nc in (8, 7, 6, 5, 4, 3, 2, 1):
        y = torch.full((8, n_out), float("nan"), device="cuda")
        assert bx.ix_mmvq_q8_0(w, x, y, n_in, n_out, nc) == 0
        outs[nc] = host(y)
        assert float((np.abs(outs[nc][:nc].astype(np.float64) - ref[:nc]) / sc[:nc]).max()) <= 1e-5
        assert np.isnan(outs[nc][nc:]).all()
        np.testing.assert_array_equal(outs[nc][:nc], outs[8][:nc])


def test_q8_0_most_rows():
    """The largest n_out the call takes (73 GB of one-block rows): the first and last rows hold codes, the others
    are zero; the row counter of a wave passes 2^31 behind the last one."""
    import torch
    n_out = 2 ** 31 - 1
    if torch.cuda.mem_get_info()[0] < 100e9:
        pytest.skip("needs 82 GB of device memory")
    wd, wq = proj.q8_blocks(0x6D4E0A07, 1, 16, 1)
    xd, xq = proj.q8_blocks(0x6D4E0A07, 5, 1, 1)
    ref, sc = proj.q8_0_ref(wd, wq, xd, xq)
    rows, x = dev(proj.pack_q8_0(wd, wq)).view(16, 34), dev(proj.pack_q8_1(xd, xq))
    w = torch.zeros(n_out * 34, dtype=torch.uint8, device="cuda")
    w[:8 * 34] = rows[:8].reshape(-1)
    w[-8 * 34:] = rows[8:].reshape(-1)
    y = torch.full((n_out + 1,), float("nan"), device="cuda")
    assert bx.ix_mmvq_q8_0(w, x, y, 32, n_out, 1) == 0
    got = host(torch.cat([y[:8], y[n_out - 8:n_out]]))
    assert float((np.abs(got.astype(np.float64) - ref[0]) / sc[0]).max()) <= 1e-5
    assert bool(torch.isnan(y[n_out])) and int(torch.count_nonzero(y[8:n_out - 8])) == 0
