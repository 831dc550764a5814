"""GPU parity at the sizes where a launch shape can go wrong: edges of tiles, remainders, the smallest
and largest of a kernel's range, against the CPU oracle (bars: tests/util.py)."""
import numpy as np
import pytest

import lastengine_amd as le
import oracle
from tests.util import acts, check_close, wbytes

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def absmag(ty, q, rows, cols, xs):
    w = oracle.dequant_rows(ty, q, rows, cols).astype(np.float64)
    return np.abs(np.atleast_2d(xs).astype(np.float64)) @ np.abs(w).T


# super-blocks that do not divide over the waves: one item or fewer than waves, 4 waves (more row
# tiles than CUs), 8 and 16 waves, items of two, and a K whose images need fewer waves
@pytest.mark.parametrize("name", list(le.MV_TYPES))
@pytest.mark.parametrize("rows,nsb", [(37, 1), (4112, 3), (100, 7), (4100, 18), (64, 27), (48, 43), (17, 54), (16, 200)])
def test_matvec_ragged_split(engine, name, rows, nsb):
    import torch
    ty, cols = le.MV_TYPES[name], 256 * nsb
    q = wbytes(ty, rows, cols, seed=rows + nsb)
    x = acts(cols, 5 + nsb)
    mag = absmag(ty, q, rows, cols, x)[0]
    y = torch.full((rows,), float("nan"), device="cuda")
    print("ragged split", name, rows, cols, flush=True)
    engine.mv(ty, dev(q), dev(x), y, rows, cols)
    check_close(y.cpu().numpy(), oracle.matvec(ty, q, rows, cols, x), mag)
    # int8 mode: exact integer products, only the fp32 sums differ (as tests/test_gpu_formats.py)
    xq, xd, xs = oracle.quant_x(x)
    y.fill_(float("nan"))
    engine.mv_q8(ty, None, dev(xq), dev(xd), dev(xs), y, rows, cols, 0, 1, w=dev(q))
    want = oracle.matvec_q8(ty, q, rows, cols, xq, xd, xs).astype(np.float64)
    assert np.all(np.abs(y.cpu().numpy() - want) <= 1e-5 * mag + 1e-30)
