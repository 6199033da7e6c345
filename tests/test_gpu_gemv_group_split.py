"""A decode group on the GEMV whose rows together would leave K unsplit.

From five activation rows on, the GEMV's unsplit workgroups are 128 threads to a staged activation.
Where few stagings fit a CU, matrices that alone are split in K keep launches of their own, so
the group's columns are bit for bit those of separate calls; elsewhere one launch takes them all.
"""
import ctypes

import numpy as np
import pytest
import torch

import _oracle as O
from test_gpu_parity import DEV, TOL_F32, _stream, gpu_mmvq, gpu_prepare, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [5, 8])
@pytest.mark.parametrize("k,rows,apart", [
    (12320, (12, 2100, 2000), True), (12320, (4100, 7), True), (3104, (4100, 7, 12300), False), (8224, (1030, 16, 3090), False)])
def test_group_keeps_each_matrix_split(kai, m, k, rows, apart):
    """Q4_0, K off whole 256-value steps: the GEMV whatever the rows."""
    print(f"gemv group split k={k} m={m} rows={rows}", flush=True)
    rng = np.random.default_rng(k + m + sum(rows))
    ws = [O.random_blocks(O.Q4_0, n, k, rng) for n in rows]
    dev = [to_dev(w) for w in ws]
    x = rng.standard_normal((m, k)).astype(np.float32)
    act = gpu_prepare(kai, to_dev(x))
    count, total = len(rows), sum(rows)
    out = torch.full((m, total), float("nan"), dtype=torch.float32, device=DEV)
    st = kai.kai_fused_mmvq_group((ctypes.c_void_p * count)(*[d.data_ptr() for d in dev]),
                                  (ctypes.c_int * count)(*[O.Q4_0] * count), (ctypes.c_int64 * count)(*rows), count, k, m,
                                  act.data_ptr(), 0, out.data_ptr(), 0, total, _stream())
    assert st == 0, kai.current_direct_error()
    off = 0
    for n, w, d in zip(rows, ws, dev):
        alone = gpu_mmvq(kai, O.Q4_0, d, n, k, act, m)
        ref = O.mul_mat(O.Q4_0, w, k, O.prepare(x), m)
        for got in (out[:, off:off + n], alone):
            assert O.normwise_rel(got.cpu().numpy(), ref) <= TOL_F32, n
        assert not apart or torch.equal(out[:, off:off + n], alone), n
        off += n
