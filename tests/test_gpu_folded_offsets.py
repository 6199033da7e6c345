"""The folded fp16 GEMM on weights whose blocks carry an offset.

Q4_K and Q2_K hold a block as scale x code - min, so weights that are not centred on zero come as
small differences of large terms. The GEMM rounds dw (c - c0) and the activation to fp16; the
offset itself must meet the blocks' unrounded sums, or both roundings scale with it. Weights of
mean -4 and +4 standard deviations, against plain activation rows and rows that sum to zero (where
the offset cancels in the result but not in a rounding). Measured on these shapes: 3.0e-4 to 7.1e-4
of the row's largest output with the offset apart, 1.1e-3 to 2.2e-3 with it inside the rounded operand.
"""
import numpy as np
import pytest

import _oracle as O
from test_gpu_parity import TOL_F32, gpu_mmq, to_dev

pytestmark = pytest.mark.gpu

# weight rows, K, activation rows: few rows with K in groups of waves, an odd number of superblocks
# (Q4_K pairs them), whole rounds of 128- and 256-row tiles
SHAPES = [(260, 5120, 40), (1000, 2304, 90), (4100, 5120, 200), (8196, 2560, 600)]


@pytest.mark.parametrize("qtype", [O.Q4_K, O.Q2_K], ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("mean", [-4.0, 4.0])
@pytest.mark.parametrize("n,k,m", SHAPES)
def test_offset_weights(kai, qtype, mean, n, k, m):
    from kaillm_amd.formats import quantize

    rng = np.random.default_rng(qtype + n + k + m)
    w = quantize((0.02 * (rng.standard_normal((n, k), dtype=np.float32) + mean)).astype(np.float32), qtype)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[1::2] -= x[1::2].mean(axis=1, keepdims=True)  # every other row sums to zero
    cols = np.unique(np.concatenate([[0, n - 1], rng.choice(n, 256)]))
    ref = O.mmq_reference(qtype, w[cols], x, threads=16)
    out = gpu_mmq(kai, [(qtype, w, to_dev(w))], to_dev(x))
    err = O.normwise_rel(out[:, cols].cpu().numpy(), ref)
    print(f"offset {O.NAMES[qtype]} mean {mean} {n}x{k} m={m}: normwise rel err {err:.3e}", flush=True)
    assert err <= TOL_F32
