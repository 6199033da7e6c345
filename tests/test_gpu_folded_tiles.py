"""Every tile configuration of the folded fp16 GEMM for every format, at shapes whose launch plan picks it.

Above 16 rows kai_fused_mmq_run picks among ten tile configurations (kai_batched_plan.h) by the
matrix's rows, K and the activation rows, each whole, with K splits, with a tail of K pieces (over all
rows, or two and more activation tiles down and beside whole tiles) or with a second launch of
quarter tiles. Each case states what it stands for and asks the plan, so a retuned plan makes the case
fail rather than test something else. Ragged weight and activation rows, odd numbers of superblocks
(Q4_K's min pass pairs them), K that ends inside a superblock for the 32-value formats, an output
slice that starts off 16 bytes. The GPU runs the whole product; the oracle checks a column of every weight
tile, the first and last rows and a seeded sample, within the bars of test_gpu_parity.
"""
import numpy as np
import pytest
import torch

import _oracle as O
import _plan as P
from test_gpu_fullsize import sample_cols
from test_gpu_parity import TOL_BF16, TOL_F32, gpu_mmq, to_dev

pytestmark = pytest.mark.gpu

# format, configuration, kind, weight rows, K, activation rows; tail: K pieces over every activation row,
# tail2: from an activation tile on, whole tiles beside them
CASES = [
    ("Q4_K", "WIDE", "whole", 7200, 256, 1060), ("Q4_K", "WIDE", "rest", 65628, 256, 132),
    ("Q4_K", "TALL", "whole", 3652, 768, 1096), ("Q4_K", "TALL", "tail2", 7516, 5888, 1080),
    ("Q4_K", "HALF", "whole", 3668, 256, 1071), ("Q4_K", "HALF", "tail2", 9644, 1792, 802),
    ("Q4_K", "HALF2", "whole", 1168, 256, 1059), ("Q4_K", "HALF2", "split", 812, 3328, 969),
    ("Q4_K", "HALF2", "tail2", 3608, 5376, 1091), ("Q4_K", "ROWS96", "whole", 4284, 256, 277),
    ("Q4_K", "ROWS96", "split", 1636, 6400, 258), ("Q4_K", "ROWS96", "tail2", 11404, 4608, 257),
    ("Q4_K", "ROWS64", "whole", 676, 256, 1066), ("Q4_K", "ROWS64", "split", 8556, 2816, 46),
    ("Q4_K", "ROWS32", "whole", 752, 256, 962), ("Q4_K", "ROWS32", "split", 8276, 2816, 30),
    ("Q4_K", "ROWS32", "tail", 32772, 1536, 19), ("Q4_K", "THIN96", "whole", 456, 256, 1095),
    ("Q4_K", "THIN96", "split", 108, 6400, 1077), ("Q4_K", "THIN64", "whole", 228, 256, 1034),
    ("Q4_K", "THIN64", "split", 36, 5376, 975), ("Q4_K", "THIN32", "whole", 36, 256, 17),
    ("Q4_K", "THIN32", "split", 36, 4352, 18),
    ("Q2_K", "WIDE", "whole", 49380, 256, 139), ("Q2_K", "TALL", "whole", 4520, 1280, 969),
    ("Q2_K", "TALL", "tail2", 9096, 3840, 907), ("Q2_K", "HALF", "whole", 2720, 256, 1074),
    ("Q2_K", "HALF", "split", 648, 6400, 953), ("Q2_K", "HALF", "tail", 66200, 1280, 67),
    ("Q2_K", "HALF", "tail2", 9352, 1280, 878), ("Q2_K", "HALF2", "tail2", 4400, 5376, 906),
    ("Q2_K", "ROWS96", "whole", 1952, 256, 1048), ("Q2_K", "ROWS96", "split", 284, 5888, 1040),
    ("Q2_K", "ROWS96", "tail", 33296, 2304, 78), ("Q2_K", "ROWS96", "tail2", 4628, 4352, 849),
    ("Q2_K", "ROWS64", "whole", 696, 256, 1077), ("Q2_K", "ROWS64", "split", 228, 5376, 1083),
    ("Q2_K", "ROWS64", "tail", 33004, 1792, 40), ("Q2_K", "ROWS32", "whole", 1368, 256, 486),
    ("Q2_K", "ROWS32", "split", 2740, 5888, 18), ("Q2_K", "ROWS32", "tail", 33344, 2304, 22),
    ("Q2_K", "THIN96", "whole", 484, 256, 1036), ("Q2_K", "THIN96", "split", 104, 6400, 1049),
    ("Q2_K", "THIN64", "whole", 228, 256, 1059), ("Q2_K", "THIN64", "split", 36, 4864, 1043),
    ("Q2_K", "THIN32", "whole", 36, 256, 17), ("Q2_K", "THIN32", "split", 36, 3840, 25),
    ("IQ3_S", "WIDE", "whole", 7188, 256, 1093), ("IQ3_S", "WIDE", "split", 4780, 5888, 924),
    ("IQ3_S", "WIDE", "rest", 67152, 256, 134), ("IQ3_S", "TALL", "whole", 5072, 2816, 1067),
    ("IQ3_S", "TALL", "tail2", 11580, 5888, 643), ("IQ3_S", "HALF", "whole", 3592, 256, 1071),
    ("IQ3_S", "HALF", "split", 3400, 6144, 612), ("IQ3_S", "HALF", "tail", 65724, 768, 25),
    ("IQ3_S", "HALF", "tail2", 7348, 2816, 1055), ("IQ3_S", "HALF2", "whole", 2836, 256, 1082),
    ("IQ3_S", "HALF2", "split", 900, 2816, 987), ("IQ3_S", "HALF2", "tail", 32968, 1792, 120),
    ("IQ3_S", "HALF2", "tail2", 3592, 3840, 1050), ("IQ3_S", "ROWS96", "whole", 1880, 256, 1090),
    ("IQ3_S", "ROWS96", "split", 264, 6400, 979), ("IQ3_S", "ROWS96", "tail", 32940, 1792, 67),
    ("IQ3_S", "ROWS96", "tail2", 17224, 2816, 159), ("IQ3_S", "ROWS64", "whole", 748, 256, 963),
    ("IQ3_S", "ROWS64", "split", 300, 5888, 811), ("IQ3_S", "ROWS64", "tail", 33288, 1280, 37),
    ("IQ3_S", "ROWS32", "whole", 2752, 256, 193), ("IQ3_S", "ROWS32", "split", 8232, 2816, 20),
    ("IQ3_S", "ROWS32", "tail", 33020, 1280, 20), ("IQ3_S", "THIN96", "whole", 460, 256, 1093),
    ("IQ3_S", "THIN96", "split", 104, 4352, 1079), ("IQ3_S", "THIN64", "whole", 228, 256, 1034),
    ("IQ3_S", "THIN64", "split", 36, 4352, 1066), ("IQ3_S", "THIN32", "whole", 36, 256, 17),
    ("IQ3_S", "THIN32", "split", 36, 2816, 18), ("IQ3_S", "THIN32", "tail", 8492, 2304, 17),
    ("Q4_0", "WIDE", "whole", 7288, 288, 1066), ("Q4_0", "WIDE", "split", 5152, 6080, 1023),
    ("Q4_0", "WIDE", "rest", 66060, 448, 129), ("Q4_0", "TALL", "whole", 4540, 800, 1013),
    ("Q4_0", "HALF", "whole", 3596, 288, 1026), ("Q4_0", "HALF", "tail", 67844, 544, 114),
    ("Q4_0", "HALF", "tail2", 8388, 1376, 897), ("Q4_0", "HALF2", "whole", 2732, 352, 1063),
    ("Q4_0", "HALF2", "split", 700, 4000, 1086), ("Q4_0", "HALF2", "tail2", 4188, 3776, 924),
    ("Q4_0", "ROWS96", "whole", 1492, 288, 903), ("Q4_0", "ROWS96", "split", 232, 4704, 1053),
    ("Q4_0", "ROWS96", "tail", 32872, 1088, 68), ("Q4_0", "ROWS96", "tail2", 3956, 4544, 1030),
    ("Q4_0", "ROWS64", "whole", 708, 288, 1072), ("Q4_0", "ROWS64", "split", 228, 4672, 1066),
    ("Q4_0", "ROWS64", "tail", 32872, 800, 44), ("Q4_0", "ROWS32", "whole", 2840, 288, 209),
    ("Q4_0", "ROWS32", "split", 2776, 5760, 17), ("Q4_0", "ROWS32", "tail", 33856, 1056, 21),
    ("Q4_0", "THIN96", "whole", 484, 288, 1031), ("Q4_0", "THIN96", "split", 68, 5184, 992),
    ("Q4_0", "THIN64", "whole", 232, 320, 1057), ("Q4_0", "THIN64", "split", 36, 4736, 1038),
    ("Q4_0", "THIN32", "whole", 36, 288, 17), ("Q4_0", "THIN32", "split", 36, 2848, 51),
    ("Q8_0", "WIDE", "whole", 8616, 288, 913), ("Q8_0", "WIDE", "split", 4168, 5856, 1027),
    ("Q8_0", "TALL", "whole", 4748, 1056, 1036), ("Q8_0", "HALF", "whole", 3732, 288, 1069),
    ("Q8_0", "HALF", "tail2", 7196, 1408, 1060), ("Q8_0", "HALF2", "whole", 2356, 288, 889),
    ("Q8_0", "HALF2", "split", 396, 5312, 1039), ("Q8_0", "HALF2", "tail2", 3944, 1120, 1052),
    ("Q8_0", "ROWS96", "whole", 2072, 288, 976), ("Q8_0", "ROWS96", "split", 264, 5504, 955),
    ("Q8_0", "ROWS96", "tail", 33580, 800, 69), ("Q8_0", "ROWS96", "tail2", 16900, 1376, 182),
    ("Q8_0", "ROWS64", "whole", 748, 288, 1043), ("Q8_0", "ROWS64", "split", 240, 4384, 1079),
    ("Q8_0", "ROWS64", "tail", 33128, 832, 49), ("Q8_0", "ROWS32", "whole", 8264, 288, 31),
    ("Q8_0", "ROWS32", "split", 8360, 1632, 18), ("Q8_0", "ROWS32", "tail", 33396, 800, 21),
    ("Q8_0", "THIN96", "whole", 556, 288, 986), ("Q8_0", "THIN96", "split", 68, 5312, 1006),
    ("Q8_0", "THIN64", "whole", 232, 288, 1092), ("Q8_0", "THIN64", "split", 40, 3936, 1066),
    ("Q8_0", "THIN32", "whole", 36, 288, 18), ("Q8_0", "THIN32", "split", 36, 2336, 43),
]


def kind_of(p):
    if p.pieces:
        return "tail2" if p.r0 > 0 and p.c0 > 0 else "tail"
    return "rest" if p.rest else "split" if p.splits > 1 else "whole"


def columns(n, bn, rng, c0=0):
    """The first and last columns, a seeded sample of all and of those from c0 on, and one in each weight
    tile of bn."""
    starts = np.arange(0, n, bn)
    inside = starts + rng.integers(0, np.minimum(bn, n - starts))
    return np.unique(np.concatenate([sample_cols(n, rng, 40), c0 + sample_cols(n - c0, rng, 40), inside]))


def worst(got, ref):
    """Normwise error by the oracle's largest output of the row's columns (a wrong output elsewhere cannot
    loosen the bar)."""
    return O.normwise_rel(got.float().cpu().numpy(), ref)


@pytest.mark.parametrize("name,config,kind,n,k,m", CASES, ids=lambda v: str(v))
def test_folded_tile(kai, name, config, kind, n, k, m):
    qtype = {v: t for t, v in O.NAMES.items()}[name]
    p = P.folded(qtype, n, k, m)
    assert (p.id, kind_of(p)) == (getattr(P, config), kind), p
    print(f"folded tile {name} {config} {kind} {n}x{k} m={m}", flush=True)
    rng = np.random.default_rng(qtype * 1000 + n + k + m)
    w = O.random_blocks(qtype, n, k, rng)
    lead = O.random_blocks(qtype, 36, k, rng)  # 72 bytes of bf16 output before the matrix's slice
    x = rng.standard_normal((m, k)).astype(np.float16)
    cols = columns(n, p.bn, rng, p.c0)
    ref = O.mmq_reference(qtype, w[cols], x, threads=16)
    x_dev, w_dev = to_dev(x), to_dev(w)
    mats = [(qtype, w, w_dev)]
    out = gpu_mmq(kai, mats, x_dev)
    assert bool(out.isfinite().all())
    assert worst(out[:, cols], ref) <= TOL_F32
    if p.pieces:
        inside = cols >= p.c0
        assert worst(out[p.r0:, cols[inside]], ref[p.r0:, inside]) <= TOL_F32
    assert torch.equal(out, gpu_mmq(kai, mats, x_dev)), "sums are added in a fixed order"
    # bf16 outputs are the same sums rounded once, in a slice of a wider output that starts off 16 bytes
    both = gpu_mmq(kai, [(qtype, lead, to_dev(lead))] + mats, x_dev, bf16=True, stride=n + 36 + 8)
    assert torch.equal(both[:, 36:n + 36], out.to(torch.bfloat16))
    assert bool(both[:, n + 36:].isnan().all())
    assert worst(both[:, :36], O.mmq_reference(qtype, lead, x)) <= TOL_BF16 + TOL_F32


# Q6_K above 80 rows on whole-number fp16 operands (kai_mmq6.cuh): each tile configuration, ragged
# weight and activation rows, fewer superblocks than K groups' turns
Q6_CASES = [("Q6_96X128", 40004, 768, 500), ("Q6_96X128_2", 7004, 768, 333), ("Q6_96X64_4", 2500, 2304, 500),
            ("Q6_64X64_4", 5004, 2304, 130), ("Q6_96X64_4", 10004, 2304, 81)]


@pytest.mark.parametrize("config,n,k,m", Q6_CASES)
@pytest.mark.parametrize("extreme", [False, True])
def test_q6_k_tile(kai, config, n, k, m, extreme):
    """extreme: scales -128 and codes -32 or 31 against activation codes of +-127, the largest block dots."""
    assert P.q6(n, k, m) == getattr(P, config)
    print(f"Q6_K tile {config} {n}x{k} m={m} extreme={extreme}", flush=True)
    rng = np.random.default_rng(n + k + m)
    w = O.random_blocks(O.Q6_K, n, k, rng)
    x = rng.standard_normal((m, k)).astype(np.float32)
    if extreme:
        b = w.reshape(n, -1, 210)
        b[:, :, 192:208] = 0x80  # every scale -128
        b[: n // 2, :, :192] = 0  # codes 0 - 32
        b[n // 2:, :, :192] = 0xff  # codes 63 - 32
        x = np.where(rng.random((m, k)) < 0.9, 1.0, -1.0).astype(np.float32)
    cols = columns(n, 64, rng)
    ref = O.mmq_reference(O.Q6_K, w[cols], x, threads=16)
    x_dev, w_dev = to_dev(x), to_dev(w)
    out = gpu_mmq(kai, [(O.Q6_K, w, w_dev)], x_dev)
    assert bool(out.isfinite().all())
    # block dots are whole numbers below 2^24: what is left are the fp32 sums over k / 32 blocks
    assert worst(out[:, cols], ref) <= 4 * (k / 32) * 2.0 ** -24
    both = gpu_mmq(kai, [(O.Q6_K, w, w_dev)], x_dev, bf16=True, stride=n + 12)
    assert worst(both[:, cols], ref) <= TOL_BF16 + TOL_F32
    assert both[:, n:].isnan().all()
