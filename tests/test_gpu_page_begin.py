"""Ranges that begin on a page but off the 64-token tile grid, more than 8
head-rows: the whole calls count their tokens from the begin (page table and
key positions included); against FP64, and against kvb_split_attention +
kvb_merge_finalize, which run the range as it is.

Bound: relative L2 1e-5 on n / l.  The rows kernel rounds weights to 2^-20 of
the largest of a scale epoch, the f16 kernel keeps 22 bits of each; over a
range of few tokens neither averages out (the per-element gate 3e-6 + 5e-5 |r|
is not reached by either there)."""
import numpy as np
import pytest
import torch

import kvbridge_amd as kvb
from kvbridge_amd import workloads as W
from oracle import oracle as O

from helpers import DeviceCase, check_against_oracle

pytestmark = pytest.mark.gpu

CASES = [
    # rows, q_heads, kv_heads, dim, page, tokens, begin, end, split, query positions
    (8, 24, 4, 256, 32, 1500, 32, 1500, 256, None),
    (8, 24, 4, 256, 32, 1500, 160, 1471, 256, [0, 159, 160, 161, 700, 1470, 1471, 5000]),
    (8, 24, 4, 256, 32, 200, 192 - 32, 192, 256, None),   # shorter than a tile
    (8, 48, 8, 128, 16, 900, 48, 899, 128, [47, 48, 100, 898, 300, -1, 899, 64]),
    (4, 24, 4, 256, 32, 1500, 1472, 1500, 512, None),     # the last page only
    (8, 24, 4, 256, 32, 1500, 96, 96, 256, None),         # empty range
]


@pytest.mark.parametrize("cfg", CASES)
def test_page_aligned_begin(gpu, cfg):
    rows, qh, kvh, d, p, t, b, e, st, qpos = cfg
    case = W.synth_case(rows, qh, kvh, d, p, t, seed=t + b, begin=b, end=e,
                        qpos=None if qpos is None else np.array(qpos, np.int64))
    dc = DeviceCase(case)
    ref = O.fp64(case, threads=8)
    mln, _, _ = dc.run_decode(st)
    def check(got, label):
        g = check_against_oracle(case, got, label, ref)
        assert g["rel_l2"] <= 1e-5, (label, g)

    check(mln, "decode")
    mma = kvb.attention_mma_supported(case.shape)
    mln2, _ = dc.run_reference_api(mma=mma)
    check(mln2, "launch_attention_mma" if mma else "launch_attention")
    scratch = dc.scratch(st)
    kvb.split_attention(case.shape, dc.inp, st, scratch)
    kvb.merge_finalize(case.shape, scratch, kvb.split_count(case.shape, st), dc.m, dc.l, dc.n)
    torch.cuda.synchronize()
    check(dc.read(), "split + merge")
