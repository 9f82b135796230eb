"""Ranges that begin off the 64-token tile grid, more than 8 head-rows: every
call that splits and merges runs the generic MFMA kernel, which takes any begin
and keeps 24 bits of every weight; against FP64 at the per-element gate 3e-6 +
5e-5 |r| of fp32 arithmetic (examples/attention_bench.cu:127).
kvb_split_attention + kvb_merge_finalize run the f16 kernel, which keeps 22 bits
(relative L2 1e-5)."""
import numpy as np
import pytest
import torch

import kvbridge_amd as kvb
from kvbridge_amd import workloads as W
from oracle import oracle as O

from helpers import DeviceCase, check_against_oracle, log
from test_gpu_fused import run_fused

pytestmark = pytest.mark.gpu

CASES = [
    # rows, q_heads, kv_heads, dim, page, tokens, begin, end, split, query positions
    (8, 24, 4, 256, 32, 1500, 32, 1500, 256, None),
    (8, 24, 4, 256, 32, 1500, 160, 1471, 256, [0, 159, 160, 161, 700, 1470, 1471, 5000]),
    (8, 24, 4, 256, 32, 200, 192 - 32, 192, 256, None),   # shorter than a tile
    (8, 48, 8, 128, 16, 900, 48, 899, 128, [47, 48, 100, 898, 300, -1, 899, 64]),
    (4, 24, 4, 256, 32, 1500, 1440, 1500, 512, None),     # the last two pages
    (8, 24, 4, 256, 32, 1500, 96, 96, 256, None),         # empty range
    (3, 24, 8, 128, 64, 700, 1, 699, 192, None),          # 9 head-rows, begin inside a page
    (16, 16, 2, 64, 16, 3000, 2032, 2999, 4096, None),    # 128 head-rows, one split
]


def assert_same(a, b, label):  # bitwise
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), label


@pytest.mark.parametrize("cfg", CASES)
def test_off_grid_begin(gpu, cfg):
    rows, qh, kvh, d, p, t, b, e, st, qpos = cfg
    case = W.synth_case(rows, qh, kvh, d, p, t, seed=t + b, begin=b, end=e,
                        qpos=None if qpos is None else np.array(qpos, np.int64))
    dc = DeviceCase(case)
    for split in (st, 256):
        assert "split_generic_i8_kernel" in kvb.selected_kernel_name(case.shape, dc.inp, split, True)
    ref = O.fp64(case, threads=8)
    mln, _, _ = dc.run_decode(st)
    check_against_oracle(case, mln, "decode", ref, strict=True)
    mma = kvb.attention_mma_supported(case.shape)
    mln2, _ = dc.run_reference_api(mma=mma)
    check_against_oracle(case, mln2, "launch_attention_mma" if mma else "launch_attention", ref, strict=True)
    scratch = dc.scratch(st)
    kvb.split_attention(case.shape, dc.inp, st, scratch)
    kvb.merge_finalize(case.shape, scratch, kvb.split_count(case.shape, st), dc.m, dc.l, dc.n)
    torch.cuda.synchronize()
    g = check_against_oracle(case, dc.read(), "split + merge", ref)
    assert g["rel_l2"] <= 1e-5, g
    counters = torch.zeros(kvh, dtype=torch.int32, device=gpu)
    assert_same(run_fused(dc, st, counters)[0], mln, "fused entry")
    assert torch.count_nonzero(counters).item() == 0


@pytest.mark.parametrize("ratio", [2.0 ** 7, 2.0 ** 20, 2.0 ** 30])
@pytest.mark.parametrize("what", ["plain_weight", "one_channel"])
def test_off_grid_begin_over_wide_v_scales(gpu, what, ratio):
    """A token whose v-scale is `ratio` times the others' takes no bits from
    them, also where it has codes in one channel only (left out of the
    comparison): 1e-6 of each head-row's norm against FP64."""
    case = W.synth_case(8, 24, 4, 256, 32, 1500, seed=3, begin=32)
    pg, sl, keep = int(case.table[123 // 32]), 123 % 32, np.ones(256, bool)
    case.vs[pg, :, sl] *= np.float32(ratio)
    if what == "one_channel":
        case.v[pg, :, :, sl] = 0
        case.v[pg, :, 9, sl] = 127
        keep[9] = False
    dc = DeviceCase(case)
    (m, l, n), _ = dc.run_reference_api(mma=True)
    ref = O.fp64(case, threads=8)[0].reshape(-1, 256)[:, keep]
    got = (n.reshape(-1, 256).astype(np.float64) / l[:, None].astype(np.float64))[:, keep]
    err = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)
    log(f"  {what} ratio={ratio:.1e}: largest error {err.max():.2e}")
    assert err.max() <= 1e-6


@pytest.mark.parametrize("what", ["v_nan", "v_inf", "k_nan", "q_nan", "v_nan_masked"])
def test_off_grid_begin_keeps_non_finite_values(gpu, what):
    """A NaN or infinity of Q or a scale reaches exactly the outputs that see
    it; a masked one reaches none."""
    qpos = np.array([1499] * 4 + [1000] * 4, np.int64)
    case = W.synth_case(8, 24, 4, 256, 32, 1500, seed=4, begin=32, qpos=qpos)
    tok = 1200 if what != "v_nan_masked" else 20  # past the last four rows; before begin
    pg, sl = int(case.table[tok // 32]), tok % 32
    if what == "q_nan":
        case.q.reshape(8, 24, 256)[0, 5, 11] = np.nan
    elif what == "k_nan":
        case.ks[pg, 1, sl] = np.nan
    else:
        case.vs[pg, 1, sl] = np.inf if what == "v_inf" else np.nan
    dc = DeviceCase(case)
    (m, l, n), _ = dc.run_reference_api(mma=True)
    bad = np.zeros((8, 24), bool)
    if what == "q_nan":
        bad[0, 5] = True
    elif what != "v_nan_masked":
        bad[:4, 6:12] = True  # kv head 1's group, rows that see the token
    n_bad = ~np.isfinite(n.reshape(8, 24, 256))
    assert np.array_equal(n_bad.any(2), bad) and np.array_equal(n_bad.all(2), bad)
    assert np.array_equal(~np.isfinite(l.reshape(8, 24)), bad if what in ("q_nan", "k_nan") else np.zeros_like(bad))
