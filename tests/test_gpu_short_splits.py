"""The int8 split kernel's one-tile chunks and the single launch's rule at
their edges: splits of 1, 4, 5, 8, 15 and 16 tiles, 1 / 4 / 8 head-rows, both
page paths, ragged and causal ends, against FP64 (the per-element gate
3e-6 + 5e-5 |r|), and the single-launch entry against the two-launch one."""
import zlib

import numpy as np
import pytest

import kvbridge_amd as kvb
from kvbridge_amd import workloads as W
from oracle import oracle as O

from helpers import DeviceCase, check_against_oracle, log
from test_gpu_batched import DeviceBatch, check_sequence_vs_oracle
from test_gpu_fused import run_fused

pytestmark = pytest.mark.gpu

SHAPES = [
    # rows, q_heads, kv_heads, dim, page, tokens, begin, split, query position
    (1, 8, 2, 64, 16, 130, 0, 64, None),       # one tile per split: waves without tiles
    (1, 8, 2, 64, 64, 2000, 7, 256, [1500]),   # four tiles, ragged begin, causal cut
    (1, 32, 8, 128, 64, 2500, 0, 320, None),   # five tiles: eight waves, two launches
    (1, 16, 4, 128, 32, 4000, 0, 512, [3333]),  # eight tiles, small grid: single launch, eight waves
    (1, 8, 8, 128, 64, 9000, 0, 960, None),    # fifteen tiles
    (1, 8, 8, 128, 64, 9000, 0, 1024, None),   # sixteen: chunks of four tiles again
    (2, 8, 2, 128, 64, 1500, 0, 256, [1499, 20]),  # 8 head-rows, four waves
    (1, 16, 2, 64, 16, 2000, 0, 576, None),    # 8 head-rows, nine tiles
    (1, 8, 8, 128, 64, 26600, 0, 832, None),   # thirteen tiles, 256 work-groups: single launch
    (1, 4, 4, 256, 64, 1200, 0, 256, None),    # dim 256, one head-row: single launch
    (1, 8, 2, 256, 32, 1200, 0, 512, None),    # dim 256, four head-rows: two launches
    (3, 32, 8, 256, 64, 4136, 0, 128, None),   # rows kernel: 264 work-groups, the last of a head short
    (3, 32, 8, 256, 64, 4224, 0, 128, [4000, 9, 4223]),  # the same, all full: two splits per work-group
    (8, 32, 8, 128, 64, 8500, 0, 256, None),   # dim 128, 272 work-groups
]


@pytest.mark.parametrize("cfg", SHAPES)
def test_short_splits(gpu, cfg):
    import torch

    rows, qh, kvh, d, p, t, b, st, qpos = cfg
    case = W.synth_case(rows, qh, kvh, d, p, t, seed=zlib.crc32(repr(cfg).encode()) & 0xFFFF, begin=b, qpos=qpos)
    dc = DeviceCase(case)
    log(f"short shape={case.shape.as_tuple()} split_tokens={st} "
        f"kernel={kvb.selected_kernel_name(case.shape, dc.inp, st)} "
        f"fused={kvb.selected_kernel_name(case.shape, dc.inp, st, True)}")
    ref = O.fp64(case, threads=8)
    mln, _, _ = dc.run_decode(st)
    check_against_oracle(case, mln, "decode", ref, strict=True)
    counters = torch.zeros(kvh, dtype=torch.int32, device=gpu)
    one, _ = run_fused(dc, st, counters)
    check_against_oracle(case, one, "fused", ref, strict=True)
    assert torch.count_nonzero(counters).item() == 0
    assert np.array_equal(one[0], mln[0])


def test_single_launch_rule(gpu):
    fake = kvb.device_input(*([0x1000] * 8))

    def fused(kv_heads, group, dim, tokens, split):
        s = kvb.make_shape(1, kv_heads * group, kv_heads, dim, 64, 4096, tokens, 0, tokens, 0.1)
        name = kvb.selected_kernel_name(s, fake, split, True)
        return name.split(",")[5] == "true"

    assert fused(2, 4, 64, 8192, 256) and fused(8, 4, 128, 4096, 512) and fused(8, 4, 128, 65536, 2048)
    assert not fused(8, 4, 128, 2048, 256) and not fused(8, 1, 128, 8192, 256)  # too many outputs / work-groups
    assert not fused(2, 4, 64, 4096, 64) and not fused(2, 8, 64, 65536, 2048)   # 64 splits / 8 head-rows
    # one head-row over 256 work-groups: from 13 tiles
    assert fused(8, 1, 128, 26600, 832) and not fused(8, 1, 128, 24500, 768) and not fused(8, 4, 128, 26600, 832)


@pytest.mark.parametrize("head_rows", [1, 3, 4])
@pytest.mark.parametrize("dim,split", [(64, 512), (128, 256), (128, 2048), (256, 320), (256, 1024)])
def test_lone_splits(gpu, dim, split, head_rows):
    """Sequences of at most one split are one launch at any dim and up to four
    head-rows, without a ticket: against the two launches, an empty sequence
    and a row that sees nothing among them, and against FP64."""
    bc = W.synth_batch(1, 2 * head_rows, 2, dim, 64, [split, 0, 1, split - 37, 200], seed=dim + head_rows,
                       split_tokens=split)
    bc.qpos[4] = -1
    db = DeviceBatch(bc.shape, bc.to_device("cuda:0"))
    assert kvb.batch_kernel_name(bc.shape, db.inp, True).split(",")[5] == "true"
    db.counters.fill_(0)
    one, two = db.run(fused=True), db.run(fused=False)
    for x, y, nm in zip(one, two, ("m", "l", "n", "out")):
        np.testing.assert_allclose(x, y, rtol=2e-6, atol=2e-6 * max(1.0, np.abs(y[np.isfinite(y)]).max()), err_msg=nm)
    for b in (0, 1, 2, 3):
        check_sequence_vs_oracle(bc, b, *one[:3], f"seq {b}")
    rows = slice(4 * 2 * head_rows, 5 * 2 * head_rows)
    assert np.isneginf(one[0][rows]).all() and not one[1][rows].any() and not one[3][rows].any()
