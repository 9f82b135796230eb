"""The order in which a batched grid takes its splits (live ones first):
batches below and above one, two and four rounds of 64 sequences, and above
the packed limit, with empty sequences and one-split sequences among them;
every sequence against the single-sequence call on the same data and the split
partials past a sequence's end empty.

Tolerance 5e-5 of the largest magnitude: a grid above 512 work-groups runs
another chunk length than the single call, and each rounds its weights to
2^-21 of its chunk's largest (at most 700 of them in a sum)."""
import numpy as np
import pytest

import kvbridge_amd as kvb
from kvbridge_amd import workloads as W

from helpers import DeviceCase, log
from test_gpu_batched import DeviceBatch, seq_slice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("page,dim", [(64, 64), (64, 80)])
@pytest.mark.parametrize("batch", [3, 63, 64, 65, 130, 256, 257])
def test_batch_order(gpu, batch, page, dim):
    rng = np.random.default_rng(batch)
    lengths = [int(x) for x in rng.integers(0, 700, size=batch)]
    lengths[0], lengths[-1] = 0, 700
    st = 64 if batch == 3 else 128
    bc = W.synth_batch(1, 8, 4, dim, page, lengths, seed=batch, split_tokens=st)
    db = DeviceBatch(bc.shape, bc.to_device("cuda:0"))
    log(f"batch={batch} kernel={kvb.batch_kernel_name(bc.shape, db.inp)}")
    m, l, n, _ = db.run(fused=False)
    splits = kvb.batch_split_count(bc.shape)
    parts = db.scratch.cpu().numpy().reshape(batch, 8, splits, dim + 2)
    for b in sorted({0, 1, batch // 2, batch - 2, batch - 1}):
        sl, t = seq_slice(bc.shape, b), bc.lengths[b]
        own = max(1, -(-t // st))
        assert np.all(np.isneginf(parts[b, :, own:, 0])) and np.all(parts[b, :, own:, 1:] == 0), b
        if t == 0:
            assert np.all(np.isneginf(m[sl])) and np.all(l[sl] == 0)
            continue
        m1, l1, n1 = DeviceCase(bc.sequence(b)).run_decode(st)[0]
        for x, y in ((m[sl], m1), (l[sl], l1), (n.reshape(-1, dim)[sl].ravel(), n1)):
            np.testing.assert_allclose(x, y, rtol=0, atol=5e-5 * np.abs(y).max(), err_msg=str(b))
