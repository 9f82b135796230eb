"""The generic family's MFMA kernels (fp32 KV, any dim that is a multiple of
4, 16-token page groups) against the FP64 oracle, and against the scalar
kernel on values a matrix product treats differently.

Tolerance: the per-element gate |a - r| <= 3e-6 + 5e-5 |r| of fp32 arithmetic
(examples/attention_bench.cu:127), as for the scalar kernel."""
import zlib

import numpy as np
import pytest

import kvbridge_amd as kvb
from kvbridge_amd import workloads as W
from oracle import oracle as O

from helpers import DeviceCase, check_against_oracle, log
from test_gpu_batched import DeviceBatch, check_sequence_vs_oracle

pytestmark = pytest.mark.gpu

SHAPES = [
    # rows, q_heads, kv_heads, dim, page, tokens, begin, end, split, int8, query positions
    (1, 4, 4, 4, 16, 200, 0, 200, 64, True, None),           # smallest dim; one wave per split
    (1, 8, 2, 60, 16, 700, 3, 690, 128, True, None),         # padded 64-dim step, ragged range
    (1, 8, 2, 68, 48, 1000, 17, 999, 256, True, None),       # just past a padded size, 48-token pages
    (1, 17, 1, 72, 32, 900, 0, 900, 512, True, None),        # 17 head-rows: two blocks
    (4, 16, 4, 112, 64, 1500, 0, 1500, 512, True, [100, 1400, -1, 777]),  # rows cut anywhere, one sees nothing
    (1, 32, 8, 132, 16, 600, 0, 600, 256, True, None),       # four-wave instances
    (1, 24, 4, 252, 16, 1100, 0, 1100, 1024, True, None),
    (1, 8, 2, 96, 16, 20000, 0, 20000, 20000, True, None),   # one split of 313 tiles: several row windows
    (3, 24, 8, 128, 64, 1500, 0, 1500, 256, True, [1499, 3, 700]),  # 9 head-rows of a tiled shape
    (1, 10, 2, 64, 32, 3000, 0, 2990, 960, True, [2500]),    # 5 head-rows, fifteen tiles
    (2, 16, 4, 128, 64, 1500, 33, 1500, 256, True, [1400, 900]),  # 8 head-rows in two rows
    (4, 16, 4, 64, 16, 1500, 5, 1490, 320, True, None),      # 16 head-rows, off-tile begin
    (2, 64, 8, 128, 32, 3000, 0, 3000, 1000, True, None),    # off-tile splits
    (1, 4, 4, 4, 16, 200, 0, 200, 64, False, None),
    (1, 8, 2, 64, 16, 700, 5, 695, 128, False, None),
    (1, 16, 1, 100, 48, 1000, 0, 1000, 256, False, None),
    (4, 16, 4, 128, 32, 1500, 33, 1500, 512, False, [100, 1400, -1, 777]),
    (1, 24, 4, 256, 64, 1100, 0, 1100, 512, False, None),
    (2, 20, 2, 132, 16, 300, 0, 300, 512, False, None),      # 20 head-rows
    (1, 8, 2, 64, 16, 9000, 0, 9000, 9000, False, None),     # one split of 563 tiles
]


@pytest.mark.parametrize("cfg", SHAPES)
def test_generic_mfma_shapes(gpu, cfg):
    rows, qh, kvh, d, p, t, b, e, st, int8, qpos = cfg
    seed = zlib.crc32(repr(cfg).encode()) & 0xFFFF
    case = W.synth_case(rows, qh, kvh, d, p, t, seed=seed, begin=b, end=e, int8=int8,
                        qpos=None if qpos is None else np.array(qpos, np.int64))
    dc = DeviceCase(case)
    name = kvb.selected_kernel_name(case.shape, dc.inp, st)
    log(f"generic mfma shape={case.shape.as_tuple()} split_tokens={st} kernel={name}")
    assert ("split_generic_i8_kernel" if int8 else "split_generic_f32_kernel") in name
    ref = O.fp64(case, threads=8)
    mln, _, _ = dc.run_decode(st)
    check_against_oracle(case, mln, "decode", ref, strict=True)
    again, _, _ = dc.run_decode(st)
    for x, y in zip(mln, again):  # bitwise repeatable
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("dim", [64, 96, 128, 192, 252])
def test_generic_int8_scores_round_little(gpu, dim):
    """m and l of the int8 MFMA kernel against FP64.  One rounding to fp32 has
    a relative rms of 2^-25 / sqrt(3) .. 2^-24 / sqrt(3), 2.4e-8 over the
    mantissas.  A score takes the rounding of its product with the k-scale, of
    Q times the scale (less: it averages out over the elements) and of the sums
    of the high pieces (the products are short: at most three in effect), so m
    is within 2.4e-8 * sqrt(6) = 6e-8; l = sum of e^(score - m) carries m's own
    absolute error (m is about 4) to 2.4e-7."""
    err = []
    for seed in (1, 2, 3, 4):
        case = W.synth_case(4, 32, 8, dim, 16, 4000, seed=seed)
        s = case.shape
        dc = DeviceCase(case)
        assert "split_generic_i8_kernel" in kvb.selected_kernel_name(s, dc.inp, 256)
        m, l, _ = dc.run_decode(256)[0]
        tok = np.arange(s.tokens)
        pg, sl = case.table[tok // 16].astype(np.int64), tok % 16
        k = case.k[pg, :, sl].astype(np.float64) * case.ks[pg, :, sl].astype(np.float64)[..., None]  # [t, kv, dim]
        q = case.q.reshape(4, 8, 4, dim).astype(np.float64)
        score = np.einsum("rhgd,thd->rhgt", q, k) * np.float64(np.float32(s.scale))
        score[np.broadcast_to((case.kpos[None, :] > case.qpos[:, None])[:, None, None, :], score.shape)] = -np.inf
        top = score.max(-1)
        ref = top.ravel(), np.exp(score - top[..., None]).sum(-1).ravel()
        err.append([np.linalg.norm(x - r) / np.linalg.norm(r) for x, r in zip((m, l), ref)])
    em, el = np.mean(err, axis=0)
    log(f"  dim {dim}: m {em:.2e} l {el:.2e}")
    assert em <= 6e-8 and el <= 2.4e-7


BATCHES = [
    # rows, q_heads, kv_heads, dim, page, lengths, split, int8
    (1, 32, 8, 128, 48, [300, 0, 1, 1000, 64], 256, True),
    (4, 32, 8, 128, 64, [500, 129, 2], 256, True),      # 16 head-rows
    (3, 24, 4, 256, 32, [200, 777], 128, True),         # 18 head-rows
    (1, 8, 2, 80, 16, [100, 4000, 33] * 20, 64, True),  # many work-groups
    (1, 8, 2, 64, 16, [300, 0, 17, 1000], 128, False),
    (1, 64, 8, 128, 64, [300, 0, 17, 1000], 256, True),  # 8 head-rows of a tiled shape
]


@pytest.mark.parametrize("cfg", BATCHES)
def test_generic_mfma_batches(gpu, cfg):
    rows, qh, kvh, d, p, lengths, st, int8 = cfg
    seed = zlib.crc32(repr(cfg).encode()) & 0xFFFF
    bc = W.synth_batch(rows, qh, kvh, d, p, lengths, seed=seed, split_tokens=st, int8=int8)
    db = DeviceBatch(bc.shape, bc.to_device("cuda:0"))
    log(f"generic batch shape={bc.shape.as_tuple()} kernel={kvb.batch_kernel_name(bc.shape, db.inp)}")
    m, l, n, _ = db.run(fused=False)
    for b, t in enumerate(bc.lengths):
        g = check_sequence_vs_oracle(bc, b, m, l, n, f"seq {b} (T={t})")
        assert g is None or g["strict_pass"], (b, g)


def _repage(case, page):
    """The same tokens in pages of `page` slots (identity page table)."""
    s = case.shape
    tok = np.arange(s.tokens)
    pg, sl = case.table[tok // s.page_tokens].astype(np.int64), tok % s.page_tokens
    pages = -(-s.tokens // page)

    def lay(rows, fill):  # [tokens, kv, ...] -> [pages, kv, page, ...]
        out = np.full((pages * page,) + rows.shape[1:], fill, rows.dtype)
        out[:s.tokens] = rows
        return np.ascontiguousarray(np.moveaxis(out.reshape((pages, page) + rows.shape[1:]), 1, 2))

    k = lay(case.k[pg, :, sl], 0)
    v = np.ascontiguousarray(np.swapaxes(lay(case.v[pg, :, :, sl], 0), 2, 3))
    ks, vs = lay(case.ks[pg, :, sl], 1), lay(case.vs[pg, :, sl], 1)
    shape = s.copy(page_tokens=page, pages=pages)
    return W.Case(shape, case.q, case.qpos, case.kpos, np.arange(pages, dtype=np.uint32), k, v, ks, vs)


NON_FINITE = ["v_inf_zero_weight", "v_nan_masked", "k_nan", "k_inf", "q_nan", "scale_nan", "scale_inf_masked"]


@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("what", NON_FINITE)
def test_non_finite_values_match_the_scalar_kernel(gpu, what, int8):
    """Infinities and NaN in Q, the cache or the scales: the same places are
    non-finite as in the scalar kernel (which the same tokens in pages of 8
    slots reach), and everything else agrees to fp32 rounding."""
    case = W.synth_case(1, 8, 2, 96, 16, 400, seed=5, permute=True, int8=int8, qpos=[370])
    tok = {"v_nan_masked": 380, "scale_inf_masked": 390}.get(what, 123)
    pg, sl = int(case.table[tok // 16]), tok % 16
    if what.startswith("v_"):
        if int8:
            case.vs[pg, 0, sl] = np.inf if what == "v_inf_zero_weight" else np.nan
        else:
            case.v[pg, 0, 5, sl] = np.inf if what == "v_inf_zero_weight" else np.nan
        if what == "v_inf_zero_weight":  # a score far below the maximum: the weight underflows to 0
            if int8:
                case.ks[pg, 0, sl] *= np.float32(1e6)
            else:
                case.k[pg, 0, sl] *= np.float32(1e6)
    elif what == "k_nan" or what == "k_inf":
        bad = np.float32(np.nan if what == "k_nan" else np.inf)
        if int8:
            case.ks[pg, 0, sl] = bad
        else:
            case.k[pg, 0, sl, 7] = bad
    elif what == "q_nan":
        case.q[2 * 96 + 11] = np.nan
    elif what == "scale_nan":
        case.vs[pg, 0, sl] = np.nan
    else:
        case.ks[pg, 0, sl], case.vs[pg, 0, sl] = np.inf, np.nan
    other = _repage(case, 8)
    a, b = DeviceCase(case), DeviceCase(other)
    name_a = kvb.selected_kernel_name(case.shape, a.inp, 128)
    assert "_kernel<128" in name_a and ":" not in kvb.selected_kernel_name(other.shape, b.inp, 128)
    for x, y, nm in zip(a.run_decode(128)[0], b.run_decode(128)[0], "mln"):
        assert np.array_equal(np.isnan(x), np.isnan(y)) and np.array_equal(np.isinf(x), np.isinf(y)), nm
        fin = np.isfinite(y)
        log(f"  {what} int8={int8} {nm}: {np.count_nonzero(~fin)} non-finite")
        if fin.any():
            np.testing.assert_allclose(x[fin], y[fin], rtol=5e-5, atol=3e-6 * max(1.0, np.abs(y[fin]).max()))


@pytest.mark.parametrize("dim,tokens,rows", [(4, 64 * 128, 1), (60, 3 * 128, 1), (68, 17 * 128, 2), (96, 64 * 128, 1),
                                             (252, 33 * 128, 1), (96, 65 * 128, 1)])
def test_padded_merge(gpu, dim, tokens, rows):
    """Merges of dims between the powers of two: 1 .. 64 splits through the
    padded merge, 65 through the scalar one, the last splits empty; against
    the oracle's merge of the same partials (fp32, other order of the sums)."""
    case = W.synth_case(rows, 8, 2, dim, 16, tokens, seed=dim, qpos=[tokens // 2] * rows)
    dc = DeviceCase(case)
    (m, l, n), out, sc = dc.run_decode(128)
    parts = sc.cpu().numpy()
    m_ref, l_ref, n_ref = O.merge_fp32(case.shape, parts, tokens // 128)
    assert np.array_equal(m, m_ref)
    np.testing.assert_allclose(l, l_ref, rtol=1e-5)
    np.testing.assert_allclose(n, n_ref, rtol=1e-5, atol=1e-5 * np.abs(n_ref).max())
    np.testing.assert_allclose(out.ravel(), (n.reshape(-1, dim) / l[:, None]).ravel(), rtol=1e-6)


@pytest.mark.parametrize("splits", [3, 64, 65])
@pytest.mark.parametrize("dim", [60, 96, 252])
def test_merge_leaves_non_finite_splits_out(gpu, dim, splits):
    """L and N are sums over the splits with l_j > 0: a split whose l is NaN
    (NaN of Q or of a K scale) reaches neither them nor the output, at 64
    splits or fewer (padded merge) as above (scalar merge)."""
    import torch

    rng = np.random.default_rng(dim + splits)
    s = W.synth_case(1, 8, 2, dim, 16, 64 * splits, seed=1).shape
    parts = rng.standard_normal((8, splits, dim + 2)).astype(np.float32)
    parts[..., 1] = rng.uniform(1, 60, (8, splits))
    parts[0, 0, 1:] = np.nan           # the split that lanes past the last one read
    parts[1, splits - 1, 1:] = np.nan
    parts[2, :, 1:] = np.nan           # no split is left
    parts[3, 1, 0], parts[3, 1, 1:] = -np.inf, 0.0
    parts[4, 1, 1] = np.inf
    good = (parts[..., 1] > 0)
    top = parts[..., 0].astype(np.float64).max(1)
    f = np.where(good, np.exp(parts[..., 0].astype(np.float64) - top[:, None]), 0.0)
    l_ref = np.where(good, f * parts[..., 1], 0.0).sum(1)
    n_ref = np.where(good[..., None], f[..., None] * parts[..., 2:], 0.0).sum(1)
    sc = torch.from_numpy(parts).cuda()
    m, l, n, out = (torch.empty(k, device="cuda") for k in (8, 8, 8 * dim, 8 * dim))
    kvb.merge_finalize(s, sc, splits, m, l, n, out, kvb.KVB_OUT_F32)
    torch.cuda.synchronize()
    assert np.array_equal(m.cpu().numpy(), top.astype(np.float32))
    np.testing.assert_allclose(l.cpu().numpy(), l_ref, rtol=1e-5)
    np.testing.assert_allclose(n.cpu().numpy().reshape(8, dim), n_ref, rtol=1e-5, atol=1e-5 * np.abs(n_ref).max())
    o_ref = np.where(l_ref[:, None] > 0, n_ref / np.where(l_ref > 0, l_ref, 1.0)[:, None], 0.0)
    np.testing.assert_allclose(out.cpu().numpy().reshape(8, dim), o_ref, rtol=1e-5, atol=1e-5 * np.abs(o_ref).max())


SMALL_PAGE_BATCHES = [
    # kv_heads, group, page, lengths, split
    (8, 4, 16, [300, 0, 1, 1000, 64, 777], 256),          # short splits, small grid
    (8, 4, 32, [5000, 1024, 2047], 1024),                 # 16 tiles
    (4, 3, 16, [130, 4000, 33, 0, 64] * 12, 256),         # four tiles, large grid
    (8, 1, 32, [100, 4000, 1500, 513] * 5, 512),          # eight tiles, large grid
    (8, 2, 16, [70000, 12], 2112),                        # 33 tiles, page window outrun
]


@pytest.mark.parametrize("cfg", SMALL_PAGE_BATCHES)
def test_small_page_batches(gpu, cfg):
    """Batches over 16- and 32-token pages are held to fp32 accuracy: error
    against FP64 at most 1e-6 of each head-row's largest numerator (two fp32
    roundings per partial and merge step)."""
    kvh, group, p, lengths, st = cfg
    bc = W.synth_batch(1, kvh * group, kvh, 128, p, lengths, seed=kvh * group + p, split_tokens=st)
    db = DeviceBatch(bc.shape, bc.to_device("cuda:0"))
    name = kvb.batch_kernel_name(bc.shape, db.inp)
    log(f"small-page batch shape={bc.shape.as_tuple()} kernel={name}")
    assert ": split_generic_i8_kernel<128," in name
    m, l, n, _ = db.run(fused=False)
    for b in range(min(6, len(lengths))):
        g = check_sequence_vs_oracle(bc, b, m, l, n, f"seq {b}")
        if g is None:
            continue
        ref, _ = O.fp64(bc.sequence(b), threads=8)
        sl = slice(b * kvh * group, (b + 1) * kvh * group)
        got = n.reshape(-1, 128)[sl].astype(np.float64) / l[sl, None].astype(np.float64)
        err = np.abs(got - ref.reshape(got.shape)).max(1) / np.abs(ref.reshape(got.shape)).max(1)
        assert g["strict_pass"] and err.max() <= 1e-6, (b, err.max())


SPREADS = ["zero_weight", "plain_weight", "full_weight", "one_channel", "q_outlier"]


@pytest.mark.parametrize("ratio", [2.0 ** 7, 2.0 ** 12, 2.0 ** 20, 2.0 ** 30, 1e12])
@pytest.mark.parametrize("page,split", [(16, 256), (32, 1024)])
@pytest.mark.parametrize("what", SPREADS)
def test_small_page_batches_over_wide_magnitudes(gpu, what, page, split, ratio):
    """One visible token whose v-scale is `ratio` times the others' must not
    take bits from them, whatever its weight (zero_weight: the weight
    underflows; full_weight: it has nearly all of it) and also where its codes
    are zero (one_channel: every channel but one, which is left out of the
    comparison); nor may one element of Q that meets only zero codes.  Same
    bound as test_small_page_batches: each weight and each element of Q keeps
    its own 24 bits."""
    bc = W.synth_batch(1, 8, 2, 128, page, [700, 30], seed=11, split_tokens=split)
    pg, sl = int(bc.table[int(bc.page_offsets[0]) + 123 // page]), 123 % page
    q = bc.q.reshape(-1, 8, 128)[0]
    keep = np.ones(128, bool)
    if what == "q_outlier":
        bc.q.reshape(-1, 8, 128)[0, :, 5] = np.float32(ratio)
        bc.k[..., 5] = 0
    else:
        bc.vs[pg, :, sl] *= np.float32(ratio)
    if what in ("zero_weight", "full_weight"):  # along the mean query of the kv head's four head-rows, or against it
        mean = q.reshape(2, 4, 128).mean(1)
        code = np.rint(mean / np.abs(mean).max(1, keepdims=True) * 127).astype(np.int8)
        bc.k[pg, :, sl] = -code if what == "zero_weight" else code
        bc.ks[pg, :, sl] = np.float32(3.0 if what == "zero_weight" else 0.1)
    elif what == "one_channel":
        bc.v[pg, :, :, sl] = 0
        bc.v[pg, :, 9, sl] = 127
        keep[9] = False
    db = DeviceBatch(bc.shape, bc.to_device("cuda:0"))
    log(f"wide magnitudes {what} page={page} split={split} ratio={ratio:.1e} "
        f"kernel={kvb.batch_kernel_name(bc.shape, db.inp)}")
    m, l, n, _ = db.run(fused=False)
    ref = O.fp64(bc.sequence(0), threads=8)[0].reshape(8, 128)[:, keep]
    got = (n.reshape(-1, 128)[:8].astype(np.float64) / l[:8, None].astype(np.float64))[:, keep]
    err = np.abs(got - ref).max(1) / np.abs(ref).max(1)
    log(f"  largest error {err.max():.2e}")
    assert err.max() <= 1e-6, err


OUT_OF_RANGE = NON_FINITE + ["q_inf", "v_scale_tiny", "q_tiny", "v_scale_huge"]


@pytest.mark.parametrize("split", [128, 512, 1024])  # one and two tiles per wave, and more
@pytest.mark.parametrize("what", OUT_OF_RANGE)
def test_small_page_batches_on_extreme_values(gpu, what, split):
    """Infinities, NaN and extreme magnitudes: as the scalar kernel, which the
    same tokens in pages of 8 slots reach."""
    bc = W.synth_batch(1, 8, 2, 128, 16, [400, 30], seed=9, split_tokens=split)
    bc.qpos[0] = 370
    tok = {"v_nan_masked": 380, "scale_inf_masked": 390}.get(what, 123)
    pg, sl = int(bc.table[int(bc.page_offsets[0]) + tok // 16]), tok % 16
    if what == "v_inf_zero_weight":
        bc.vs[pg, 0, sl] = np.inf
        bc.ks[pg, 0, sl] *= np.float32(1e6)
    elif what in ("v_nan_masked", "scale_nan"):
        bc.vs[pg, 0, sl] = np.nan
    elif what in ("k_nan", "k_inf"):
        bc.ks[pg, 0, sl] = np.nan if what == "k_nan" else np.inf
    elif what in ("q_nan", "q_inf"):
        bc.q[2 * 128 + 11] = np.nan if what == "q_nan" else np.inf
    elif what == "scale_inf_masked":
        bc.ks[pg, 0, sl], bc.vs[pg, 0, sl] = np.inf, np.nan
    elif what == "v_scale_tiny":
        bc.vs *= np.float32(2.0 ** -100)
    elif what == "v_scale_huge":
        bc.vs[pg, 0, sl] = np.float32(2.0 ** 126.5)
    else:  # scores of ordinary size from tiny queries
        bc.q *= np.float32(2.0 ** -100)
        bc.ks *= np.float32(2.0 ** 100)
    db = DeviceBatch(bc.shape, bc.to_device("cuda:0"))
    assert ": split_generic_i8_kernel<128," in kvb.batch_kernel_name(bc.shape, db.inp)
    other = _repage(bc.sequence(0), 8)
    dc = DeviceCase(other)
    assert ":" not in kvb.selected_kernel_name(other.shape, dc.inp, split)
    got = [x[:size] for x, size in zip(db.run(fused=False)[:3], (8, 8, 8 * 128))]
    for x, y, nm in zip(got, dc.run_decode(split)[0], "mln"):
        assert np.array_equal(np.isnan(x), np.isnan(y)) and np.array_equal(np.isinf(x), np.isinf(y)), nm
        fin = np.isfinite(y)
        log(f"  {what} split={split} {nm}: {np.count_nonzero(~fin)} non-finite")
        if fin.any():
            np.testing.assert_allclose(x[fin], y[fin], rtol=5e-5, atol=3e-6 * np.abs(y[fin]).max())
