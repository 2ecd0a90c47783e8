"""Decode work split and merge chosen by the batch: the host's table of work
items against the kernel's scan (more than 256 sequences), the in-kernel merge
of ragged launches against the combine kernel, and sequences shorter than a
workgroup's waves, against the oracle (2e-3 abs + 1e-2 rel)."""
import numpy as np
import pytest

import smallaios_amd as S
from _gpu_util import Case, assert_close, err_tol_ratio, log

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    import torch
    assert torch.cuda.is_available()
    r = S.Runtime(0)
    yield r
    r.close()


CASES = [
    # quant, hq, hkv, d, past lengths, window, launches (1: merged in-kernel)
    (S.KV_INT8, 8, 2, 128, [0, 19, 63, 64, 700, 1500], 0, 1),
    (S.KV_INT8, 8, 1, 256, [1100, 3, 300], 0, 1),
    (S.KV_INT8, 4, 4, 64, [520, 2000, 1], 600, 1),
    (S.KV_INT8, 8, 8, 168, [900, 100], 0, 1),
    (S.KV_INT4, 8, 2, 128, [0, 1300, 64, 2100], 0, 1),
    (S.KV_INT4, 2, 2, 64, [2500, 700, 15], 0, 1),
    (S.KV_INT8, 8, 1, 128, [9000, 8700], 0, 2),   # 17 and more splits: the combine kernel
    (S.KV_INT4, 8, 1, 64, [9000, 600], 0, 2),
]


@pytest.mark.parametrize("case", CASES, ids=[f"case{i}" for i in range(len(CASES))])
def test_decode_ragged_merges(rt, case):
    """The automatic merge, and both merges forced: each within tolerance of
    the oracle, repeated calls bit-identical, and the two merges within a few
    f32 roundings of each other."""
    quant, hq, hkv, d, past, window, launches = case
    log(f"decode ragged merges: quant {quant} hq {hq} hkv {hkv} d {d} past {past}")
    c = Case(rt, 0x5D1 + d + len(past), len(past), hq, hkv, d, past, 1, theta=5e5, quant=quant,
             permute_pages=True)
    c.step_kv()
    q = c.query("f32")
    ref = c.oracle_attend(q, mask_window=window)
    got = c.gpu_decode(q, window=window)
    assert rt.last_decode_launches() == launches
    log(f"  worst err/tol {err_tol_ratio(got, ref):.4f}")
    assert_close(got, ref, "ragged decode")
    assert np.array_equal(got, c.gpu_decode(q, window=window))
    prev = rt.set_decode_merge(0)
    try:
        a = c.gpu_decode(q, window=window)
        rt.set_decode_merge(1)
        b = c.gpu_decode(q, window=window)
    finally:
        rt.set_decode_merge(prev)
    # both merge the same partials in f32 in split order: a few roundings of
    # weights <= 1 on outputs bounded by max|v| < 6
    assert np.abs(a - b).max() <= 64 * 2.0 ** -24 * 6


@pytest.mark.parametrize("quant,hq,hkv,d", [
    (S.KV_INT8, 1, 1, 64), (S.KV_INT8, 4, 1, 64), (S.KV_INT8, 4, 2, 128), (S.KV_INT8, 4, 1, 128),
    (S.KV_INT8, 2, 2, 168), (S.KV_INT8, 1, 1, 256), (S.KV_INT4, 2, 2, 64), (S.KV_INT4, 8, 1, 64),
    (S.KV_INT4, 4, 1, 128), (S.KV_INT4, 8, 1, 128), (S.KV_INT4, 1, 1, 256), (S.KV_INT4, 2, 1, 256)])
def test_decode_merge_split_counts(rt, quant, hq, hkv, d):
    """The in-kernel merge over 2 to 17 splits, where its loads' width and its
    path change (an entry or a pair of dims per thread; heads x head_dim below,
    at and above a workgroup's threads): against the oracle, and within a few
    f32 roundings of the combine kernel's merge of the same partials."""
    prev_split, prev_merge = rt.set_decode_split(64), rt.set_decode_merge(1)
    try:
        for n in (2, 3, 4, 5, 8, 9, 16, 17):
            log(f"decode merge: quant {quant} hq {hq} hkv {hkv} d {d} splits {n}")
            past = [64 * n - 1, 64 * n - 64]  # the second's last split holds one token
            c = Case(rt, 0x5D3 + d + n, 2, hq, hkv, d, past, 1, theta=5e5, quant=quant,
                     permute_pages=True)
            c.step_kv()
            q = c.query("f32")
            rt.set_decode_merge(1)
            got = c.gpu_decode(q)
            assert rt.last_decode_shape() == (2 * n * hkv, 64) and rt.last_decode_launches() == 1
            assert_close(got, c.oracle_attend(q), f"{n} splits")
            rt.set_decode_merge(0)
            assert np.abs(got - c.gpu_decode(q)).max() <= 64 * 2.0 ** -24 * 6
    finally:
        rt.set_decode_split(prev_split)
        rt.set_decode_merge(prev_merge)


@pytest.mark.parametrize("quant,batch", [(S.KV_INT8, 65), (S.KV_INT4, 130), (S.KV_INT8, 256),
                                         (S.KV_INT4, 256), (S.KV_INT8, 257), (S.KV_INT4, 300)])
def test_decode_many_ragged_sequences(rt, quant, batch):
    """Up to 256 sequences take the table of work items, read 64 entries at a
    time, more take the scan; both over 1 to several splits a sequence."""
    log(f"decode, {batch} ragged sequences, quant {quant}")
    lens = [int(x) for x in np.random.default_rng(batch).integers(0, 1500, size=batch)]
    c = Case(rt, 0x5D2 + batch, batch, 2, 1, 64, lens, 1, theta=1e4, quant=quant)
    c.step_kv()
    q = c.query("f32")
    got = c.gpu_decode(q)
    wg, split = rt.last_decode_shape()
    splits = [(n + split) // split for n in lens]
    assert wg == sum(splits) and len(set(splits)) > 1  # several splits, not all alike
    assert_close(got, c.oracle_attend(q), "many ragged sequences")
