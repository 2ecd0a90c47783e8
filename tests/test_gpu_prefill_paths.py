"""Prefill kernel paths chosen by sizes, types and alignment, against the
oracle (2e-3 abs + 1e-2 rel) or bit for bit against the path they replace."""
import numpy as np
import pytest

import smallaios_amd as S
from _gpu_util import (Case, assert_close, assert_close_weighted, dev, err_tol_ratio, log,
                       outlier_keys, weighted_abs_v)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    import torch
    assert torch.cuda.is_available()
    r = S.Runtime(0)
    yield r
    r.close()


@pytest.mark.parametrize("quant,hq,hkv,d,dtype,interleaved", [
    (S.KV_INT8, 8, 2, 64, "bf16", False), (S.KV_INT8, 8, 2, 128, "f32", True),
    (S.KV_INT8, 4, 4, 168, "bf16", False), (S.KV_INT8, 8, 4, 168, "f32", True),
    (S.KV_INT8, 8, 1, 256, "bf16", True), (S.KV_INT4, 8, 2, 128, "bf16", False),
    (S.KV_INT4, 4, 2, 256, "f32", False)])
def test_prefill_query_alignment(rt, quant, hq, hkv, d, dtype, interleaved):
    """A query one element into its buffer takes the elementwise loads: the
    same bits as the 16-byte loads of an aligned one, and the oracle's values."""
    import torch
    log(f"prefill query alignment quant {quant} d {d} {dtype} interleaved {interleaved}")
    c = Case(rt, 0x9A1 + d, 2, hq, hkv, d, [70, 9], 37, quant=quant, kv_dtype="bf16",
             interleaved=interleaved)
    c.step_kv()
    q = c.query(dtype)
    ref = c.gpu_prefill(q, dtype)
    qa = dev(q, dtype)
    buf = torch.empty(qa.numel() + 1, dtype=qa.dtype, device="cuda")
    buf[1:] = qa.ravel()
    out = torch.zeros(q.shape, device="cuda")
    c.cache.prefill(0, buf[1:], out, c.batch, c.new_tokens, hq, c.cos_d, c.sin_d,
                    c.cos.shape[0], True, interleaved)
    got = out.cpu().numpy()
    assert np.array_equal(got, ref)
    assert_close(got, c.oracle_attend(q), "prefill, unaligned query")


@pytest.mark.parametrize("hq,hkv,d", [(4, 2, 64), (4, 1, 128), (2, 1, 256)])
def test_prefill_int4_large_query_sums(rt, hq, hkv, d):
    """int4: group sums of the query past binary16's range (the zero points'
    step takes them 2^-5 smaller). Keys are small, so the scores stay ordinary."""
    log(f"prefill int4, large query sums, d {d}")
    c = Case(rt, 0x9A2 + d, 1, hq, hkv, d, [100], 40, quant=S.KV_INT4, do_rotary=False,
             k_transform=lambda rng, k: k * np.float32(2e-4))
    c.step_kv()
    q = c.query("f32") * np.float32(2e3) + np.float32(1.2e4 * np.sqrt(d / 64))
    assert 32 * q.mean() / np.sqrt(d) * 1.44 > 32768
    got = c.gpu_prefill(q, "f32")
    ref = c.oracle_attend(q)
    log(f"  worst err/tol {err_tol_ratio(got, ref):.4f}")
    assert_close(got, ref, "prefill int4, large query sums")


KEY_GROUPS = [
    # hq, hkv, d, past, new, window, large V: 32, 33, 128 and 129 rows a kv
    # head, one row, tiles that do not fill the last round of 2 or 4, rows
    # whose first keys are another key group's
    (8, 2, 128, [700, 0], 8, 0, False), (8, 1, 128, [300], 4, 0, False),
    (2, 2, 64, [129, 64], 32, 0, False), (1, 1, 128, [1023], 1, 0, False),
    (3, 3, 128, [200], 33, 0, False), (8, 2, 64, [450, 31], 32, 100, False),
    (4, 4, 128, [5], 129, 0, False), (16, 2, 128, [63], 16, 0, False),
    (32, 8, 128, [0], 300, 0, False), (8, 1, 64, [0, 500], 90, 70, False),
    (8, 2, 128, [500], 8, 0, True), (8, 2, 128, [260], 60, 0, True),
    (4, 1, 64, [1200], 7, 130, True),
]


@pytest.mark.parametrize("case", KEY_GROUPS, ids=[f"case{i}" for i in range(len(KEY_GROUPS))])
def test_prefill_key_groups(rt, case):
    """int8 chunks whose workgroups split the keys among their waves (4 key
    groups up to 32 rows a kv head, 2 up to 128 or while workgroups are few);
    large V takes the same split through the precise pass, bounded as in
    test_prefill_key_split_large_v."""
    key_groups_case(rt, S.KV_INT8, *case)


@pytest.mark.parametrize("case", [
    (8, 2, 128, [700, 0], 8, 0, False), (2, 2, 64, [129, 64], 128, 0, False),
    (1, 1, 128, [1023], 1, 0, False), (3, 3, 64, [200], 33, 100, False),
    (32, 8, 128, [0], 300, 0, False), (8, 1, 128, [400, 70], 90, 70, False)],
    ids=[f"case{i}" for i in range(6)])
def test_prefill_key_groups_int4(rt, case):
    """Two key groups over the int4 cache (its parameters in a ring of four)."""
    key_groups_case(rt, S.KV_INT4, *case)


def key_groups_case(rt, quant, hq, hkv, d, past, new, window, big):
    log(f"prefill key groups quant {quant} hq {hq} hkv {hkv} d {d} past {past} new {new} window {window} "
        f"large V {big}")
    # large V in some tokens only: the groups' tiles have different exponents
    big_v = (lambda rng, v: v * np.where(rng.random(v.shape[:2] + (1,)) < 0.02, 1e5, 1.0)
             .astype(np.float32)) if big else None
    c = Case(rt, 0x9A3 + d + new, len(past), hq, hkv, d, past, new, theta=5e5, quant=quant,
             permute_pages=True, k_transform=outlier_keys(d, (3, 40)) if not big else None,
             v_transform=big_v)
    c.step_kv()
    q = c.query("f32")
    got = c.gpu_prefill(q, "f32", window=window)
    ref = c.oracle_attend(q, mask_window=window)
    if big and window == 0:
        assert np.isfinite(got).all()
        assert_close_weighted(got, ref, weighted_abs_v(c, q), 2.0 ** -12, "key groups, large V")
    elif big:
        # Sum p|v| of the window is at most the rows' largest |v| there
        assert (np.abs(got - ref) <= 2e-3 + 1e-2 * np.abs(ref) + 2.0 ** -12 * 6e5).all()
    else:
        log(f"  worst err/tol {err_tol_ratio(got, ref):.4f}")
        assert_close(got, ref, "prefill key groups")
