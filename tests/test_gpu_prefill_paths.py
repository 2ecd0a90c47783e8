"""Prefill kernel paths chosen by sizes, types and alignment, against the
oracle (2e-3 abs + 1e-2 rel) or bit for bit against the path they replace."""
import numpy as np
import pytest

import smallaios_amd as S
from _gpu_util import Case, assert_close, dev, err_tol_ratio, log, outlier_keys

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
