"""The exact engine matvec on the matrix cores (trx_gemv_rows.hip): every output and status bit equal to
the oracle's at the edges of its tiles (32 rows, eight waves over the groups) and of its range."""

import numpy as np
import pytest

from oracle import bitexact as ob
from trixium_amd import _lib, layout as L
from trixium_amd.bons import encode_rows

pytestmark = pytest.mark.gpu


def _call(rows, kind, M, K, x8, B, R, offset=0):
    n = x8.shape[0]
    rb = _lib.DeviceBuffer(rows.nbytes + 64)
    rb.upload(rows)
    xb = _lib.DeviceBuffer(x8.nbytes + 16)
    xb.upload(x8, offset=offset)
    yb, st = _lib.DeviceBuffer(4 * n * M), _lib.DeviceBuffer.from_array(np.zeros(1, np.int32))
    if n == 1:
        _lib.call("trx_gemv_ternary_exact", rb.ptr, kind, M, K, xb.ptr + offset, B, R, yb.ptr, st.ptr, None)
    else:
        _lib.call("trx_gemv_ternary_exact_rows", rb.ptr, kind, M, K, xb.ptr, n, B, R, yb.ptr, st.ptr, None)
    _lib.synchronize()
    return yb.download(np.int32, n * M).reshape(n, M), int(st.download(np.int32)[0])


def _want(codes, scales, x8, B, R):
    m11, e16 = ob.fp16_decompose(scales)
    out, status = [], 0
    for x in x8:
        prod, sh = ob.group_sums(codes, x) * m11, e16 + B
        acc = np.where(sh >= 0, prod << np.maximum(sh, 0), prod >> np.minimum(np.maximum(-sh, 0), 63)).sum(axis=1)
        res = acc >> R
        status |= int(np.any(np.abs(acc) >= 2**47)) | 2 * int(np.any(np.abs(res) >= 2**31))
        out.append(res.astype(np.int32))
    return np.stack(out), status


@pytest.mark.parametrize("kind", [L.KIND_TERNARY5, L.KIND_TERNARY])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("M,K", [(1, 128), (31, 256), (33, 1024), (64, 1152), (95, 2176), (40, 14336)])
def test_rows_match_oracle(kind, n, M, K):
    rng = np.random.default_rng(M + K + n)
    codes = rng.integers(0, 4 if kind == L.KIND_TERNARY else 3, (M, K)).astype(np.uint8)
    scales = rng.uniform(-0.05, 0.05, (M, K // 128)).astype(np.float16)
    x8 = rng.integers(-128, 128, (n, K)).astype(np.int8)
    # (12, 0): scales shifted left by little and right; (27, 13): as images have them; (-10, 0): right only;
    # (48, 0): both overflows.
    for B, R in ((12, 0), (27, 13), (-10, 0), (48, 0)):
        got, status = _call(encode_rows(kind, K, scales, codes), kind, M, K, x8, B, R)
        want, wst = _want(codes, scales, x8, B, R)
        print(f"kind {kind} n {n} M {M} K {K} B {B} R {R} status {status}", flush=True)
        assert np.array_equal(got, want) and status == wst


@pytest.mark.parametrize("kind", [L.KIND_TERNARY5, L.KIND_TERNARY])
@pytest.mark.parametrize("offset", [1, 4, 7])
def test_one_vector_at_any_byte(kind, offset):
    rng = np.random.default_rng(offset)
    M, K = 50, 512
    codes = rng.integers(0, 3, (M, K)).astype(np.uint8)
    scales = rng.uniform(0.01, 0.05, (M, K // 128)).astype(np.float16)
    x8 = rng.integers(-128, 128, (1, K)).astype(np.int8)
    got, status = _call(encode_rows(kind, K, scales, codes), kind, M, K, x8, 27, 10, offset)
    want, wst = _want(codes, scales, x8, 27, 10)
    assert np.array_equal(got, want) and status == wst


@pytest.mark.parametrize("kind", [L.KIND_TERNARY5, L.KIND_TERNARY])
def test_one_vector_of_many_rows(kind):
    """A large matrix through the multi-row entry point: one vector takes the single-vector kernel."""
    rng = np.random.default_rng(kind)
    K, part, M = 128, 256, 1 << 18                   # 2^25 weights, rounds of 4096 rows full
    codes = rng.integers(0, 3, (part, K)).astype(np.uint8)
    scales = rng.uniform(0.01, 0.05, (part, 1)).astype(np.float16)
    x8 = rng.integers(-128, 128, (1, K)).astype(np.int8)
    rows = np.tile(encode_rows(kind, K, scales, codes).reshape(part, -1), (M // part, 1))
    rb, xb = _lib.DeviceBuffer(rows.nbytes + 64), _lib.DeviceBuffer.from_array(x8)
    rb.upload(rows)
    yb, st = _lib.DeviceBuffer(4 * M), _lib.DeviceBuffer.from_array(np.zeros(1, np.int32))
    _lib.call("trx_gemv_ternary_exact_rows", rb.ptr, kind, M, K, xb.ptr, 1, 27, 10, yb.ptr, st.ptr, None)
    _lib.synchronize()
    want, wst = _want(codes, scales, x8, 27, 10)
    assert np.array_equal(yb.download(np.int32, M).reshape(M // part, part), np.tile(want, (M // part, 1)))
    assert int(st.download(np.int32)[0]) == wst
