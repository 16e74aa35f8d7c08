"""The ternary GEMM's digit planes and tile shapes on the GPU (trx_gemm.hip), against float64.

The bound is derived: what the five digits leave of x is at most 2^-23 of its own leading power or 2^-25
of its 32-column block's, whichever is more (2^-106 where the block lies below 2^-80, the smallest
exponent): 2^-24 of the largest value plus two of the sums' half units cover both. A group's ten
matrix instructions and the sums over the G groups round in float32 (2^-24 of the partial sums each,
which the sum of |w x| bounds), and the output adds a few roundings (the RMSNorm's scale, the
residual). Where values lie 2^7 or more above the rest of their block, the rest's own largest counts.
"""

import ctypes

import numpy as np
import pytest

from trixium_amd import _lib, layout as L
from trixium_amd.bons import encode_rows

pytestmark = pytest.mark.gpu

EPS = 1e-6


def _matrix(kind, M, K, rng, silent=None):
    codes = rng.integers(0, 4 if kind == L.KIND_TERNARY else 3, (M, K)).astype(np.uint8)
    if silent is not None:
        codes[:, silent] = 1
    sc = rng.uniform(0.01, 0.05, (M, K // 128)).astype(np.float16)
    w = (codes.astype(np.float64) - 1).reshape(M, -1, 128) * sc.astype(np.float64)[:, :, None]
    return encode_rows(kind, K, sc, codes), w.reshape(M, K)


def _run(rows, kind, M, K, x, gain, epi, y0, work_offset=0):
    n = x.shape[0]
    cols = M // 2 if epi == _lib.EPI_SWIGLU else M
    rb, xb = _lib.DeviceBuffer.from_array(rows), _lib.DeviceBuffer.from_array(x)
    gb = _lib.DeviceBuffer.from_array(gain) if gain is not None else None
    yb = _lib.DeviceBuffer.from_array(y0) if y0 is not None else _lib.DeviceBuffer(4 * n * cols)
    wb = _lib.DeviceBuffer(4 * n * (K + 1) + work_offset)
    _lib.call("trx_gemm_ternary_f32", rb.ptr, kind, M, K, xb.ptr, n, gb.ptr if gb else None, ctypes.c_float(EPS),
              yb.ptr, epi, wb.ptr + work_offset, None)
    _lib.synchronize()
    return yb.download(np.float32, n * cols).reshape(n, cols).astype(np.float64)


def _check(kind, M, K, n, epi, norm, x, rng, work_offset=0, top=None, silent=None):
    rows, W = _matrix(kind, M, K, rng, silent)
    gain = rng.uniform(0.8, 1.2, K).astype(np.float32) if norm else None
    y0 = rng.standard_normal((n, M)).astype(np.float32) if epi == _lib.EPI_RESID else None
    v = x.astype(np.float64)
    r = np.ones((n, 1))
    if norm:
        r = 1.0 / np.sqrt(np.mean(v * v, axis=1, keepdims=True) + EPS)
        v = v * gain.astype(np.float64)
    G = K // 128
    # Half 1 of a trit5 group takes its columns one later, so a block spans two of the 32-column runs.
    if top is None:
        top = np.abs(v).reshape(n, G, 128).max(axis=2).repeat(128, axis=1)
    ref, mag = (v @ W.T) * r, (np.abs(v) @ np.abs(W).T) * r
    err = 2.0**-24 * ((np.maximum(top, 2.0**-81) @ np.abs(W).T) * r + (G + 16) * mag)
    if epi == _lib.EPI_SWIGLU:
        F = M // 2
        g, u = ref[:, :F], ref[:, F:]
        s = 1 / (1 + np.exp(-np.clip(g, -700, 700)))
        ref = g * s * u
        # |silu'| <= 1.1; the exponential and the division add a few float32 roundings of the result.
        err = 1.1 * err[:, :F] * np.abs(u) + np.abs(g * s) * err[:, F:] + 2.0**-20 * np.abs(ref) + 1e-12
    elif y0 is not None:
        ref = ref + y0
        err = err + 2.0**-23 * np.abs(ref)
    got = _run(rows, kind, M, K, x, gain, epi, y0, work_offset)
    worst = float(np.max(np.abs(got - ref) / err))
    print(f"kind {kind} M {M} K {K} n {n} epi {epi} norm {norm}: worst error / bound {worst:.3f}", flush=True)
    assert worst <= 1.0


# Rows and positions around the tiles' edges (32 and 128 positions, 32 to 256 rows), one group (fewer
# than the waves that split K), groups that eight waves share unevenly, and shapes that take each of
# the launcher's four tiles on 256 CUs (128 x 256: the last three).
@pytest.mark.parametrize("kind", [L.KIND_TERNARY5, L.KIND_TERNARY])
@pytest.mark.parametrize("epi", [_lib.EPI_STORE, _lib.EPI_RESID, _lib.EPI_SWIGLU])
@pytest.mark.parametrize("M,K,n", [(2, 128, 1), (34, 128, 33), (64, 256, 31), (66, 1152, 32), (1000, 1280, 3),
                                   (2046, 2048, 65), (4096, 384, 97), (6144, 1152, 200), (2050, 640, 512),
                                   (12290, 384, 513), (24576, 256, 385), (8190, 128, 1100)])
def test_tiles_match_float64(kind, epi, M, K, n):
    rng = np.random.default_rng(M + 7 * K + n + epi)
    x = (rng.standard_normal((n, K)) * rng.uniform(0.2, 4.0, (n, 1))).astype(np.float32)
    _check(kind, M, K, n, epi, epi != _lib.EPI_RESID, x, rng)


@pytest.mark.parametrize("kind", [L.KIND_TERNARY5, L.KIND_TERNARY])
def test_magnitudes(kind):
    """Rows from 1e-30 to 1e30, outliers, zero blocks and denormals: every block has its own exponent."""
    rng = np.random.default_rng(5)
    n, K = 40, 768
    x = rng.standard_normal((n, K))
    x[:20] *= 10.0 ** np.linspace(-30, 30, 20)[:, None]
    x[20:30, ::97] *= 1e4
    x[30, :256] = 0
    x[31] = 0
    x[32] *= 1e-42
    x[33, 5] = 2.0**127
    _check(kind, 160, K, n, _lib.EPI_STORE, False, x.astype(np.float32), rng)


def test_workspace_at_a_dword():
    rng = np.random.default_rng(6)
    x = rng.standard_normal((37, 512)).astype(np.float32)
    _check(L.KIND_TERNARY5, 300, 512, 37, _lib.EPI_STORE, True, x, rng, work_offset=4)


@pytest.mark.parametrize("n", [5, 300])
def test_non_finite_rows_stay_apart(n):
    """A row that holds an infinity or a NaN gives NaN; the other rows are as without it."""
    rng = np.random.default_rng(8)
    M, K, kind = 24576 if n == 300 else 512, 384, L.KIND_TERNARY5
    rows, _ = _matrix(kind, M, K, rng)
    x = rng.standard_normal((n, K)).astype(np.float32)
    clean = _run(rows, kind, M, K, x, None, _lib.EPI_STORE, None)
    x[1, 7], x[3, 200] = np.inf, np.nan
    got = _run(rows, kind, M, K, x, None, _lib.EPI_STORE, None)
    bad = np.isin(np.arange(n), (1, 3))
    assert np.isnan(got[bad]).all()
    assert np.array_equal(got[~bad], clean[~bad])


@pytest.mark.parametrize("kind", [L.KIND_TERNARY5, L.KIND_TERNARY])
@pytest.mark.parametrize("M,n", [(260, 40), (24576, 400)])
def test_lone_values_keep_the_rest(kind, M, n):
    """One to three values 10^4 to 10^30 times the rest, in every place of a group and group of a row in turn: the
    outputs whose weight there is 0 stay as exact as without it."""
    rng = np.random.default_rng(M + kind)
    K = 384 if M > 1000 else 1280
    x = rng.standard_normal((n, K))
    rest = 128 * np.abs(x).reshape(n, K // 128, 128).max(axis=2).repeat(128, axis=1)
    at = (np.arange(n) * 37) % K
    x[np.arange(n), at] = rng.choice([-1, 1], n) * 10.0 ** rng.uniform(4, 30, n)
    for step, c, f in ((1, 0, 1.0), (3, 5, 0.3), (6, 9, -0.05)):     # two and three in one block
        for r in range(0, n, step):
            col = (at[r] & ~31) + (at[r] + c) % 32
            x[r, col] = f * x[r, at[r]]
            rest[r, col] = abs(x[r, at[r]])          # they share a scale of their own
    _check(kind, M, K, n, _lib.EPI_STORE, False, x.astype(np.float32), rng, top=rest)


def _fp16_pair(x):
    """x as a float32 sum of two fp16 values of its row's scale (what the kernel's predecessor multiplied)."""
    xs = 2.0 ** np.maximum(0, np.frexp(np.abs(x).max(axis=1, keepdims=True))[1] - 14)
    y = (x / xs).astype(np.float32)
    hi = y.astype(np.float16).astype(np.float32)
    return ((hi + (y - hi).astype(np.float16).astype(np.float32)) * xs).astype(np.float64)


# Inputs as projections meet them: a normed residual stream with and without larger channels, products of
# two normals, SwiGLU activations.
def _inputs(name, n, K, rng):
    x = rng.standard_normal((n, K))
    if name == "channels":
        x[:, rng.permutation(K)[:K // 512]] *= 20
    elif name == "product":
        x *= rng.standard_normal((n, K))
    elif name == "swiglu":
        x *= (lambda g: g / (1 + np.exp(-g)))(3 * rng.standard_normal((n, K)))
    elif name == "large":
        x *= 100
    return x.astype(np.float32)


@pytest.mark.parametrize("kind", [L.KIND_TERNARY5, L.KIND_TERNARY])
@pytest.mark.parametrize("name", ["normal", "channels", "product", "swiglu", "large"])
@pytest.mark.parametrize("M,n", [(512, 200), (8192, 1100)])
def test_operands(kind, name, M, n):
    """Weights of one trit a row and scale 1 hand x back as the products see it. Every value is held to 2^-23 of
    its own leading power or 2^-25 of its block's, whichever is more (half 1 of a trit5 group takes its columns one
    later: the bound takes the 128-column group's), and the sum rounds to float32 (two half units); over all
    values the error is no larger than that of a pair of fp16 values."""
    rng = np.random.default_rng(M + n + len(name))
    K = 512
    codes = np.ones((M, K), np.uint8)
    codes[np.arange(M), np.arange(M) % K] = 2
    rows = encode_rows(kind, K, np.ones((M, K // 128), np.float16), codes)
    x = _inputs(name, n, K, rng)
    got = _run(rows, kind, M, K, x, None, _lib.EPI_STORE, None).reshape(n, M // K, K)
    assert np.array_equal(got, np.broadcast_to(got[:, :1], got.shape))
    v = x.astype(np.float64)
    err, lead = np.abs(got[:, 0] - v), 2.0 ** (np.frexp(v)[1] - 1)
    top = lead.reshape(n, K // 128, 128).max(axis=2).repeat(128, axis=1)
    assert np.all(err <= np.maximum(2.0**-23 * lead, 2.0**-25 * top) + 2.0**-23 * lead)
    rms = [float(np.sqrt(np.mean(e * e))) for e in (err, _fp16_pair(x) - v)]
    print(f"{name} rms error {rms[0]:.2e}, of an fp16 pair {rms[1]:.2e}", flush=True)
    assert rms[0] <= rms[1]


# A kernel's waves remember the groups that hold such blocks 64 apart: the last two shapes have more groups.
LARGE = [(kind, big, count, M, K, n) for kind in (L.KIND_TERNARY5, L.KIND_TERNARY) for big in (3e2, 1e4, 1e18)
         for count in (1, 3, 4, 8, 17, 24) for M, K, n in ((130, 1280, 41), (8190, 384, 1100))]
LARGE += [(L.KIND_TERNARY5, 1e4, 6, 8192, 8448, 1100), (L.KIND_TERNARY, 1e4, 6, 34, 67584, 5)]


@pytest.mark.parametrize("kind,big,count,M,K,n", LARGE)
def test_large_values_leave_the_rest(kind, big, count, M, K, n):
    """Any number of values far above the rest of their block, in some blocks of every row: outputs whose weights on
    them are 0 are as exact as if they were small (the bound takes the rest's largest value)."""
    rng = np.random.default_rng(count + M)
    x = rng.standard_normal((n, K))
    cols = np.zeros(K, bool)
    for b in list(rng.permutation(K // 32 - 1)[:4]) + [K // 32 - 1]:
        # From the block's second column on: the blocks of a trit5 half 1 end one column later.
        cols[32 * b + 1 + rng.permutation(31)[:count]] = True
    rest = np.abs(x * ~cols).reshape(n, K // 128, 128).max(axis=2).repeat(128, axis=1)
    x[:, cols] = rng.choice([-1, 1], (n, cols.sum())) * big * rng.uniform(1, 1.9, (n, cols.sum()))
    _check(kind, M, K, n, _lib.EPI_STORE, False, x.astype(np.float32), rng, top=rest, silent=cols)


def test_few_values_among_zeros():
    rng = np.random.default_rng(11)
    x = np.zeros((40, 512), np.float32)
    x[:, 5], x[:, 9], x[:, 20] = 1e6, 1.5, -0.7
    x[:, 300] = 0.9
    silent = np.zeros(512, bool)
    silent[5] = True
    _check(L.KIND_TERNARY5, 200, 512, 40, _lib.EPI_STORE, False, x, rng, top=np.ones(x.shape), silent=silent)


def test_planes_past_4_gib():
    """Four positions of 2^28 columns: their planes are past what 32-bit offsets reach. Weights of 1, a few columns of
    x set."""
    n, K, M, G = 4, 1 << 28, 2, 1 << 21
    row = np.concatenate([np.full(G, 1, np.float16).view(np.uint8), np.full(32 * G, 0xAA, np.uint8)])
    rb = _lib.DeviceBuffer.from_array(np.concatenate([row] * M))
    xb, wb, yb = _lib.DeviceBuffer(4 * n * K), _lib.DeviceBuffer(4 * n * (K + 1)), _lib.DeviceBuffer(4 * n * M)
    _lib.call("trx_memset_d8", xb.ptr, 0, 4 * n * K, None)
    want = np.zeros(n)
    for r in range(n):
        for i, c in enumerate((5, K // 3, K // 2 + 70, K - 1)):
            v = np.array([(r + 1) * 1.5 + i], np.float32)
            xb.upload(v, offset=4 * (r * K + c))
            want[r] += float(v[0])
    _lib.call("trx_gemm_ternary_f32", rb.ptr, L.KIND_TERNARY, M, K, xb.ptr, n, None, ctypes.c_float(EPS), yb.ptr,
              _lib.EPI_STORE, wb.ptr, None)
    _lib.synchronize()
    assert np.array_equal(yb.download(np.float32, n * M).reshape(n, M), np.repeat(want[:, None], M, 1))
