"""The calls whose time counts, over the sizes that the shipped configurations run.

Two kinds of case. Single projections go through the C entry points that a program calls with its
own device buffers: the packed float GEMV of decoding, many GEMVs in one dispatch, the engine's
exact integer matvec, the multi-position GEMM of prefill. Whole calls go through `Decoder`:
prompts, decoding at a context, teacher-forced scoring; most with the widths of a shipped
configuration and a few of its layers, two with all of them.

Weights are random trits with P(0) = 0.4 and fp16 group scales U(0.01, 0.05), stored as row packets
as an image holds them. Projection inputs are normal with a few channels 20 times larger, as a
residual stream has them; a down projection's input is a product of two normals.
"""

import ctypes
import dataclasses

import numpy as np
import torch

from trixium_amd import _lib
from trixium_amd import configs as C
from trixium_amd import layout as L
from trixium_amd.model import Decoder

KINDS = {"trit5": L.KIND_TERNARY5, "2bit": L.KIND_TERNARY}
EPILOGUES = {"store": _lib.EPI_STORE, "resid": _lib.EPI_RESID, "swiglu": _lib.EPI_SWIGLU}
MODELS = {"1.7b": C.QWEN3_1P7B, "8b": C.QWEN3_8B, "27b": C.QWEN35_27B}
SCALE_LO, SCALE_SPAN = 0.01, 0.04
EPS = 1e-6
GUARD = 256                        # readable bytes past the end of a buffer that a kernel reads


def listed():
    return [
        # One small projection with its residual add: Qwen3-1.7B's attention output (launch latency).
        {"name": "gemv-o-1.7b", "op": "gemv", "M": 2048, "K": 2048, "kind": "trit5", "norm": False,
         "epilogue": "resid"},
        # The projection that dominates a decoded token: Qwen3-8B's gate|up with RMSNorm and SwiGLU.
        {"name": "gemv-gate-up-8b", "op": "gemv", "M": 24576, "K": 4096, "kind": "trit5", "norm": True,
         "epilogue": "swiglu"},
        # Many independent matvecs over one vector in one dispatch (the isolated matvec benchmark).
        {"name": "matvecs-1.7b", "op": "matvecs", "M": 2048, "K": 2048, "kind": "trit5", "count": 293},
        # The engine's exact integer matvec of eight vectors, Qwen3-1.7B's FFN shape.
        {"name": "engine-rows-1.7b", "op": "engine", "M": 6144, "K": 2048, "kind": "trit5", "n": 8},
        # The same of one vector, the larger FFN projection of Qwen3-8B in 2-bit codes.
        {"name": "engine-one-8b", "op": "engine", "M": 4096, "K": 12288, "kind": "2bit", "n": 1},
        # A short chat turn through one projection: Qwen3-8B's q|k|v for 24 positions.
        {"name": "gemm-turn-qkv-8b", "op": "gemm", "M": 6144, "K": 4096, "kind": "trit5", "n": 24,
         "norm": True, "epilogue": "store"},
        # A prompt of ragged length through Qwen3-1.7B's down projection, 2-bit codes.
        {"name": "gemm-down-1.7b", "op": "gemm", "M": 2048, "K": 6144, "kind": "2bit", "n": 509,
         "norm": False, "epilogue": "resid"},
        # A long prompt through Qwen3-8B's gate|up with SwiGLU.
        {"name": "gemm-gate-up-8b", "op": "gemm", "M": 24576, "K": 4096, "kind": "trit5", "n": 2048,
         "norm": True, "epilogue": "swiglu"},
        # Decoding with Qwen3-8B's shape after a 2048-token prompt, every layer and the head.
        {"name": "decode-8b", "op": "decode", "model": "8b", "layers": 36, "context": 2048, "tokens": 8},
        # The prompt of a request: Qwen3-1.7B's shape, every layer, to the logits of its last token.
        {"name": "prompt-1.7b", "op": "prompt", "model": "1.7b", "layers": 28, "tokens": 512},
        # One period of the 27B hybrid (three DeltaNet layers, one gated attention layer).
        {"name": "prompt-27b-period", "op": "prompt", "model": "27b", "layers": 4, "tokens": 1024},
        # Teacher-forced scoring of a passage (perplexity): four layers of Qwen3-1.7B and its head.
        {"name": "score-1.7b-layers", "op": "score", "model": "1.7b", "layers": 4, "tokens": 192},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(("gemv", "gemv", "matvecs", "engine", "gemm", "gemm", "gemm", "decode", "prompt", "prompt",
                     "score"))
    kind = rng.choice(("trit5", "trit5", "2bit"))
    if op in ("gemv", "engine", "gemm"):
        K = 128 * _log_int(rng, 16, 136 if op != "engine" else 96)
        M = _log_int(rng, 1024, 24576)
    if op == "gemv":
        epi = rng.choice(tuple(EPILOGUES))
        M -= M % 4 if epi == "swiglu" else 0
        return {"op": op, "M": M, "K": K, "kind": kind, "norm": epi != "resid" and rng.random() < 0.7,
                "epilogue": epi}
    if op == "matvecs":
        M, K = rng.choice(C.MICROBENCH_SHAPES)
        return {"op": op, "M": M, "K": K, "kind": kind, "count": max(2, _log_int(rng, 16, 300) * 2048 * 2048 // (M * K))}
    if op == "engine":
        return {"op": op, "M": M, "K": K, "kind": kind, "n": rng.randint(1, 8)}
    if op == "gemm":
        n = _log_int(rng, 2, 2048)
        n = max(2, min(n, 24576 * 4096 * 2048 // (M * K)))
        epi = rng.choice(tuple(EPILOGUES))
        M -= M % 2 if epi == "swiglu" else 0
        return {"op": op, "M": M, "K": K, "kind": kind, "n": n, "norm": epi != "resid" and rng.random() < 0.7,
                "epilogue": epi}
    model = rng.choice(tuple(MODELS))
    layers = 4 if model == "27b" else rng.randint(2, 6)
    if op == "decode":
        context = _log_int(rng, 16, MODELS[model].max_ctx - 20)
        return {"op": op, "model": model, "layers": layers, "context": context, "tokens": rng.randint(4, 16)}
    if op == "prompt":
        return {"op": op, "model": model, "layers": layers,
                "tokens": _log_int(rng, 8, {"1.7b": 1000, "8b": 2048, "27b": 1024}[model])}
    return {"op": op, "model": model, "layers": layers, "tokens": _log_int(rng, 16, 192)}


# Weights and inputs -----------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)


def _geometry(kind, K):
    """(bytes of the scales, bytes of a row) of a row packet."""
    G = K // 128
    head = 32 * -(-G // 16)
    return head, head + (32 * -(-26 * G // 32) if kind == "trit5" else 32 * G)


def _rows(kind, M, K, gen):
    """Codes in {0, 1, 2} [M, K], scales [M, K / 128] (fp16) and the row packets that hold them."""
    G = K // 128
    u = torch.randint(0, 10, (M, K), generator=gen, device="cuda", dtype=torch.uint8)
    codes = (u >= 3).to(torch.uint8) + (u >= 7).to(torch.uint8)
    scales = (SCALE_LO + SCALE_SPAN * torch.rand((M, G), generator=gen, device="cuda")).to(torch.float16)
    head, size = _geometry(kind, K)
    buf = torch.zeros(M * size + GUARD, dtype=torch.uint8, device="cuda")
    rows = buf[:M * size].view(M, size)
    rows[:, :2 * G] = scales.view(torch.uint8).view(M, 2 * G)
    if kind == "trit5":
        lanes = torch.zeros((M, G, 130), dtype=torch.uint8, device="cuda")
        lanes[:, :, :128] = codes.view(M, G, 128)
        lanes = lanes.view(M, G * 26, 5)
        packed = lanes[:, :, 4].clone()
        for k in (3, 2, 1, 0):
            packed = packed * 3 + lanes[:, :, k]
        rows[:, head:head + 26 * G] = packed
    else:
        lanes = codes.view(M, K // 4, 4)
        rows[:, head:] = lanes[:, :, 0] | lanes[:, :, 1] << 2 | lanes[:, :, 2] << 4 | lanes[:, :, 3] << 6
    return codes, scales, buf


def _padded(t):
    """The values of t in a buffer with readable bytes behind them."""
    out = torch.zeros(t.numel() + GUARD // t.element_size(), dtype=t.dtype, device="cuda")
    out[:t.numel()] = t.reshape(-1)
    return out


def _activations(n, K, gen, product=False):
    x = torch.randn((n, K), generator=gen, device="cuda")
    if product:
        return x * torch.randn((n, K), generator=gen, device="cuda")
    big = torch.randperm(K, generator=gen, device="cuda")[:max(1, K // 512)]
    x[:, big] *= 20.0
    return x


def _float_inputs(case, seed):
    """(codes, scales, packets, x [n, K], gain or None, residual or None) of a projection case."""
    gen = _generator(seed)
    M, K, n = case["M"], case["K"], case.get("n", 1)
    codes, scales, rows = _rows(case["kind"], M, K, gen)
    x = _activations(n, K, gen, case["epilogue"] == "resid")
    gain = 0.8 + 0.4 * torch.rand(K, generator=gen, device="cuda") if case["norm"] else None
    resid = torch.randn((n, M), generator=gen, device="cuda") if case["epilogue"] == "resid" else None
    return codes, scales, rows, x, gain, resid


def _engine_inputs(case, seed):
    gen = _generator(seed)
    codes, scales, rows = _rows(case["kind"], case["M"], case["K"], gen)
    x8 = torch.randint(-127, 128, (case["n"], case["K"]), generator=gen, device="cuda", dtype=torch.int8)
    # The accumulator's bias and the result's shift as an image's tensor of these scales has them: the
    # largest scale's exponent at 2^12, the result in 32 bits.
    return codes, scales, rows, x8, 27, 12


def _matvec_inputs(case, seed):
    gen = _generator(seed)
    copies = [_rows(case["kind"], case["M"], case["K"], gen) for _ in range(8)]
    return copies, _activations(1, case["K"], gen)


def _ptr(t):
    return None if t is None else t.data_ptr()


def _packed(kind, M, K, rows, swiglu):
    pb, wb = ctypes.c_size_t(), ctypes.c_size_t()
    _lib.call("trx_pack_geometry", KINDS[kind], M, K, ctypes.byref(pb), ctypes.byref(wb))
    packed = torch.zeros(pb.value + GUARD, dtype=torch.uint8, device="cuda")
    _lib.call("trx_pack_ternary", _ptr(rows), KINDS[kind], M, K, int(swiglu), _ptr(packed), None)
    return packed, pb.value, wb.value


def _model(case):
    mc = MODELS[case["model"]]
    if case["layers"] != mc.n_layer:
        mc = dataclasses.replace(mc, n_layer=case["layers"], layer_types=tuple(mc.layer_types[:case["layers"]]))
    return mc


def _gate_rows(mc, seed):
    """The Q8 rows of every DeltaNet layer's beta and alpha, {(role, layer): (int8 [nv, E], fp16
    scales per 32)}, scaled so that the gates' inputs are of order one."""
    rng = np.random.default_rng(seed + 7)
    nv, E = mc.dn_num_v_heads, mc.n_embd
    return {(r, l): (rng.integers(-127, 128, (nv, E), dtype=np.int8),
                     rng.uniform(0.0001, 0.0004, (nv, E // 32)).astype(np.float16))
            for l in range(mc.n_layer) if mc.layer_type(l) == "deltanet" for r in (L.ROLE_SSM_BETA, L.ROLE_SSM_ALPHA)}


def _tokens(case, mc, seed):
    n = case["tokens"] + case.get("context", 0)
    return np.random.default_rng(seed).integers(0, mc.vocab, n).astype(np.int32)


def prepare(case, seed):
    op = case["op"]
    if op == "gemv":
        codes, scales, rows, x, gain, resid = _float_inputs(case, seed)
        M, K = case["M"], case["K"]
        packed, _, wb = _packed(case["kind"], M, K, rows, case["epilogue"] == "swiglu")
        return {"case": case, "packed": packed, "x": _padded(x), "gain": None if gain is None else _padded(gain),
                "resid": resid, "y": torch.empty(M // 2 if case["epilogue"] == "swiglu" else M, device="cuda"),
                "work": torch.zeros(wb + GUARD, dtype=torch.uint8, device="cuda")}
    if op == "matvecs":
        copies, x = _matvec_inputs(case, seed)
        M, K, n = case["M"], case["K"], case["count"]
        one = [_packed(case["kind"], M, K, c[2], False) for c in copies]
        stride = -(-one[0][1] // 256) * 256
        packed = torch.zeros(n * stride + GUARD, dtype=torch.uint8, device="cuda")
        for i in range(n):
            packed[i * stride:i * stride + one[0][1]] = one[i % len(one)][0][:one[0][1]]
        wb = ctypes.c_size_t()
        _lib.call("trx_pack_batched_geometry", KINDS[case["kind"]], M, K, n, ctypes.byref(wb))
        return {"case": case, "packed": packed, "stride": stride, "x": _padded(x),
                "y": torch.empty((n, M), device="cuda"),
                "work": torch.zeros(wb.value + GUARD, dtype=torch.uint8, device="cuda")}
    if op == "engine":
        _, _, rows, x8, bias, shift = _engine_inputs(case, seed)
        return {"case": case, "rows": rows, "x8": _padded(x8), "bias": bias, "shift": shift,
                "y": torch.empty((case["n"], case["M"]), dtype=torch.int32, device="cuda"),
                "status": torch.zeros(1, dtype=torch.int32, device="cuda")}
    if op == "gemm":
        codes, scales, rows, x, gain, resid = _float_inputs(case, seed)
        M, K, n = case["M"], case["K"], case["n"]
        cols = M // 2 if case["epilogue"] == "swiglu" else M
        return {"case": case, "rows": rows, "x": _padded(x), "gain": None if gain is None else _padded(gain),
                "resid": resid, "y": torch.empty((n, cols), device="cuda"),
                "work": torch.empty(4 * n * (K + 1) + GUARD, dtype=torch.uint8, device="cuda")}
    mc = _model(case)
    dec = Decoder.synthetic(mc, seed=seed, max_new=32, prefill_chunk=2048)
    if mc.n_dn_layers:
        from trixium_amd.bons import encode_rows
        for (role, layer), (q, sc) in _gate_rows(mc, seed).items():
            dec.set_tensor(role, layer, encode_rows(L.KIND_Q8, mc.n_embd, sc, q))
    tokens = _tokens(case, mc, seed)
    dec.reset()
    if op == "decode":
        ctx = case["context"]
        dec.feed(tokens[:ctx])
        dec.prefill(ctx - 1)
        dec.step(1)
        dec.checkpoint()
        dec.synchronize()
        tokens = tokens[ctx:]
    return {"case": case, "dec": dec, "tokens": tokens}


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "gemv":
        epi, y = EPILOGUES[case["epilogue"]], state["y"]
        _lib.call("trx_gemv_packed_f32", _ptr(state["packed"]), KINDS[case["kind"]], case["M"], case["K"],
                  _ptr(state["x"]), _ptr(state["gain"]), EPS, _ptr(y), epi, _ptr(state["resid"]), _ptr(state["work"]),
                  None)
        return y
    if op == "matvecs":
        _lib.call("trx_gemv_packed_batched_f32", _ptr(state["packed"]), state["stride"], case["count"], case["count"],
                  KINDS[case["kind"]], case["M"], case["K"], _ptr(state["x"]), 0, _ptr(state["y"]), case["M"],
                  _ptr(state["work"]), None)
        return state["y"]
    if op == "engine":
        if case["n"] == 1:
            _lib.call("trx_gemv_ternary_exact", _ptr(state["rows"]), KINDS[case["kind"]], case["M"], case["K"],
                      _ptr(state["x8"]), state["bias"], state["shift"], _ptr(state["y"]), _ptr(state["status"]), None)
        else:
            _lib.call("trx_gemv_ternary_exact_rows", _ptr(state["rows"]), KINDS[case["kind"]], case["M"], case["K"],
                      _ptr(state["x8"]), case["n"], state["bias"], state["shift"], _ptr(state["y"]),
                      _ptr(state["status"]), None)
        return state["y"], state["status"]
    if op == "gemm":
        y = state["y"]
        if state["resid"] is not None:       # the residual epilogue adds in place
            y.copy_(state["resid"])
        _lib.call("trx_gemm_ternary_f32", _ptr(state["rows"]), KINDS[case["kind"]], case["M"], case["K"],
                  _ptr(state["x"]), case["n"], _ptr(state["gain"]), EPS, _ptr(y), EPILOGUES[case["epilogue"]],
                  _ptr(state["work"]), None)
        return y
    dec, tokens = state["dec"], state["tokens"]
    if op == "decode":
        dec.restore()
        dec.feed(tokens, head_from=case["context"])
        dec.step(len(tokens))
        return dec.logits()
    if op == "prompt":
        dec.reset()
        return dec.forward(tokens)
    nll, hidden = dec.score(tokens)
    return nll, hidden


# Work -------------------------------------------------------------------------------------------


def _weight_count(mc):
    """(ternary weights of a layer stack, of the head)."""
    total = 0
    for l in range(mc.n_layer):
        if mc.layer_type(l) == "deltanet":
            vd = mc.dn_num_v_heads * mc.dn_v_head_dim
            total += mc.n_embd * (2 * mc.dn_num_k_heads * mc.dn_k_head_dim + vd + vd) + vd * mc.n_embd
        else:
            total += mc.n_embd * (mc.q_dim * (2 if mc.attn_gated else 1) + 2 * mc.kv_dim) + mc.q_dim * mc.n_embd
        total += 3 * mc.n_embd * mc.ffn_dim
    return total, mc.vocab * mc.n_embd


def work(case):
    op = case["op"]
    if op in ("gemv", "matvecs", "engine", "gemm"):
        M, K, kind = case["M"], case["K"], case["kind"]
        G, n = K // 128, case.get("n", 1)
        weights = M * (2 * G + (26 if kind == "trit5" else 32) * G)
        if op == "matvecs":
            count = case["count"]
            return {"bytes": count * (weights + 4 * M) + 4 * K, "flops": 2 * count * M * K}
        if op == "engine":
            return {"bytes": weights + n * (K + 4 * M), "flops": 2 * n * M * K}
        out = M // 2 if case["epilogue"] == "swiglu" else M
        x = 4 * n * K + (4 * K if case["norm"] else 0)
        return {"bytes": weights + x + 4 * n * out * (2 if case["epilogue"] == "resid" else 1), "flops": 2 * n * M * K}
    mc = _model(case)
    body, head = _weight_count(mc)
    per_weight = 28 / 128                        # trit5 codes and the scales
    attn = sum(1 for l in range(mc.n_layer) if mc.layer_type(l) != "deltanet")
    dn = mc.n_layer - attn
    state = 2 * 4 * dn * mc.dn_num_v_heads * mc.dn_v_head_dim * mc.dn_k_head_dim
    kv = attn * 2 * 2 * mc.kv_dim                # bytes of a position in the cache
    n = case["tokens"]
    if op == "decode":
        past = n * case["context"] + n * (n + 1) // 2
        return {"bytes": int(n * (per_weight * (body + head) + state) + past * kv + 4 * mc.vocab),
                "flops": int(2 * n * (body + head) + 4 * past * attn * mc.q_dim + 4 * n * state // 4)}
    heads = n if op == "score" else 1
    past = n * (n + 1) // 2
    out = 4 * mc.vocab if op == "prompt" else 4 * n * (mc.n_embd + 1)
    return {"bytes": int(per_weight * (body + head) + state + n * kv + out),
            "flops": int(2 * (n * body + heads * head) + 4 * past * attn * mc.q_dim + 4 * n * state // 4)}


def tolerance(case):
    """About four times the distance from 64 bits: 0.7-1.9e-7 for a GEMV, 0.6-1.2e-6 for a GEMM, and for
    the calls through a model the roundings of the fp16 cache through its layers (a DeltaNet period
    4e-6, two to six attention layers 3e-5 to 1e-4, 28 and 36 of them 1.3e-4 and 1.8e-4)."""
    return {"gemv": {"rel": 8e-7}, "matvecs": {"rel": 4e-7}, "engine": "exact", "gemm": {"rel": 4e-6},
            "decode": {"rel": 8e-4}, "prompt": {"rel": 6e-4}, "score": {"rel": 4e-4}}[case["op"]]


# The same in 64 bits ----------------------------------------------------------------------------


def _project(codes, scales, x):
    """x [n, K] times the rows' weights, in float64."""
    out = torch.empty((x.shape[0], codes.shape[0]), dtype=torch.float64, device="cuda")
    for r in range(0, codes.shape[0], 8192):
        c, s = codes[r:r + 8192], scales[r:r + 8192]
        w = (c.double() - 1).view(c.shape[0], -1, 128) * s.double()[:, :, None]
        out[:, r:r + 8192] = x @ w.view(c.shape).T
    return out


def _rms(x, gain):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain


def _silu(x):
    return x * torch.sigmoid(x)


def exact(case, seed):
    op = case["op"]
    if op in ("gemv", "gemm"):
        codes, scales, _, x, gain, resid = _float_inputs(case, seed)
        x = x.double()
        if gain is not None:
            x = _rms(x, gain.double())
        y = _project(codes, scales, x)
        if case["epilogue"] == "swiglu":
            gate, up = y.chunk(2, dim=1)
            y = _silu(gate) * up
        elif resid is not None:
            y = y + resid.double()
        return y[0] if op == "gemv" else y
    if op == "matvecs":
        copies, x = _matvec_inputs(case, seed)
        ys = [_project(c, s, x.double())[0] for c, s, _ in copies]
        return torch.stack([ys[i % len(ys)] for i in range(case["count"])])
    if op == "engine":
        codes, scales, _, x8, bias, shift = _engine_inputs(case, seed)
        w = (codes.double() - 1).view(case["M"], -1, 128)
        sums = torch.stack([(w * x.double().view(1, -1, 128)).sum(2) for x in x8]).to(torch.int64)
        bits = scales.view(torch.int16).to(torch.int64) & 0x7FFF
        m11, e16 = (bits & 0x3FF) | 0x400, (bits >> 10) - 25       # normal numbers: m11 * 2^e16
        y = (sums * m11 << (bias + e16)).sum(2) >> shift
        return y.to(torch.int32), torch.zeros(1, dtype=torch.int32, device="cuda")
    return _exact_model(case, seed)


M64 = (1 << 64) - 1


def _mix(z):
    """splitmix64 of a Python integer."""
    z = (z + 0x9E3779B97F4A7C15) & M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
    return z ^ (z >> 31)


def _signed(v):
    return v - (1 << 64) if v >> 63 else v


def _mixed(start, count, key):
    """splitmix64((start + i) ^ key) for i < count, as int64 bit patterns."""
    def down(z, n):
        return (z >> n) & ((1 << (64 - n)) - 1)
    z = torch.arange(start, start + count, dtype=torch.int64, device="cuda") ^ _signed(key)
    z = z + _signed(0x9E3779B97F4A7C15)
    z = (z ^ down(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ down(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ down(z, 31)


class _Hashed:
    """The tensors that `Decoder.synthetic` fills from its counter-based generator."""

    def __init__(self, seed):
        self.seed = seed

    def _key(self, role, layer, stream):
        return _mix((self.seed & 0xFFFFFFFF) << 32 | ((layer * 32 + role) & 0xFFFFFF) << 8 | stream)

    def uniform(self, role, layer, stream, start, count, lo, hi):
        u = (_mixed(start, count, self._key(role, layer, stream)) >> 40) & 0xFFFFFF
        lo32, span = np.float32(lo), np.float32(hi) - np.float32(lo)
        return u.to(torch.float32) * (1.0 / (1 << 24)) * float(span) + float(lo32)

    def codes_scales(self, role, layer, r0, rows, K):
        h = _mixed(r0 * (K // 4), rows * (K // 4), self._key(role, layer, 1))
        u = torch.stack([(h >> (16 * k)) & 0xFFFF for k in range(4)], dim=1)
        codes = ((u >= 19661).to(torch.uint8) + (u >= 45875).to(torch.uint8)).view(rows, K)
        G = K // 128
        scales = self.uniform(role, layer, 2, r0 * G, rows * G, 0.01, 0.05).to(torch.float16).view(rows, G)
        return codes, scales

    def project(self, role, layer, M, x):
        K = x.shape[1]
        out = torch.empty((x.shape[0], M), dtype=torch.float64, device="cuda")
        for r in range(0, M, 8192):
            n = min(8192, M - r)
            out[:, r:r + n] = _project(*self.codes_scales(role, layer, r, n, K), x)
        return out

    def vector(self, role, layer, count, lo=0.8, hi=1.2):
        return self.uniform(role, layer, 3, 0, count, lo, hi).double()

    def embedding(self, token, E):
        """The row as the int16 table holds it: every weight as an integer at the row's smallest
        scale exponent, the largest shifted into 15 bits, the shift rounding down."""
        codes, scales = self.codes_scales(L.ROLE_TOK_EMB, 0, int(token), 1, E)
        bits = scales[0].view(torch.int16).to(torch.int64) & 0x7FFF
        m11, e16 = (bits & 0x3FF) | 0x400, (bits >> 10) - 25
        e0 = int(e16.min())
        v = ((codes.to(torch.int64) - 1).view(-1, 128) * (m11 << (e16 - e0))[:, None]).view(-1)
        shift = int(v.abs().max()).bit_length() - 15
        v = v >> shift if shift >= 0 else v << -shift
        return v.double() * 2.0 ** (e0 + shift)


def _attention(w, mc, l, h, freq):
    T, hd, nh, nkv = h.shape[0], mc.head_dim, mc.n_head, mc.n_kv_head
    q = w.project(L.ROLE_ATTN_Q, l, nh * hd * (2 if mc.attn_gated else 1), h).view(T, nh, -1)
    k = w.project(L.ROLE_ATTN_K, l, nkv * hd, h).view(T, nkv, hd)
    v = w.project(L.ROLE_ATTN_V, l, nkv * hd, h).view(T, nkv, hd)
    gate = q[:, :, hd:] if mc.attn_gated else None
    q = _rms(q[:, :, :hd], w.vector(L.ROLE_ATTN_Q_NORM, l, hd))
    k = _rms(k, w.vector(L.ROLE_ATTN_K_NORM, l, hd))
    # The angles are float32 products, as the model defines them.
    angle = (torch.arange(T, dtype=torch.float32, device="cuda")[:, None] * freq[None, :]).double()
    cos, sin, half = angle.cos()[:, None, :], angle.sin()[:, None, :], freq.numel()

    def rope(t):
        a, b = t[:, :, :half], t[:, :, half:2 * half]
        return torch.cat([a * cos - b * sin, a * sin + b * cos, t[:, :, 2 * half:]], dim=2)

    # The cache holds k and v in fp16.
    q, k, v = rope(q) / hd ** 0.5, rope(k).half().double(), v.half().double()
    out = torch.empty((T, nh, hd), dtype=torch.float64, device="cuda")
    mask = torch.ones((T, T), dtype=torch.bool, device="cuda").tril()
    for head in range(nh):
        g = head // (nh // nkv)
        s = (q[:, head] @ k[:, g].T).masked_fill(~mask, float("-inf"))
        out[:, head] = torch.softmax(s, dim=1) @ v[:, g]
    if gate is not None:
        out = out * torch.sigmoid(gate)
    return w.project(L.ROLE_ATTN_OUT, l, mc.n_embd, out.reshape(T, -1))


def _deltanet(w, mc, l, h, gates):
    T, nk, hk, nv, hv, taps = (h.shape[0], mc.dn_num_k_heads, mc.dn_k_head_dim, mc.dn_num_v_heads, mc.dn_v_head_dim,
                               mc.dn_conv_kernel)
    width = 2 * nk * hk + nv * hv
    raw = w.project(L.ROLE_ATTN_QKV, l, width, h)
    z = w.project(L.ROLE_ATTN_ZGATE, l, nv * hv, h).view(T, nv, hv)

    def gate_input(role):
        q, sc = gates[role, l]
        wt = (q.astype(np.float16).reshape(nv, -1, 32) * sc[:, :, None]).astype(np.float16).reshape(nv, -1)
        return h @ torch.from_numpy(wt.astype(np.float64)).cuda().T

    beta = torch.sigmoid(gate_input(L.ROLE_SSM_BETA))
    alpha = gate_input(L.ROLE_SSM_ALPHA) + w.vector(L.ROLE_SSM_DT, l, nv, -2.0, 0.5)
    a = -torch.exp(w.vector(L.ROLE_SSM_A, l, nv, -1.5, 0.5))
    decay = torch.exp(torch.nn.functional.softplus(alpha) * a)
    conv_w = w.vector(L.ROLE_SSM_CONV, l, width * taps, -0.5, 0.5).view(width, taps)
    padded = torch.cat([torch.zeros((taps - 1, width), dtype=torch.float64, device="cuda"), raw])
    c = _silu(sum(padded[i:i + T] * conv_w[:, i] for i in range(taps)))

    def unit(t):
        return t / t.norm(dim=-1, keepdim=True).clamp_min(EPS)

    q, k = unit(c[:, :nk * hk].view(T, nk, hk)), unit(c[:, nk * hk:2 * nk * hk].view(T, nk, hk))
    v = c[:, 2 * nk * hk:].reshape(T, nv, hv)
    heads = torch.arange(nv, device="cuda") % nk
    state = torch.zeros((nv, hv, hk), dtype=torch.float64, device="cuda")
    out = torch.empty((T, nv, hv), dtype=torch.float64, device="cuda")
    q, k = q[:, heads, :, None], k[:, heads, :, None]
    for t in range(T):
        state *= decay[t, :, None, None]
        delta = (v[t] - (state @ k[t])[:, :, 0]) * beta[t, :, None]
        state += delta[:, :, None] * k[t].transpose(1, 2)
        out[t] = (state @ q[t])[:, :, 0]
    out = _rms(out / hk ** 0.5, w.vector(L.ROLE_SSM_NORM, l, hv)) * _silu(z)
    grouped = torch.empty_like(out)
    grouped[:, heads * (nv // nk) + torch.arange(nv, device="cuda") // nk] = out
    return w.project(L.ROLE_SSM_OUT, l, mc.n_embd, grouped.reshape(T, -1))


def _exact_model(case, seed):
    mc = _model(case)
    w, gates, tokens = _Hashed(seed), _gate_rows(mc, seed), _tokens(case, mc, seed)
    n = mc.rope_dims or mc.head_dim
    f32 = np.float32
    freq = torch.tensor([f32(f32(mc.rope_theta) ** f32(-2.0 * i / n)) for i in range(n // 2)], device="cuda")
    E = mc.n_embd
    x = torch.stack([w.embedding(t, E) for t in tokens])
    for l in range(mc.n_layer):
        h = _rms(x, w.vector(L.ROLE_ATTN_NORM, l, E))
        x = x + (_deltanet(w, mc, l, h, gates) if mc.layer_type(l) == "deltanet" else _attention(w, mc, l, h, freq))
        h = _rms(x, w.vector(L.ROLE_FFN_NORM, l, E))
        act = _silu(w.project(L.ROLE_FFN_GATE, l, mc.ffn_dim, h)) * w.project(L.ROLE_FFN_UP, l, mc.ffn_dim, h)
        x = x + w.project(L.ROLE_FFN_DOWN, l, E, act)
    hidden = _rms(x, w.vector(L.ROLE_OUT_NORM, 0, E))
    role = L.ROLE_TOK_EMB if mc.tie_embeddings else L.ROLE_LM_HEAD
    if case["op"] != "score":
        return w.project(role, 0, mc.vocab, hidden[-1:])[0]
    logits = w.project(role, 0, mc.vocab, hidden[:-1])
    target = torch.from_numpy(tokens[1:].astype(np.int64)).cuda()
    return torch.logsumexp(logits, 1) - logits.gather(1, target[:, None])[:, 0], hidden
