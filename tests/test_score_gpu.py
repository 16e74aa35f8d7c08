"""Decoder.score over the batched prefill (model/fastref.py:244-273), for models with a ternary LM head:
NLLs and hidden states against one-position forwards, and what the call leaves behind."""

import ctypes

import numpy as np
import pytest

from trixium_amd import _lib, bons, configs as C, layout as L
from trixium_amd import synth
from trixium_amd.model import Decoder, make_config

pytestmark = pytest.mark.gpu


def _rel_err(got, ref):
    return float(np.max(np.abs(np.asarray(got, np.float64) - ref)) / np.max(np.abs(ref)))


# One and two tokens, three and four (the fewest that are batched), one and two of the head's blocks of 128 positions with remainders; a rotated model.
@pytest.mark.parametrize("mc,rot", [(C.TINY, 0), (C.TINY_HYBRID, 0), (C.TINY, 128)])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 128, 129, 300])
def test_score_matches_forwards(mc, rot, n):
    mc = mc.replace(max_ctx=320)
    toks = synth.random_prompt(mc, n, n)
    dec = Decoder.synthetic(mc, seed=3, hadamard_block=rot)
    dec.reset()
    logits, hidden = [], []
    for t in toks:
        logits.append(dec.forward([t]).astype(np.float64))
        hidden.append(dec.hidden())
    want = [np.log(np.exp(lg - lg.max()).sum()) + lg.max() - lg[toks[i + 1]] for i, lg in enumerate(logits[:-1])]
    nll, hid = dec.score(toks)
    print(mc.name, n, "hidden err", _rel_err(hid, np.stack(hidden)), flush=True)
    assert _rel_err(hid, np.stack(hidden)) <= 2e-3
    assert nll.shape == (n - 1,) and np.all(np.abs(nll - want) <= 2e-3 * max(1.0, np.max(np.abs(want), initial=0)))
    # The last position's outputs and state are a forward's.
    assert dec.position() == n - 1
    assert _rel_err(dec.logits(), logits[-1]) <= 2e-3
    nxt = dec.forward([toks[0]])
    dec.reset()
    for t in toks:
        dec.forward([t])
    assert _rel_err(nxt, dec.forward([toks[0]])) <= 2e-3
    # With the sampler on (it draws at every position) the positions run one by one.
    dec.set_sampling(0.8, 0.9, 1.1, 7)
    nll1, hid1 = dec.score(toks)
    assert _rel_err(hid1, hid) <= 2e-3 and np.all(np.abs(nll1 - want) <= 2e-3 * max(1.0, np.max(np.abs(want), initial=0)))
    dec.close()


def test_kv_pin_holds_through_a_score():
    """A pin holds for the next reset, which is the score's own, also where the model's head (here in the other
    code format) is one that the batched pass does not take."""
    mc = C.TINY.replace(tie_embeddings=False)
    dec = Decoder(mc, make_config(mc, L.KIND_TERNARY5, L.KIND_TERNARY, False, 1, L.KIND_TERNARY5))
    ranges = np.array([0.01, 0.04, 0.8, 0.4], np.float32)
    _lib.call("trx_model_synthesize", dec._h, 3, ranges.ctypes.data_as(ctypes.POINTER(ctypes.c_float)))
    toks = synth.random_prompt(mc, 20, 1)
    for pin in (9, 12):
        dec.set_kv_ring(1, pin)
        dec.score(toks)
        assert dec.kv_pin == pin
    dec.close()


def test_nan_logit_shows():
    """One vocabulary row whose scale is NaN: every position's logits hold one, and no NLL hides it."""
    mc = C.TINY.replace(vocab=1000)
    dec = Decoder.synthetic(mc, seed=5)
    rng = np.random.default_rng(5)
    codes = rng.integers(0, 3, (mc.vocab, mc.n_embd)).astype(np.uint8)
    scales = rng.uniform(0.01, 0.05, (mc.vocab, mc.n_embd // 128)).astype(np.float16)
    scales[777, 1] = np.nan
    dec.set_tensor(L.ROLE_TOK_EMB, 0, bons.encode_rows(L.KIND_TERNARY5, mc.n_embd, scales, codes))
    nll, _ = dec.score(rng.integers(0, 700, 20))
    assert np.isnan(nll).all()
    dec.close()
