"""The batched DeltaNet passes over a chunk (conv window, SiLU, q/k norm, scan and gated norm): conv
windows shorter and longer than the kernel's register window of four rows, in prompts cut at the conv
block's eight positions, one more and one less.

The tolerance is the other prefill tests' 2e-3 of the logits against the float oracle, whose KV rows
are fp16 as the decoder's are."""

import numpy as np
import pytest

from oracle.floatref import FloatRef
from trixium_amd import bons, configs as C, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kc", [2, 3, 4, 6])
def test_conv_windows_and_ragged_chunks(tmp_path, kc):
    from trixium_amd.model import Decoder
    cfg = C.TINY_HYBRID.replace(name=f"tiny-hybrid-conv{kc}", dn_conv_kernel=kc)
    p = str(tmp_path / "c.img")
    bons.write_image(cfg, synth.small_model_tensors(cfg, 40 + kc, True), 1, p, trit5=True)
    ref = FloatRef(bons.BONSReader(p), kv_fp16=True)
    tokens = [int(t) for t in np.random.default_rng(kc).integers(1, cfg.vocab, 46)]
    for chunk in (7, 8, 9, 64):
        dec = Decoder.from_image(p, prefill_chunk=chunk)
        ref.reset()
        at = 0
        for n in (2, 10, 18, 16):        # the last token of a piece is a step: 1, 9, 17 and 15 prefilled
            piece, at = tokens[at:at + n], at + n
            got = dec.forward(piece)
            for i, t in enumerate(piece):
                want = ref.step(t, want_logits=i == len(piece) - 1)
            err = float(np.max(np.abs(got - want)) / np.max(np.abs(want)))
            print("conv", kc, "chunk", chunk, "prefilled", n - 1, "err", err)
            assert err <= 2e-3
        dec.close()


def test_longest_chunk():
    """The longest chunk of a context that the decode attention takes, 8191 positions, against chunks of 512."""
    from trixium_amd.model import Decoder
    mc = C.TINY_HYBRID.replace(max_ctx=8192)
    toks = synth.random_prompt(mc, 8192, 2)
    out = []
    for chunk in (512, 8191):
        dec = Decoder.synthetic(mc, seed=2, prefill_chunk=chunk)
        out.append(dec.forward(toks).astype(np.float64))
        dec.close()
    assert np.max(np.abs(out[1] - out[0])) <= 2e-3 * np.max(np.abs(out[0]))


def test_value_heads_of_half_a_block(tmp_path):
    """Key heads of 128 with value heads of 8 rows: half of the scan's block of 16 rows is empty."""
    from trixium_amd.model import Decoder
    cfg = C.TINY_HYBRID.replace(name="tiny-hybrid-hv8", dn_k_head_dim=128, dn_v_head_dim=8, dn_num_v_heads=16)
    p = str(tmp_path / "c.img")
    bons.write_image(cfg, synth.small_model_tensors(cfg, 7, True), 1, p, trit5=True)
    ref = FloatRef(bons.BONSReader(p), kv_fp16=True)
    tokens = [int(t) for t in np.random.default_rng(7).integers(1, cfg.vocab, 60)]
    dec = Decoder.from_image(p, prefill_chunk=25)
    got = dec.forward(tokens)
    for i, t in enumerate(tokens):
        want = ref.step(t, want_logits=i == len(tokens) - 1)
    assert np.max(np.abs(got - want)) <= 2e-3 * np.max(np.abs(want))
    dec.close()
