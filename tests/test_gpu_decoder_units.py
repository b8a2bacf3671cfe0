"""Residual units of 96, 192 and 384 channels (one launch each) against the oracle
and against the same decoder with every layer a launch of its own: lengths off
the 64-, 128- and 256-position blocks and shorter than a window, the largest
dilation the unit takes and one past it, SnakeBeta factors up to e^3, and the
first convolution's operand scale where SnakeBeta's largest factor says
nothing about its largest value."""
import numpy as np
import pytest

import qtts
from oracle import oracle
from shapes import rel_err, within

pytestmark = pytest.mark.gpu


UNITS = ((64, 384, 2, 1), (384, 192, 6, 3), (192, 96, 4, 2))


def _decoder(ctx, dilations, big=False, change=None, vocos=UNITS):
    cfg = qtts.DecoderConfig(hidden=32, heads=2, head_dim=16, inter=64, window=8, codebook_dim=16, codebook_size=64,
                             vq_dim=32, latent=32, num_rest=3, layers=1, upsample=(1,), vocos_channels=64,
                             vocos=vocos, dilations=dilations, rope_rows=64)
    w = qtts.DecoderWeights(17, cfg)
    if big:
        # SnakeBeta at arguments of tens of periods.  Its slope 1 + exp(alpha -
        # beta) sin(2 t) stays below 2, so that four units' two SnakeBetas
        # magnify a rounding at most 2^8 times (steeper ones are chaotic and
        # compare nothing).
        for b in w.blocks:
            for r in b["residuals"]:
                r["act1_alpha"][::5] = r["act1_beta"][::5] = 3.0
                r["act2_alpha"][::3] = r["act2_beta"][::3] = 4.0
    if change:
        change(w)
    return w, qtts.SpeechDecoder(ctx, w)


@pytest.mark.parametrize("frames,dilations,big", [(1, (1, 3, 9), False), (43, (1, 3, 9), False), (44, (10,), False),
                                                  (60, (11, 2), False), (64, (9, 1), True), (128, (3,), True)])
def test_residual_units(ctx, monkeypatch, frames, dilations, big):
    w, dec = _decoder(ctx, dilations, big)
    codes = w.synthetic_codes(18, frames)
    got = dec.decode_to_audio(codes)
    ref = oracle.decode_to_audio(w, codes)
    monkeypatch.setenv("QTTS_DEC_CONV", "tiles")
    apart = dec.decode_to_audio(codes)
    print(f"{frames} frames: {got.size} samples, rel err {rel_err(got, ref):.2e}, apart {rel_err(apart, ref):.2e}")
    assert got.shape == ref.shape
    # f32 rounding through the same stages as the small decoder's (2e-6 there),
    # times the magnification above where it applies
    assert within(got, ref, tight=2.0 ** 8 * 2e-6 if big else 3e-5)
    assert rel_err(got, ref) <= 3.0 * rel_err(apart, ref) + 1e-6


def _zero_channel(conv, c):
    """Output channel c of a causal convolution: weights [out][in][k]."""
    conv["weight"].reshape(conv["out_channels"], -1)[c] = 0.0
    conv["bias"][c] = 0.0


def _silent_channel(w):
    """A channel that stays 0 and whose SnakeBeta would reach e^30."""
    for b in w.blocks:
        u = b["upsample"]
        u["weight"].reshape(u["in_channels"], u["out_channels"], -1)[:, 5] = 0.0
        u["bias"][5] = 0.0
        for r in b["residuals"]:
            r["act1_beta"][5] = -30.0
            _zero_channel(r["conv2"], 5)


def _quiet(w):
    """A signal of 1e-9 under SnakeBetas that would reach 1 and more."""
    w.vocos_init["weight"] *= 1e-9
    for c in [w.vocos_init, w.output_conv] + [b["upsample"] for b in w.blocks] + [
            r[n] for b in w.blocks for r in b["residuals"] for n in ("conv1", "conv2")]:
        c["bias"][:] = 0.0


# the units' first bound by a launch of its own, and (1,536 blocks) recorded by
# the transposed convolution
@pytest.mark.parametrize("frames,vocos", [(43, UNITS), (128, ((64, 64, 16, 8), (64, 64, 16, 8), (64, 96, 16, 8)))])
@pytest.mark.parametrize("change", [_silent_channel, _quiet])
def test_operand_scale_follows_the_signal(ctx, monkeypatch, frames, vocos, change):
    w, dec = _decoder(ctx, (1, 3, 9), change=change, vocos=vocos)
    codes = w.synthetic_codes(19, frames)
    got = dec.decode_to_audio(codes)
    monkeypatch.setenv("QTTS_DEC_CONV", "tiles")
    apart = dec.decode_to_audio(codes)
    ref = oracle.decode_to_audio(w, codes)
    print(f"{frames} frames: rel err {rel_err(got, ref):.2e}, apart {rel_err(apart, ref):.2e}")
    assert np.max(np.abs(ref)) > 0.0 and within(got, ref, tight=3e-5)
    assert rel_err(got, ref) <= 3.0 * rel_err(apart, ref) + 1e-6
