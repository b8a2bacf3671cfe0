"""Transposed convolutions whose output phases are rows of one convolution,
against the oracle and against the K-split kernels: strides whose phases are
stored 16 bytes at a time (4, 8) and one by one (2, 3, 5), whole and padded
row tiles, tile counts of every kernel, lengths off the 128-position blocks;
and a launch long enough to be taken unforced, whose recorded maximum scales
a fused residual unit's operand."""
import pytest

import qtts
from oracle import oracle
from shapes import rel_err, within

pytestmark = pytest.mark.gpu


def _decoder(ctx, vocos):
    cfg = qtts.DecoderConfig(hidden=32, heads=2, head_dim=16, inter=64, window=8, codebook_dim=16, codebook_size=64,
                             vq_dim=32, latent=32, num_rest=3, layers=1, upsample=(1,), vocos_channels=64,
                             vocos=vocos, dilations=(3,), rope_rows=200)
    w = qtts.DecoderWeights(23, cfg)
    return w, qtts.SpeechDecoder(ctx, w)


# f32 rounding through the same stages as the small decoder's (2e-6 there)
TIGHT = 3e-5


@pytest.mark.parametrize("stride,cout,frames", [
    (2, 32, 129),   # 2 tiles: k_dec_conv_mfma
    (3, 32, 127),   # 3 tiles
    (3, 40, 1),     # 4 tiles, the last padded
    (4, 24, 128),   # 3 tiles, 16-byte stores
    (4, 28, 130),   # 4 tiles, the last half padding, 16-byte stores
    (5, 20, 128),   # 4 tiles, padded
    (5, 32, 31),    # 5 tiles: k_dec_conv_mfma, one tile at a time
    (8, 16, 129),   # 4 tiles, 16-byte stores
])
def test_phases_as_rows(ctx, monkeypatch, stride, cout, frames):
    w, dec = _decoder(ctx, ((64, cout, 2 * stride, stride),))
    codes = w.synthetic_codes(24, frames)
    ref = oracle.decode_to_audio(w, codes)
    monkeypatch.setenv("QTTS_DEC_CONV", "tiles")
    got = dec.decode_to_audio(codes)
    monkeypatch.setenv("QTTS_DEC_CONV", "split")
    split = dec.decode_to_audio(codes)
    print(f"stride {stride}, {cout} channels: rel err {rel_err(got, ref):.2e}, split {rel_err(split, ref):.2e}")
    assert got.shape == split.shape == ref.shape
    assert within(got, ref, tight=TIGHT)
    assert within(split, ref, tight=TIGHT)


def test_recorded_maximum(ctx, monkeypatch):
    # 8,192 positions of 64 channels into 8 x 96 rows: 1,536 blocks at one
    # tile, then units of 96 channels
    w, dec = _decoder(ctx, ((64, 64, 16, 8), (64, 64, 16, 8), (64, 96, 16, 8)))
    codes = w.synthetic_codes(25, 128)
    ref = oracle.decode_to_audio(w, codes)
    got = dec.decode_to_audio(codes)
    monkeypatch.setenv("QTTS_DEC_CONV", "split")
    split = dec.decode_to_audio(codes)
    print(f"{got.size} samples: rel err {rel_err(got, ref):.2e}, split {rel_err(split, ref):.2e}")
    assert got.shape == ref.shape
    assert within(got, ref, tight=TIGHT)
    assert rel_err(got, ref) <= 3.0 * rel_err(split, ref) + 1e-6
