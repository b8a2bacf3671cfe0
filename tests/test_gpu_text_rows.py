"""The text projection's two paths (up to 4 rows: the GEMV; from 5 the matrix
cores with all four partial products) against float64 at the edges of both,
and the rows of one call against the same tokens one at a time."""
import numpy as np
import pytest
import torch

import qtts

pytestmark = pytest.mark.gpu

HIDDEN, TEXT_HIDDEN = 256, 192


def _text(ctx, hidden, text_hidden):
    cfg = qtts.StackConfig(layers=1, hidden=hidden, heads=2, kv_heads=1, head_dim=128, inter=256, vocab=320,
                           max_position=64)
    w = qtts.TextWeights(41, qtts.TEXT_VOCAB_1P7B, text_hidden, hidden)
    t = qtts.Talker(ctx, qtts.TalkerWeights(41, cfg))
    t.attach_text(w)
    return t, w


@pytest.fixture(scope="module")
def text(ctx):
    return _text(ctx, HIDDEN, TEXT_HIDDEN)


@pytest.fixture(scope="module")
def wide(ctx):
    return _text(ctx, 2048, 2048)


def _check_rows(text, rows, width, rms):
    t, w = text
    tok = np.random.default_rng(rows).integers(0, qtts.TEXT_VOCAB_1P7B, rows).astype(np.uint32)
    got = t.build_trailing_text(np.concatenate([[0], tok[:-1]]))  # tokens[1..], then TTS_EOS
    tok[-1] = qtts.TTS_EOS
    e = w.text_embedding
    x = qtts.Q4Weight(e.packed[tok], e.scales[tok], rows, e.n).dequantize().astype(np.float64)
    f1, f2 = w.fc1.dequantize().astype(np.float64), w.fc2.dequantize().astype(np.float64)
    h = x @ f1 + w.fc1_bias
    s = h / (1.0 + np.exp(-h))
    # per product: x's split (2^-22) and one f32 rounding per 16-row MFMA of
    # each of four, on the magnitudes; silu' <= 1.1 carries fc1's on, silu
    # itself rounds a few times
    eps = 2.0 ** -22 + (width / 4 + 32) * 2.0 ** -24
    dh = eps * (np.abs(x) @ np.abs(f1) + np.abs(w.fc1_bias))
    bound = (1.1 * dh + 2.0 ** -20 * np.abs(s)) @ np.abs(f2) + eps * (np.abs(s) @ np.abs(f2) + np.abs(w.fc2_bias))
    err = np.abs(got - (s @ f2 + w.fc2_bias))
    assert np.all(err <= bound), float(np.max(err / bound))
    assert np.linalg.norm(err) <= rms * np.linalg.norm(got)
    one = np.stack([t.embed_text_token(int(v)) for v in tok[:3]])
    far = np.abs(one - (s @ f2 + w.fc2_bias)[:3])
    assert np.all(far <= bound[:3])
    print(f"{rows} rows: from 64 bits {err[:3].max() / np.abs(one).max():.1e}, one at a time {far.max() / np.abs(one).max():.1e}")
    return got[:3], one


@pytest.mark.parametrize("rows", [1, 4, 5, 32, 33, 64, 65, 97, 300])
def test_text_projection_rows(text, rows):
    got, one = _check_rows(text, rows, TEXT_HIDDEN, 4e-7)
    assert np.allclose(got, one, rtol=0, atol=1e-6 * np.abs(one).max())


# 2048 -> 2048: four chunks of K up to 16 rows, 17 to 64, and five in row
# blocks, each with all four partial products
@pytest.mark.parametrize("rows", [5, 16, 17, 64, 65, 96, 200])
def test_text_projection_in_chunks(wide, rows):
    _check_rows(wide, rows, 2048, 4e-7)


def test_first_projection_makes_no_operand_copies():
    """The matrix cores' copies and scratch come with the text weights: the
    first projection allocates its rows and no more (three buffers of 96 x
    2048 floats and the tokens, each at most rounded up to 2 MiB)."""
    ctx = qtts.Context(0)
    cfg = qtts.StackConfig(layers=1, hidden=2048, heads=2, kv_heads=1, head_dim=128, inter=256, vocab=320,
                           max_position=64)
    t = qtts.Talker(ctx, qtts.TalkerWeights(43, cfg))
    t.attach_text(qtts.TextWeights(43, qtts.TEXT_VOCAB_1P7B, 2048, 2048))
    t.embed_text_token(5)
    free = torch.cuda.mem_get_info()[0]
    first = t.build_trailing_text(np.arange(97, dtype=np.uint32))
    assert free - torch.cuda.mem_get_info()[0] <= 4 * 2 ** 21
    assert np.array_equal(first, t.build_trailing_text(np.arange(97, dtype=np.uint32)))
    ctx.close()
