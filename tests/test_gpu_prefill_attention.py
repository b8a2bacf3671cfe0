"""The prefill's attention up to 16 rows (one launch with QK-norm, RoPE and
the append) and past 64 (32-row tiles, four waves over the keys) against the
oracle: the limits and one past them, whole and ragged tiles, one to four
query heads per kv head; and a row of NaNs, which the rows before it must not
see and which must not cost the rows after it anything."""
import time

import numpy as np
import pytest

import qtts
from oracle import oracle
from shapes import within

pytestmark = pytest.mark.gpu


def _talker(ctx, heads, kv_heads, seed=31):
    cfg = qtts.StackConfig(layers=2, hidden=256, heads=heads, kv_heads=kv_heads, head_dim=128, inter=512, vocab=320,
                           max_position=4096)
    tw = qtts.TalkerWeights(seed, cfg)
    return cfg, tw, qtts.Talker(ctx, tw)


@pytest.mark.parametrize("heads,kv_heads", [(4, 4), (4, 2), (4, 1), (18, 18)])
@pytest.mark.parametrize("rows", [8, 9, 16, 17, 64, 65, 96, 129, 257])
def test_prefill_attention(ctx, rows, heads, kv_heads):
    cfg, tw, t = _talker(ctx, heads, kv_heads)
    ot = oracle.Talker(tw)
    x = qtts.synth_normal_f32(31, f"attn.x.{rows}", rows * cfg.hidden)
    kv, okv = t.new_kv(rows + 3), ot.new_kv(rows + 3)
    lh, olh = t.prefill_talker_raw(x, rows, kv), ot.prefill_talker_raw(x, rows, okv)
    assert within(lh, olh)
    for got, ref in zip(kv.store(), okv.store()):  # layer 1's rows carry every row's attention
        assert within(got, ref)


@pytest.mark.parametrize("rows,bad", [(16, 9), (96, 95), (100, 70), (129, 128), (200, 3)])
def test_prefill_rows_before_a_nan_row_are_unchanged(ctx, rows, bad):
    cfg, tw, t = _talker(ctx, 4, 2)
    x = qtts.synth_normal_f32(32, f"nan.x.{rows}", rows * cfg.hidden).reshape(rows, -1).copy()
    kv = t.new_kv(rows)
    t.prefill_talker_raw(x, rows, kv)
    clean = kv.store()
    x[bad, 7] = np.inf  # its normed row is NaN
    kv.clear()
    t.prefill_talker_raw(x, rows, kv)
    for got, ref in zip(kv.store(), clean):
        assert np.all(np.isfinite(got[:, :bad])) and within(got[:, :bad], ref[:, :bad])
        assert np.all(np.isnan(got[1, bad:]).any(axis=(1, 2)))


@pytest.mark.parametrize("bad", [slice(3, 4), slice(1499, 1500), slice(0, 1500, 32)])
def test_prefill_time_with_nan_rows(ctx, bad):
    """Where a tile's own rows hold a NaN its wave goes over its keys once more
    on the vector units: 1.5 to 1.95 times the whole call here (20 times when
    every tile after the bad row did it row by row)."""
    rows = 1500
    cfg, tw, t = _talker(ctx, 4, 2)
    x = qtts.synth_normal_f32(33, "nan.t", rows * cfg.hidden).reshape(rows, -1).copy()
    kv = t.new_kv(rows)

    def best():
        times = []
        for _ in range(5):
            kv.clear()
            t0 = time.perf_counter()
            t.prefill_talker_raw(x, rows, kv)
            times.append(time.perf_counter() - t0)
        return min(times)

    clean = best()
    x[bad, 7] = np.inf
    slow = best()
    print(f"{rows} rows: {clean * 1e6:.0f} us, with NaN rows {slow * 1e6:.0f}")
    assert slow < 3.0 * clean
