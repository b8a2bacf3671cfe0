"""The Q4 product of 8 and more rows against float64, on every kernel variant and
at the edges of its tiles: one row past a pass, rows off the 16-, 32- and
128-row tiles, an odd number of 16-row K steps, panel counts off a block's 4 or
8, one and several K chunks; and the scale split's last accepted scales."""
import time

import numpy as np
import pytest
import torch

import qtts

pytestmark = pytest.mark.gpu


def _bound(x, w, K):
    """Per output: the terms' dropped part (|xl| <= 2^-12 |x| times |sb| <=
    2^-8 s, one bit spare) and one f32 rounding per 16-row product of each of
    the three partial products, on the sum of magnitudes."""
    return (2.0 ** -19 + (3 * K / 16 + 32) * 2.0 ** -24) * (np.abs(x.astype(np.float64)) @ np.abs(w))


# tests/test_gemm_plans.py holds these to every kernel variant that a product
# can take, with one chunk of K and with several.
SHAPES = [
    # up to 16 rows
    (8, 16, 32), (9, 48, 96), (15, 272, 1056), (16, 1040, 2048), (13, 2064, 64), (16, 6144, 2048), (12, 512, 64),
    (11, 144, 96), (10, 1024, 96),
    # 17 to 64: one and two 32-row tiles, 1 to 16 steps a wave
    (17, 1040, 96), (18, 2048, 2048), (31, 2048, 4096), (32, 16, 6144), (33, 6144, 2048), (40, 272, 96), (48, 1040, 12288),
    (20, 1040, 12288), (24, 6144, 2048), (63, 2048, 2048), (64, 2064, 4096), (50, 48, 6176),
    (30, 144, 96), (55, 256, 64), (48, 2048, 4096), (20, 272, 64), (20, 1024, 64), (40, 1024, 64),
    # more, in row blocks: 1 to 4 tiles of 4 panels
    (65, 1040, 160), (96, 2048, 2048), (97, 16, 32), (128, 48, 288), (129, 6144, 96), (300, 1024, 1056),
    (1000, 272, 2048), (1064, 2048, 4096), (4097, 32, 64), (1064, 2048, 2048), (500, 2048, 6144), (1000, 1024, 6176),
    (160, 6144, 2048), (400, 272, 6176), (70, 2048, 4096), (200, 272, 12288), (1000, 3072, 1056),
    # 4 tiles of 8 panels, whole and with a part of a block past the last panel
    (1064, 2048, 12288), (1000, 6144, 2048), (1030, 2064, 12320), (200, 6144, 4128),
    # two passes
    (65, 2048, 8192), (80, 1040, 16384), (96, 1024, 8224),
]


@pytest.mark.parametrize("rows,K,N", SHAPES)
def test_gemm_row_blocks(ctx, rows, K, N):
    w = qtts.Q4Weight.synthetic(21, f"tiles.{K}.{N}", K, N)
    x = qtts.synth_normal_f32(21, f"tiles.x.{rows}.{K}", rows * K).reshape(rows, K)
    x[rows // 2] *= 1e4
    x[rows - 1] *= 1e-6
    d = qtts.DeviceQ4(ctx, w)
    y = d.gemm(x, rows).reshape(rows, N)
    wd = w.dequantize().astype(np.float64)
    err = np.abs(y - x.astype(np.float64) @ wd)
    assert np.all(err <= _bound(x, wd, K) + 1e-38), float(np.max(err / (_bound(x, wd, K) + 1e-38)))
    assert np.array_equal(y, d.gemm(x, rows).reshape(rows, N))


@pytest.mark.parametrize("rows", [16, 80])
@pytest.mark.parametrize("scale", [8188.0, 8160.0, 8128.0, 4100.0, 6e-8, 6.1e-5])
def test_gemm_scale_split_is_exact(ctx, rows, scale):
    """One-hot rows give the dequantized rows bit for bit: s = sa + sb exactly,
    also where rounding sa up would pass binary16."""
    K, N = 96, 64
    w = qtts.Q4Weight.synthetic(22, "split", K, N)
    w.scales[:] = np.float16(scale).view(np.uint16)
    w.scales[1::2] += np.arange(K // 2, dtype=np.uint16)[:, None] if scale < 8000 else 0
    x = np.zeros((rows, K), dtype=np.float32)
    x[np.arange(rows), np.arange(rows) * 7 % K] = 1.0
    y = qtts.DeviceQ4(ctx, w).gemm(x, rows).reshape(rows, N)
    assert np.array_equal(y, w.dequantize()[np.arange(rows) * 7 % K])


@pytest.mark.parametrize("rows", [65, 96])
def test_rows_past_a_pass_cost_no_more_than_two(ctx, rows):
    """Wide weights, read from memory: one call of 65 to 96 rows against one of
    64 and one of 32 (row blocks took 1.2 times as long)."""
    K, N = 2048, 12288
    ws = [qtts.DeviceQ4(ctx, qtts.Q4Weight.synthetic(23, f"wide.{i}", K, N)) for i in range(8)]
    x = torch.from_numpy(qtts.synth_normal_f32(23, "wide.x", rows * K)).cuda()
    y = torch.empty(rows * N, device="cuda")
    torch.cuda.synchronize()

    def best(parts):
        times = []
        for _ in range(12):
            t0 = time.perf_counter()
            for _ in range(4):
                for w in ws:
                    for m in parts:
                        w.gemm_device(x.data_ptr(), m, y.data_ptr())
            ctx.synchronize()
            times.append(time.perf_counter() - t0)
        return min(times)

    one, two = best([rows]), best([64, 32])
    print(f"{rows} rows: {one / 32 * 1e6:.1f} us, in two calls {two / 32 * 1e6:.1f}")
    assert one < 1.12 * two
