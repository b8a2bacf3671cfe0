"""The scratch of qtts_gemm_device: settled by a weight's first product at any
number of rows, and kept when a larger weight outgrows it, so that captured
products stay valid."""
import pytest
import torch

import qtts

pytestmark = pytest.mark.gpu


def _weight(ctx, K, N):
    return qtts.DeviceQ4(ctx, qtts.Q4Weight.synthetic(51, f"scratch.{K}.{N}", K, N))


def _rows(K, rows):
    return torch.from_numpy(qtts.synth_normal_f32(51, f"scratch.x.{rows}", rows * K)).cuda()


@pytest.mark.parametrize("K,N", [(2048, 1056), (6144, 2048)])
def test_row_counts_allocate_nothing(K, N):
    ctx = qtts.Context(0)
    w = _weight(ctx, K, N)
    xs = {rows: _rows(K, rows) for rows in (64, 1000, 65, 353, 2049, 8)}
    ys = {rows: torch.empty(rows * N, device="cuda") for rows in xs}
    first = torch.empty(64 * N, device="cuda")
    torch.cuda.synchronize()
    w.gemm_device(xs[64].data_ptr(), 64, first.data_ptr())
    ctx.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for rows, x in xs.items():
        w.gemm_device(x.data_ptr(), rows, ys[rows].data_ptr())
    ctx.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 2 ** 21  # 25 and 122 MB when each row count had its own
    w.gemm_device(xs[64].data_ptr(), 64, ys[64].data_ptr())
    ctx.synchronize()
    assert torch.equal(ys[64], first)
    w.close()
    ctx.close()


def test_captured_products_outlive_a_larger_weight():
    ctx = qtts.Context(0)
    K, N = 272, 96
    w, larger = _weight(ctx, K, N), _weight(ctx, 4096, 1024)
    stream = torch.cuda.ExternalStream(ctx.stream)
    rows = (64, 1000)
    xs = [_rows(K, r) for r in rows]
    ref, got = ([torch.empty(r * N, device="cuda") for r in rows] for _ in range(2))
    big, out = _rows(4096, 300), torch.empty(300 * 1024, device="cuda")
    torch.cuda.synchronize()
    w.gemm_device(xs[0].data_ptr(), 8, got[0].data_ptr())  # the first product: what may allocate
    ctx.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for x, r, y in zip(xs, rows, got):
            w.gemm_device(x.data_ptr(), r, y.data_ptr())
    for x, r, y in zip(xs, rows, ref):
        w.gemm_device(x.data_ptr(), r, y.data_ptr())
    ctx.synchronize()
    for _ in range(4):
        larger.gemm_device(big.data_ptr(), 300, out.data_ptr())
        ctx.synchronize()
        for y in got:
            y.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        ctx.synchronize()
        for y, r in zip(got, ref):
            assert torch.equal(y, r)
    del graph
    w.close()
    larger.close()
    ctx.close()
