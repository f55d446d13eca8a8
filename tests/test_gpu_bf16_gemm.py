"""The bf16 GEMM of M > 32 rows (bf16_gemm.hip): shapes its dispatch rule
takes on a 256-CU part, at the edges of its tiles and stages: N not a multiple
of 8, 16 or 128, K not a multiple of the 64-k stage, one stage (K = 8, 64), odd
numbers of stages, M one row past each tile height; the tile-major copy
(N % 16 == 0, K % 256 == 0) in both tile heights, with a last weight block that is
not whole, and past K = 1024. Outputs must equal, bit for bit, those of calls of
at most 32 rows, which the stream kernel serves (every row of a batched call
equals the single-row call on it), for normal data, for operands spread over
2^-60 .. 2^60 and for non-finite activations; and the calls must launch it."""
import pytest
import torch

from launched_kernels import launched_kernels

pytestmark = pytest.mark.gpu


def _inputs(dev, N, K, M, spread, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    out = []
    for rows in (N, M):
        t = torch.randn(rows, K, device=dev, generator=g)
        if spread:
            t = t * torch.exp2(torch.randint(-60, 61, (rows, K), device=dev, generator=g).float())
        out.append(t.to(torch.bfloat16))
    return out


def _same(a, b, label):
    diff = (a.view(torch.int16) != b.view(torch.int16)) & ~(a.isnan() & b.isnan())
    torch.cuda.synchronize()
    assert int(diff.sum()) == 0, (label, int(diff.sum()), a.shape)


@pytest.mark.parametrize("N,K,M", [(33000, 1024, 33), (33001, 1000, 64), (16384, 512, 97),
                                   (50003, 8, 65), (20007, 64, 129), (40001, 72, 257),
                                   (9001, 1088, 96), (4104, 3072, 150),
                                   # tile-major copy: 64-row tiles, 128-row ones
                                   (33008, 1024, 33), (33008, 1024, 64), (8208, 3072, 64),
                                   (24592, 256, 65), (8208, 2048, 130)])
@pytest.mark.parametrize("spread", [False, True])
def test_gemm_equals_stream_kernel(w4, dev, N, K, M, spread):
    w, x = _inputs(dev, N, K, M, spread, 0xBF6 + N + K + M)
    for bad in (False, True):
        if bad:
            x[M // 2, K // 3] = float("inf")
            x[M - 1, K - 1] = float("nan")
        ref = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        for m0 in range(0, M, 32):
            xc = x[m0:m0 + 32].contiguous()
            w4.bf16_gemv_any(w, xc, N, K, xc.shape[0], y=ref[m0:m0 + 32])
        y = torch.empty_like(ref)
        w4.bf16_gemv_any(w, x, N, K, M, y=y)
        _same(y, ref, ("file", bad))
        w4.bf16_gemv_any(w, x, N, K, M, y=y, variant="stream")  # the chunks, forced
        _same(y, ref, ("stream", bad))
        if N % 16 == 0 and K % 256 == 0:
            y = torch.empty_like(ref)
            w4.bf16_gemv_prepacked(w4.bf16_repack(w, N, K), x, N, K, M, y=y)
            _same(y, ref, ("packed", bad))
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        y = torch.empty_like(ref)
        calls = [lambda: w4.bf16_gemv_any(w, x, N, K, M, y=y)]
        if N % 16 == 0 and K % 256 == 0:
            p = w4.bf16_repack(w, N, K)
            calls.append(lambda: w4.bf16_gemv_prepacked(p, x, N, K, M, y=y))
        for call in calls:
            names = launched_kernels(call)
            assert len(names) == 1 and "bf16_gemm" in names[0], names
    buf = torch.empty(M * N + 1, dtype=torch.bfloat16, device=dev)
    y = buf[1:].view(M, N)  # an output base off 16 bytes
    w4.bf16_gemv_any(w, x, N, K, M, y=y)
    _same(y, ref, "output base")
