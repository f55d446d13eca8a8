"""Which kernel the dispatch rules pick on a 256-CU part, at shapes where both
sides were timed: where a rule on the new kernel's own tiles alone (the wide
GEMM and its k-slices, the SwiGLU GEMM, the bf16 GEMM) had taken calls that the
kernel beside it serves faster, and beside them shapes that it keeps."""
import pytest
import torch

from launched_kernels import launched_kernels

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _part(dev):
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the shapes stand at the rules' lines of a 256-CU part")


def _weights(dev, N, K):
    return (torch.zeros(N, K // 2, dtype=torch.uint8, device=dev),
            torch.ones(N, K // 128, dtype=torch.float16, device=dev))


def _x(dev, M, K):
    return torch.zeros(M, K, dtype=torch.bfloat16, device=dev)


@pytest.mark.parametrize("packed,N,K,M,kernel", [
    # M one row into a second 64-row tile, or a third 32-row one
    (False, 20342, 1024, 80, "gemm32_split"), (False, 41863, 1024, 65, "gemm_unit"),
    (False, 22110, 1024, 160, "gemm_unit"), (False, 19595, 2048, 65, "gemm_unit"),
    (True, 50045, 2048, 72, "gemm_unit"), (True, 40335, 3584, 72, "gemm_unit"),
    # N of a few rows, very many activation rows
    (True, 19, 1024, 16391, "gemm32_split"), (False, 17, 2048, 7735, "gemm_unit"),
    # what the wide kernel keeps, ragged sizes among them
    (False, 6144, 1024, 2048, "gemm_wide"), (True, 4096, 1024, 1024, "gemm_wide"),
    (True, 248320, 1024, 256, "gemm_wide"), (False, 22420, 512, 129, "gemm_wide"),
    (False, 3584, 3584, 777, "gemm_wide"), (True, 6152, 640, 513, "gemm_wide"),
    # its k-slices over three units: column tiles even in number, odd, and few
    # 128 x 32 tiles
    (True, 3050, 3072, 276, "gemm_unit"), (True, 1130, 3072, 768, "gemm_wide"),
    (True, 2216, 2816, 227, "gemm_wide"), (True, 1024, 3584, 777, "gemm_wide")])
def test_prefill_kernel(w4, dev, packed, N, K, M, kernel):
    w, s = _weights(dev, N, K)
    x, y = _x(dev, M, K), torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    if packed:
        p = w4.repack(w, s, N, K)
        names = launched_kernels(lambda: w4.gemv_prepacked(p, x, N, K, M, y=y))
    else:
        names = launched_kernels(lambda: w4.gemv(w, s, x, N, K, M, y=y))
    assert len(names) == 1 and kernel in names[0], names


@pytest.mark.parametrize("packed,Ns,K,M,kernel", [
    (False, (18, 23, 33), 1024, 11605, "gemm_unit"), (True, (28, 47), 1024, 8091, "gemm_unit"),
    (True, (6144, 2048, 16, 16), 1024, 1024, "gemm_wide"),
    (False, (3584, 3584), 1024, 512, "gemm_wide"),
    # 17 to 32 rows of long K: one 64-row block past a round, and a round
    (True, (239, 8145, 7938), 2560, 17, "w4a16_stream"),
    (False, (9926, 1951, 4454), 2432, 25, "w4a16_stream"),
    (True, (256, 8128, 8000), 2560, 17, "gemm_unit")])
def test_prefill_group_kernel(w4, dev, packed, Ns, K, M, kernel):
    pairs = [_weights(dev, N, K) for N in Ns]
    x = _x(dev, M, K)
    ys = [torch.empty(M, N, dtype=torch.bfloat16, device=dev) for N in Ns]
    ws = [w4.repack(w, s, N, K) if packed else w for (w, s), N in zip(pairs, Ns)]
    ss = None if packed else [s for _, s in pairs]
    names = launched_kernels(lambda: w4.gemv_multi(ws, ss, x, Ns, K, M, ys=ys, prepacked=packed))
    assert len(names) == 1 and kernel in names[0], names


@pytest.mark.parametrize("packed,N,K,M,kernel", [
    # the chunks' workgroups fit one round
    (False, 1024, 1152, 109, "split_piece_pair"), (False, 306, 2304, 359, "w4a16_swiglu"),
    (True, 434, 2816, 221, "w4a16_swiglu"),
    # the second chunk has at most 16 rows
    (False, 3672, 768, 35, "split_piece_pair"), (False, 3784, 640, 48, "split_piece_pair"),
    (False, 3672, 768, 49, "gemm_unit_swiglu"), (True, 3672, 768, 35, "gemm_unit_swiglu"),
    (False, 4097, 768, 35, "gemm_unit_swiglu"), (False, 3672, 896, 35, "gemm_unit_swiglu"),
    # they take two
    (True, 1112, 2560, 102, "gemm_unit_swiglu"), (False, 1024, 1152, 130, "gemm_unit_swiglu"),
    (True, 3584, 1024, 64, "gemm_unit_swiglu"), (True, 3584, 1024, 1000, "gemm_wide")])
def test_swiglu_kernel(w4, dev, packed, N, K, M, kernel):
    (gw, gs), (uw, us) = _weights(dev, N, K), _weights(dev, N, K)
    if packed:
        gw, uw, gs, us = w4.repack(gw, gs, N, K), w4.repack(uw, us, N, K), None, None
    x, y = _x(dev, M, K), torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    names = launched_kernels(lambda: w4.swiglu(gw, gs, uw, us, x, N, K, M, y=y, prepacked=packed))
    assert len(names) == 1 and kernel in names[0], names


@pytest.mark.parametrize("packed,N,K,M,kernel", [
    # a round of chunks and a few rows more, two rounds of long K
    (True, 4160, 2304, 101, "gemv_stream"), (True, 864, 3840, 362, "gemv_stream"),
    (True, 3072, 4352, 111, "gemv_stream"), (True, 2016, 5632, 108, "gemv_stream"),
    (True, 1280, 7680, 131, "gemv_stream"), (False, 1152, 8640, 158, "gemv_stream"),
    (True, 1024, 3840, 330, "gemv_stream"), (False, 2019, 6848, 113, "gemv_stream"),
    (False, 628, 7568, 252, "gemv_stream"), (True, 8176, 256, 174, "gemv_stream"),
    # a little more of them
    (True, 2048, 3840, 330, "bf16_gemm"), (False, 2019, 6856, 180, "bf16_gemm"),
    (False, 4200, 6848, 113, "bf16_gemm"), (True, 16384, 256, 174, "bf16_gemm"),
    # enough of them, and 64-row tiles
    (True, 2800, 2304, 192, "bf16_gemm"), (True, 8192, 5632, 108, "bf16_gemm"),
    (False, 8192, 3072, 64, "bf16_gemm"), (True, 8704, 2304, 64, "bf16_gemm"),
    (False, 248320, 1024, 64, "bf16_gemm")])
def test_bf16_head_kernel(w4, dev, packed, N, K, M, kernel):
    w = torch.zeros(N, K, dtype=torch.bfloat16, device=dev)
    x, y = _x(dev, M, K), torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    if packed:
        p = w4.bf16_repack(w, N, K)
        names = launched_kernels(lambda: w4.bf16_gemv_prepacked(p, x, N, K, M, y=y))
    else:
        names = launched_kernels(lambda: w4.bf16_gemv_any(w, x, N, K, M, y=y))
    assert len(names) == 1 and kernel in names[0], names
