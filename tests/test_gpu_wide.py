"""The 64 x 64 wave-tile GEMM (w4a16_gemm_wide.hip): shapes its dispatch rule
takes on a 256-CU part, its k-slice form among them, at the edges of its tiles. N
not a multiple of 8 (one output per lane in the stores), of 32 or of 256, M one
row past a tile, one group (K = 128), odd and even numbers of groups, K of whole
8-group units and of several with a short last one, file-layout scale rows that
are not 4 B aligned. Outputs must equal, bit for bit, those of calls of at most 16
rows, which the decode kernels serve whatever N and K are (every row of a batched
call equals the single-row call on it), for bf16 and fp16 activations, both weight
layouts, non-finite activations, and for the SwiGLU forms of it and of the unit
GEMM; the bf16 outputs also the forced tile kernel's. Where a case stands for one
kernel, the test checks that the call launches it."""
import numpy as np
import pytest
import torch

from launched_kernels import launched_kernels

pytestmark = pytest.mark.gpu

# the calls of each shape that take the wide kernel: prepacked, file layout, and
# file layout with scale rows off 4 bytes
ALL = ("prepacked", "file", "scales")
SHAPES = [(51201, 128, 33, ALL), (25617, 384, 65, ALL), (3584, 1024, 897, ALL),
          (6152, 640, 513, ALL), (5000, 1152, 700, ALL), (2056, 2176, 1473, ALL),
          # whole units, an even number of groups with a short last unit
          (2056, 2048, 1473, ALL), (1001, 4096, 3300, ALL), (2056, 2304, 1473, ALL),
          # k-slices: four units, a short last one, three units, ragged N and M
          (1024, 3584, 777, ALL), (1001, 2176, 600, ("file", "scales")),
          (2040, 4096, 489, ("prepacked", "scales")), (8100, 2688, 100, ("file", "scales")),
          (8050, 2688, 100, ALL)]


def _launches(dev, kernel, call, label):
    """On a 256-CU part, where the shapes stand: `call` is one launch of `kernel`."""
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        names = launched_kernels(call)
        assert len(names) == 1 and kernel in names[0], (label, names)


def _inputs(dev, N, K, M, dtype, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    w = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=dev, generator=g)
    s = (torch.rand(N, K // 128, device=dev, generator=g) * 0.01 + 0.001).to(torch.float16)
    return w, s, torch.randn(M, K, device=dev, generator=g).to(dtype)


def _bits(t):
    return t.contiguous().view(torch.int16)


def _same(a, b, label):
    # equal bits, except that any NaN equals any other
    diff = (_bits(a) != _bits(b)) & ~(a.isnan() & b.isnan())
    torch.cuda.synchronize()
    assert int(diff.sum()) == 0, (label, int(diff.sum()), a.shape)


def _by_chunks(call, x, N):
    y = torch.empty(x.shape[0], N, dtype=x.dtype, device=x.device)
    for m0 in range(0, x.shape[0], 16):
        xc = x[m0:m0 + 16].contiguous()
        call(xc, xc.shape[0], y[m0:m0 + 16])
    return y


@pytest.mark.parametrize("N,K,M,wide", SHAPES)
@pytest.mark.parametrize("f16", [False, True])
def test_wide_equals_decode_kernels(w4, dev, N, K, M, wide, f16):
    dtype = torch.float16 if f16 else torch.bfloat16
    w, s, x = _inputs(dev, N, K, M, dtype, 0x71DE + N + K + M)
    # scales 2 bytes past a 4-byte boundary
    buf = torch.empty(s.numel() + 1, dtype=torch.float16, device=dev)
    s2 = buf[1:].view_as(s)
    s2.copy_(s)
    assert s2.data_ptr() % 4 == 2
    p = w4.repack(w, s, N, K)
    file_call = w4.gemv_f16 if f16 else w4.gemv
    packed_call = w4.gemv_f16_prepacked if f16 else w4.gemv_prepacked
    for bad in (False, True):
        if bad:
            x[M // 2, K // 3] = float("inf")
            x[M - 1, 1] = float("nan")
            x[0, K - 1] = -float("inf")
        ref = _by_chunks(lambda xc, m, yc: packed_call(p, xc, N, K, m, y=yc), x, N)
        for label, call in (("prepacked", lambda y: packed_call(p, x, N, K, M, y=y)),
                            ("file", lambda y: file_call(w, s, x, N, K, M, y=y)),
                            ("scales", lambda y: file_call(w, s2, x, N, K, M, y=y))):
            y = torch.empty(M, N, dtype=dtype, device=dev)
            call(y)
            _same(y, ref, (label, bad))
            if label in wide and not bad:
                _launches(dev, "gemm_wide", lambda: call(y), label)
        if not f16:
            y = torch.empty(M, N, dtype=dtype, device=dev)
            w4.gemv(w, s, x, N, K, M, y=y, variant="tile32")
            _same(y, ref, ("tile32", bad))
    # an output base off 16 bytes
    yb = torch.empty(M * N + 1, dtype=dtype, device=dev)
    y = yb[1:].view(M, N)
    packed_call(p, x, N, K, M, y=y)
    _same(y, ref, "output base")


@pytest.mark.parametrize("N,K,M,kernel", [
    (3584, 1024, 833, "gemm_wide"), (8200, 384, 190, "gemm_wide"), (16385, 128, 129, "gemm_wide"),
    (2048, 2176, 600, "gemm_wide"), (2048, 2048, 600, "gemm_wide"), (3000, 3584, 700, "gemm_wide"),
    # unit GEMM: 128- and 64-row tiles, two k-slices, more units than the slices
    # keep, ragged N
    (3584, 1024, 100, "gemm_unit_swiglu"), (8200, 384, 70, "gemm_unit_swiglu"),
    (4201, 512, 40, "gemm_unit_swiglu"), (6001, 640, 33, "gemm_unit_swiglu"),
    (1030, 3584, 97, "gemm_unit_swiglu"), (1024, 2048, 129, "gemm_unit_swiglu"),
    (1029, 9216, 100, "gemm_unit_swiglu"),
    # a few tiles short of it: the chunks
    (3001, 512, 40, "split_piece_pair")])
def test_gemm_swiglu_equals_chunks(w4, dev, N, K, M, kernel):
    gw, gs, x = _inputs(dev, N, K, M, torch.bfloat16, 0x51F + N + M)
    uw, us, _ = _inputs(dev, N, K, 1, torch.bfloat16, 0x520 + K)
    gp, up = w4.repack(gw, gs, N, K), w4.repack(uw, us, N, K)
    for bad in (False, True):
        if bad:
            x[M // 2, K // 3] = float("inf")
            x[M - 1, 1] = float("nan")
        ref = _by_chunks(lambda xc, m, yc: w4.swiglu(gp, None, up, None, xc, N, K, m, y=yc,
                                                     prepacked=True), x, N)
        y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        w4.swiglu(gp, None, up, None, x, N, K, M, y=y, prepacked=True)
        _same(y, ref, ("prepacked", bad))
        y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        w4.swiglu(gw, gs, uw, us, x, N, K, M, y=y)
        _same(y, ref, ("file", bad))
    _launches(dev, kernel, lambda: w4.swiglu(gp, None, up, None, x, N, K, M, y=y, prepacked=True),
              "prepacked")
    _launches(dev, kernel, lambda: w4.swiglu(gw, gs, uw, us, x, N, K, M, y=y), "file")


# the smaller-tiled prefill kernels on fp16 activations: each of the split
# kernel's widths (2, 8 and 4 waves a set), the 32 x 32 kernel and the unit GEMM's
# forms (at 6144 x 1024 the file layout takes the wide kernel)
@pytest.mark.parametrize("N,K,M,kernel", [
    (4096, 1024, 33, "split_kernelINS_6ActF16ELi2"), (3584, 1024, 512, "split_kernelINS_6ActF16ELi8"),
    (6144, 1024, 512, "split_kernelINS_6ActF16ELi4"), (3584, 512, 512, "gemm32_kernel"),
    (512, 1024, 128, "gemm_unit"), (1000, 640, 70, "gemm_unit"), (37, 3584, 65, "gemm_unit"),
    (3584, 640, 200, "gemm_unit_kernelINS_6ActF16ELi1ELi2ELi8")])
def test_f16_prefill_equals_decode_kernels(w4, dev, N, K, M, kernel):
    w, s, x = _inputs(dev, N, K, M, torch.float16, 0xF16 + N + K + M)
    p = w4.repack(w, s, N, K)
    x[M // 2, 3] = float("inf")
    ref = _by_chunks(lambda xc, m, yc: w4.gemv_f16_prepacked(p, xc, N, K, m, y=yc), x, N)
    y = torch.empty(M, N, dtype=torch.float16, device=dev)
    w4.gemv_f16_prepacked(p, x, N, K, M, y=y)
    _same(y, ref, "prepacked")
    _launches(dev, kernel, lambda: w4.gemv_f16_prepacked(p, x, N, K, M, y=y), "prepacked")
    y = torch.empty(M, N, dtype=torch.float16, device=dev)
    w4.gemv_f16(w, s, x, N, K, M, y=y)
    _same(y, ref, "file")


@pytest.mark.parametrize("Ns,K,M,kernel", [
    ((6144, 2048, 16, 16), 1024, 33, "gemm_unit"), ((4096, 512, 512), 1024, 300, "gemm_unit"),
    ((3584, 3584), 1024, 577, "gemm_wide"), ((1001, 37, 130), 640, 65, "gemm_unit"),
    ((512,) * 8, 2176, 70, "gemm_unit"), ((1000, 16, 2049), 4096, 129, "gemm_unit"),
    ((1, 5000, 129, 3000), 128, 700, "gemm_wide"), ((3000, 17), 9216, 40, "gemm_unit"),
    ((2056, 16, 2000), 2176, 1473, "gemm_wide"), ((2056, 16, 2000), 2048, 1473, "gemm_wide"),
    ((2056, 16, 2000), 2304, 1473, "gemm_wide")])
def test_prefill_group_equals_single_calls(w4, dev, Ns, K, M, kernel):
    # one launch over all projections' tiles: the unit GEMM's forms (two
    # k-slices, more units than they keep) and the wide kernel's
    ws, ss = [], []
    for j, N in enumerate(Ns):
        w, s, _ = _inputs(dev, N, K, 1, torch.bfloat16, 0x6E0 + j + K)
        ws.append(w)
        ss.append(s)
    x = _inputs(dev, 1, K, M, torch.bfloat16, 0x6F0 + M)[2]
    x[M // 2, 7] = float("inf")
    packed = [w4.repack(w, s, N, K) for w, s, N in zip(ws, ss, Ns)]
    refs = [w4.gemv_prepacked(p, x, N, K, M, y=torch.empty(M, N, dtype=torch.bfloat16, device=dev))
            for p, N in zip(packed, Ns)]
    buf = torch.empty(ss[0].numel() + 1, dtype=torch.float16, device=dev)
    s2 = buf[1:].view_as(ss[0])  # one projection's scales off 4 bytes
    s2.copy_(ss[0])
    for label, got in (("prepacked", w4.gemv_multi(packed, None, x, Ns, K, M, prepacked=True)),
                       ("file", w4.gemv_multi(ws, ss, x, Ns, K, M)),
                       ("scales", w4.gemv_multi(ws, [s2] + ss[1:], x, Ns, K, M))):
        for y, ref in zip(got, refs):
            _same(y, ref, (label, ref.shape))
    ys = [torch.empty_like(ref) for ref in refs]
    _launches(dev, kernel,
              lambda: w4.gemv_multi(packed, None, x, Ns, K, M, ys=ys, prepacked=True), "prepacked")
    _launches(dev, kernel, lambda: w4.gemv_multi(ws, ss, x, Ns, K, M, ys=ys), "file")


@pytest.mark.parametrize("N,K,M", [(6144, 2432, 17), (4113, 2304, 32), (2048, 2432, 32),
                                   (5001, 3584, 25), (60001, 4096, 31), (1000, 9216, 32),
                                   (4096, 3584, 32)])
def test_long_k_batches_equal_sixteen_row_calls(w4, dev, N, K, M):
    # 17 to 32 rows whose x fills the LDS or does not fit it: the prefill
    # kernels, against calls of at most 16 rows
    for dtype, packed_call, file_call in ((torch.bfloat16, w4.gemv_prepacked, w4.gemv),
                                          (torch.float16, w4.gemv_f16_prepacked, w4.gemv_f16)):
        w, s, x = _inputs(dev, N, K, M, dtype, 0x10F + N + K + M)
        p = w4.repack(w, s, N, K)
        x[M - 1, 5] = float("nan")
        ref = torch.empty(M, N, dtype=dtype, device=dev)
        for m0 in range(0, M, 16):
            xc = x[m0:m0 + 16].contiguous()
            packed_call(p, xc, N, K, xc.shape[0], y=ref[m0:m0 + 16])
        y = torch.empty_like(ref)
        packed_call(p, x, N, K, M, y=y)
        _same(y, ref, "prepacked")
        y = torch.empty_like(ref)
        file_call(w, s, x, N, K, M, y=y)
        _same(y, ref, "file")
        if dtype == torch.bfloat16:
            for ns in (1, 2):
                for y in w4.gemv_multi([p] * ns, None, x, [N] * ns, K, M, prepacked=True):
                    _same(y, ref, ("group", ns))
