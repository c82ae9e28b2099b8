"""Operands at addresses that are aligned to their element only: the same results,
bit for bit, as aligned ones give (the sums are integers, or taken in the same
order on the same kernel), and nothing written outside the result.
"""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C
    from cider_amd import _lib

DEV = "cuda"


def off_by_one(t):
    """t's values one element past an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 == t.element_size()
    return out


def bits(t):
    return t.view(torch.int16)


# int4 kernels that take x in an order of their own, the scalar quantization
# writing it: the ping-pong kernel (with an odd number of row blocks), the one-set
# per-group kernel, its split-K slices; and kernels that take it in order
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("fmt,M,N,K", [
    ("w4", 1334, 6152, 640), ("w4", 257, 12288, 512), ("w4", 100, 520, 640), ("w4", 5, 264, 512),
    ("w4g64", 700, 6144, 1024), ("w4g128", 2051, 2568, 512), ("w4g128", 512, 4096, 12288),
    ("w4g64", 130, 520, 1024), ("w4g128", 7, 264, 512),
    ("pc", 300, 520, 640), ("pc", 3, 264, 512), ("pc", 33, 100, 72)])
def test_x(fmt, M, N, K, dtype):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV, generator=g).to(getattr(torch, dtype))
    x[0, 1::2] *= 50.0  # the two halves of a block differ
    if fmt == "pc":
        w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
        s = torch.rand(N, device=DEV, generator=g) * 1e-2 + 1e-4
        layer = C.CiderLinear(w, s, 0, K, N)
    elif fmt == "w4":
        w = torch.randint(0, 256, (K // 2, N), device=DEV, generator=g).to(torch.uint8)
        layer = C.W4A8Linear(w, torch.rand(N, device=DEV, generator=g) * 0.1 + 1e-3, K)
    else:
        gs = int(fmt[3:])
        w = torch.randint(0, 256, (N, K // 2), device=DEV, generator=g).to(torch.uint8)
        s = (torch.rand(K // gs, N, device=DEV, generator=g) * 0.1 + 1e-3).half()
        layer = C.W4A8GroupLinear(w, s, gs)
    assert torch.equal(bits(layer(off_by_one(x))), bits(layer(x)))


def guarded(shape, dtype):
    """An empty result one element past an aligned address, and its buffer."""
    n = shape[0] * shape[1]
    buf = torch.full((n + 33,), 77, dtype=dtype, device=DEV)
    return buf[1:1 + n].view(shape), buf


def untouched(buf, n):
    return bool((buf[:1] == 77).all() and (buf[1 + n:] == 77).all())


# y and the weight scales at element alignment, N and K whole: GEMV, few rows,
# 64 x 64 LDS-DMA tiles, larger ones, a split-K shape, a shape of the ping-pong kernel
SHAPES = [(2, 512, 1024), (16, 4096, 512), (40, 512, 1024), (56, 1024, 512), (96, 2048, 512),
          (300, 4096, 512), (128, 512, 8192), (1000, 6144, 512), (2500, 10248, 128)]


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_y_and_scales(M, N, K, bias):
    g = torch.Generator(device=DEV).manual_seed(M)
    lib = _lib.load()
    x = torch.randn(M, K, device=DEV, generator=g).half()
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
    sw = torch.rand(N, device=DEV, generator=g) * 1e-2 + 1e-4
    b = torch.randn(N, device=DEV, generator=g).half() if bias else None
    q, sa = C.quantize_per_token(x)
    nb = lib.cider_workspace_bytes(_lib.CIDER_OP_PERCHANNEL, M, N, K, 0)
    ws = torch.empty(max(nb, 1), dtype=torch.uint8, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    expected = C.perchannel_gemm(q, sa, w, sw, b)

    def run(linear, scales, bias_):
        y, buf = guarded((M, N), torch.float16)
        bp = bias_.data_ptr() if bias else None
        if linear:
            rc = lib.cider_perchannel_linear(x.data_ptr(), w.data_ptr(), scales.data_ptr(), bp,
                                             y.data_ptr(), ws.data_ptr(), nb, M, N, K, st)
        else:
            rc = lib.cider_perchannel_gemm(q.data_ptr(), sa.data_ptr(), w.data_ptr(),
                                           scales.data_ptr(), bp, y.data_ptr(), M, N, K, st)
        assert rc == 0
        assert torch.equal(bits(y.clone()), bits(expected)) and untouched(buf, M * N)

    for linear in (False, True):
        for scales in (sw, off_by_one(sw)):
            run(linear, scales, b)
        if bias:
            run(linear, sw, off_by_one(b))


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int32_y(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M)
    a, b = (torch.randint(-128, 128, (n, K), dtype=torch.int8, device=DEV, generator=g)
            for n in (M, N))
    y, buf = guarded((M, N), torch.int32)
    rc = _lib.load().cider_int8_matmul_int32(a.data_ptr(), b.data_ptr(), y.data_ptr(), M, N, K,
                                             torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(y.double(), a.double() @ b.double().t().contiguous())
    assert untouched(buf, M * N)
