"""bf16 activations and results (cider_linear_bf16) against casting around the
fp16 linear, bit for bit, in every kernel that a linear can run: the casts are
the reference's own order (x rounded to fp16, the fp16 result rounded to bf16).
"""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C

DEV = "cuda"


def inputs(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, device=DEV, generator=g) * 3
    x[:, : K // 64] *= 20.0
    if M > 2:  # beyond fp16's range, subnormal there, infinite, NaN, zero rows
        x[0, 0], x[0, 1] = 1e6, -1e-7
        x[1] *= 1e-8
        x[2, 3] = float("nan")
        x[M - 1] = 0
    w = torch.randint(-8, 8, (N, K), dtype=torch.int8, device=DEV, generator=g)
    b = torch.randn(N, device=DEV, generator=g).half()
    return x.bfloat16(), w, b, g


def same(a, e):
    assert a.dtype == e.dtype == torch.bfloat16 and a.shape == e.shape
    assert torch.equal(a.isnan(), e.isnan())
    ok = ~e.isnan()
    assert torch.equal(a.view(torch.int16)[ok], e.view(torch.int16)[ok])


def calls(x, w, b, g):
    (M, K), N = x.shape, w.shape[0]

    def rand(*s):
        return torch.rand(*s, device=DEV, generator=g) * 1e-2 + 1e-3

    u = w.to(torch.uint8) & 15
    w4 = (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()
    sw = rand(N)
    yield "pc", lambda v: C.perchannel_linear(v, w, sw, b)
    yield "w4", lambda v: C.w4a8_linear_packed(v, w4, sw)
    for gs in (64, 128, 256):
        if K % gs:
            continue
        sg = rand(K // gs, N)
        yield "pg%d" % gs, lambda v: C.pergroup_linear(v, w, sg, gs, b)
        if gs < 256:
            yield "w4g%d" % gs, lambda v: C.w4a8_pergroup_linear(v, w4, sg.half(), gs, b)


# every row count a dispatch rule looks at, short and long K, a K that only the
# lane-order MV takes, ragged N and K (the register-staged kernel and the
# scalar quantize), shapes split over K, large grids
@pytest.mark.parametrize("M,N,K", [
    (1, 264, 1024), (1, 2560, 10240), (1, 40, 320), (2, 264, 1024), (4, 512, 4096),
    (4, 64, 640), (16, 264, 2048), (16, 264, 640), (24, 264, 1024), (48, 8200, 512),
    (64, 1032, 512), (137, 2560, 4096), (129, 130, 192), (200, 264, 1024), (300, 4104, 640),
    (1500, 6152, 512), (2048, 8200, 512)])
def test_bf16_equals_casting(M, N, K):
    x, w, b, g = inputs(M, N, K, M + N + K)
    for name, f in calls(x, w, b, g):
        same(f(x), f(x.half()).bfloat16())


def test_views_and_layers():
    """Strided and unaligned x, and the layers' own forward."""
    x, w, b, g = inputs(40, 264, 1024, 9)
    wide = torch.zeros(40, 1032, dtype=torch.bfloat16, device=DEV)
    wide[:, 1:1025] = x
    flat = torch.zeros(40 * 1024 + 1, dtype=torch.bfloat16, device=DEV)
    flat[1:] = x.reshape(-1)
    for name, f in calls(x, w, b, g):
        e = f(x)
        same(f(wide[:, 1:1025]), e)
        same(f(flat[1:].view(40, 1024)), e)
        same(f(x.t().contiguous().t()), e)
    lin = C.CiderLinear(w, torch.rand(264, device=DEV, generator=g), 0, 1024, 264, b)
    same(lin(x.view(5, 8, 1024)), lin(x.half()).bfloat16().view(5, 8, 264))


def test_captured():
    x, w, b, g = inputs(137, 2560, 4096, 3)
    for name, f in calls(x, w, b, g):
        e = f(x).clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = f(x)
        for _ in range(3):
            y.zero_()
            graph.replay()
            same(y, e)
            f(x)  # eager work between replays
