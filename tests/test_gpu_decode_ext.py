"""The decode step's longer fusions against the launches they replace, bit for
bit: cider_gate_up_mv against the (RMSNorm and) gate + up MV and SwiGLU, and
RMSNorm inside an MV of two rows per wave against the two launches.
"""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C
    from cider_amd import fused as F

DEV = "cuda"


def linear(N, K, g, bias):
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
    s = torch.rand(N, device=DEV, generator=g) * 2e-3 + 1e-4
    b = torch.randn(N, device=DEV, generator=g).half() if bias else None
    return C.CiderLinear(w, s, 0, K, N, b)


def bits(t):
    return t.view(torch.int16)


# every K of the table; I of one output, a ragged wave and workgroup, and both
# row counts of K = 4096 (the wider one from 24 outputs per compute unit on)
@pytest.mark.parametrize("mode", ["plain", "norm", "addnorm"])
@pytest.mark.parametrize("I,K", [(1, 1024), (7, 1024), (1037, 2048), (6144, 2048), (9, 3072),
                                 (6143, 4096), (6145, 4096), (12288, 4096), (33, 5120),
                                 (10, 6144), (11, 7168), (500, 8192)])
def test_gate_up_mv(I, K, mode):
    g = torch.Generator(device=DEV).manual_seed(I + K)
    lin = linear(2 * I, K, g, bias=mode != "norm")
    x = torch.randn(1, K, device=DEV, generator=g).half()
    add = torch.randn(1, K, device=DEV, generator=g).half() if mode == "addnorm" else None
    nw = None if mode == "plain" else torch.rand(K, device=DEV, generator=g).half() + 0.5
    h, y = F.gate_up_mv(x, lin, nw, 1e-6, add)
    if nw is None:
        h2, gu = x, lin(x)
    else:
        r = F.rmsnorm_quantize(x, nw, 1e-6, add=add, want_q=False)
        h2, gu = r.h, lin(r.y)
    y2, _, _ = F.silu_mul_quantize(gu, want_q=False) if I % 8 == 0 else (None, None, None)
    if y2 is None:  # the SwiGLU kernel takes multiples of 8
        pad = (-I) % 8
        two = torch.nn.functional.pad(gu.view(2, I), (0, pad)).reshape(1, -1).contiguous()
        y2 = F.silu_mul_quantize(two, want_q=False)[0][:, :I]
    assert torch.equal(bits(h), bits(h2))
    assert torch.equal(bits(y), bits(y2.contiguous()))


def test_gate_up_mv_not_taken():
    g = torch.Generator(device=DEV).manual_seed(1)
    lin = linear(64, 1280, g, False)
    assert F.gate_up_mv(torch.zeros(1, 1280, dtype=torch.float16, device=DEV), lin) is None
    lin = linear(64, 1024, g, False)
    off = torch.zeros(1025, dtype=torch.float16, device=DEV)[1:].view(1, 1024)
    assert F.gate_up_mv(off, lin) is None


@pytest.mark.parametrize("N", [6136, 6144, 6149, 8192])
def test_rmsnorm_mv_rows_per_wave(N):
    g = torch.Generator(device=DEV).manual_seed(N)
    lin = linear(N, 4096, g, True)
    x = torch.randn(1, 4096, device=DEV, generator=g).half()
    nw = torch.rand(4096, device=DEV, generator=g).half() + 0.5
    _, y = F.rmsnorm_mv(x, nw, 1e-6, lin)
    y2 = lin(F.rmsnorm_quantize(x, nw, 1e-6, want_q=False).y)
    assert torch.equal(bits(y), bits(y2))


# every K with two rows per wave, from the N where they begin (24 per compute unit)
@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("K", [3072, 5120, 6144, 7168, 8192])
@pytest.mark.parametrize("N", [6143, 6144, 6149])
def test_rmsnorm_mv_two_rows(N, K, add):
    g = torch.Generator(device=DEV).manual_seed(N + K)
    lin = linear(N, K, g, True)
    x = torch.randn(1, K, device=DEV, generator=g).half()
    a = torch.randn(1, K, device=DEV, generator=g).half() if add else None
    nw = torch.rand(K, device=DEV, generator=g).half() + 0.5
    h, y = F.rmsnorm_mv(x, nw, 1e-6, lin, add=a)
    e = F.rmsnorm_quantize(x, nw, 1e-6, add=a, want_q=False)
    assert torch.equal(bits(h), bits(e.h))
    assert torch.equal(bits(y), bits(lin(e.y)))


# slot at the edges of a 128-row chunk, at the cache's last row, past the valid
# length (written, not attended) and outside the cache; rope_row outside the
# tables; every grouping
@pytest.mark.parametrize("H,KV", [(4, 4), (16, 8), (32, 8), (16, 2)])
@pytest.mark.parametrize("n,slot,row", [(1, 0, 0), (128, 127, 127), (129, 128, 128),
                                        (300, 299, 17), (384, 383, 383), (500, 383, 1),
                                        (100, 200, 5), (300, -1, 3), (300, 384, 3),
                                        (300, 299, 400), (300, 299, -1)])
def test_attn_decode_rope(H, KV, n, slot, row):
    T, P, D = 384, 400, 128
    g = torch.Generator(device=DEV).manual_seed(H * 1000 + n + slot)

    def rand(*s):
        return torch.randn(*s, device=DEV, generator=g).half()

    qkv, qw, kw = rand((H + 2 * KV) * D), rand(D), rand(D)
    cos, sin, kc, vc = rand(P, D), rand(P, D), rand(KV, T, D), rand(KV, T, D)
    i64 = dict(dtype=torch.int64, device=DEV)
    rr, sl, nv = (torch.tensor([v], **i64) for v in (row, slot, n))
    k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    out = F.attn_decode_rope(qkv, qw, kw, 1e-6, cos, sin, rr, sl, k1, v1, nv, 0.09, H, KV)
    q = F.qk_norm_rope(qkv.view(1, -1), qw, kw, 1e-6, cos, sin, rr, sl, k2, v2, H, KV)
    e = F.attn_decode(q, k2, v2, nv, 0.09)
    assert torch.equal(bits(k1), bits(k2)) and torch.equal(bits(v1), bits(v2))
    assert torch.equal(out.isnan(), e.isnan())
    assert torch.equal(bits(out)[~e.isnan()], bits(e)[~e.isnan()])


@pytest.mark.parametrize("sub", ["keys", "queries", "values"])
def test_attn_decode_subnormal(sub):
    # fp16 subnormals are operands as good as any: flushed, every score (or the
    # output) would be 0.  Bound: 128 products summed in fp32 (2^-24 each, scores
    # up to ~8) and one fp16 rounding of the result (2^-11; subnormal: 2^-25).
    T, D, n, H = 256, 128, 200, 4
    g = torch.Generator(device=DEV).manual_seed(3)

    def rand(*s):
        return torch.randn(*s, device=DEV, generator=g)

    tiny = 2.0 ** -17
    q = (rand(H, D) * (tiny if sub == "queries" else 2.0 ** 12)).half()
    k = (rand(1, T, D) * (tiny if sub == "keys" else 2.0 ** 12)).half()
    v = (rand(1, T, D) * (tiny if sub == "values" else 1.0)).half()
    scale = {"values": 2.0 ** -27}.get(sub, 1.0)
    nv = torch.tensor([n], dtype=torch.int64, device=DEV)
    out = F.attn_decode(q, k, v, nv, scale).double().view(H, D).cpu()
    s = q.double().cpu() @ k[0, :n].double().cpu().T * scale
    e = torch.softmax(s, -1) @ v[0, :n].double().cpu()
    bound = 1e-3 * e.abs() + (2.0 ** -24 if sub == "values" else 2.0 ** -13)
    assert ((out - e).abs() <= bound).all()


# The decode attention's partial results of a chunk (its largest score, and P.V
# before the division) against the stated arithmetic, bit for bit: fp32, every
# product and every sum rounded once, ascending order inside and over the slices
# of 8.  The probabilities are read from a first call whose values are one-hot.
# n: one position, a part of a slice, whole slices, a whole chunk.
@pytest.mark.parametrize("H,KV", [(1, 1), (2, 1), (4, 1), (8, 1)])
@pytest.mark.parametrize("n", [1, 5, 100, 104, 128])
def test_attn_decode_rounding(H, KV, n):
    np = pytest.importorskip("numpy")
    D = T = 128
    g = torch.Generator(device=DEV).manual_seed(H + n)
    q = torch.randn(H, D, device=DEV, generator=g).half()
    k = torch.randn(KV, T, D, device=DEV, generator=g).half()
    v = torch.randn(KV, T, D, device=DEV, generator=g).half()
    nv = torch.tensor([n], dtype=torch.int64, device=DEV)
    scale = np.float32(0.0883883461356163)
    G = min(H, 4)

    def partials(values):
        ws = F.attn_decode_workspace(H, T, DEV)
        F.attn_decode(q, k, values, nv, float(scale), ws=ws)
        f = ws.view(torch.float32)[:H * (D + 2)].cpu().numpy().reshape(H // G, G * (D + 2))
        return f[:, :G * D].reshape(H, D), f[:, G * D:G * D + G].reshape(H)

    def summed(terms):  # [..., 128, x]: slices of 8 in order, then their sums in order
        t = terms.reshape(*terms.shape[:-2], 16, 8, terms.shape[-1])
        part = np.zeros(t.shape[:-2] + t.shape[-1:], np.float32)
        for i in range(8):
            part = part + t[..., i, :]
        out = np.zeros(part.shape[:-2] + part.shape[-1:], np.float32)
        for i in range(16):
            out = out + part[..., i, :]
        return out

    qf, kf, vf = (t.float().cpu().numpy() for t in (q, k[0], v[0]))
    scores = summed(qf[:, :, None] * kf.T[None]) * scale  # [H, T]
    p, m = partials(torch.eye(T, device=DEV).half()[None].contiguous())
    assert np.array_equal(m, scores[:, :n].max(1))
    assert (p[:, n:] == 0).all()
    o, _ = partials(v)
    expected = summed(p[:, :, None] * vf[None])  # positions past n: p is 0
    assert np.array_equal(o, expected)
