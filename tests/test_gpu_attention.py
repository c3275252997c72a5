"""lq_attention against softmax attention evaluated in fp32 on the same 16-bit operands."""
import ctypes as C

import pytest
import torch

# (batch, queries, keys, heads, head_dim): one key, tiles of 64 keys less / exactly / more than full, 32-query wavefronts and the
# blocks of 128 and 256 queries at their edges; with 24 heads 1408 queries are 264 blocks of 128, more than there are compute
# units, which takes the form with two wavefront groups (head_dim 128), 1280 are 240
SHAPES = [(1, 1, 1, 1, 128), (2, 33, 63, 3, 128), (1, 127, 64, 2, 64), (2, 128, 65, 3, 64), (1, 129, 77, 5, 64), (1, 257, 129, 2, 128),
          (3, 96, 300, 4, 64), (1, 1280, 191, 24, 128), (1, 1408, 1, 24, 128), (1, 1409, 64, 24, 128), (1, 1471, 65, 24, 128),
          (1, 1408, 128, 24, 128), (1, 1535, 260, 24, 128), (2, 1025, 1025, 16, 128)]


def _reference(q, k, v, scale):
    """(O, softmax(S) |V|) in fp32, head by head."""
    o = torch.empty(q.shape, dtype=torch.float32, device=q.device)
    mag = torch.empty_like(o)
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            p = ((q[b, :, h].float() @ k[b, :, h].float().t().contiguous()) * scale).softmax(-1)
            vf = v[b, :, h].float().contiguous()
            o[b, :, h], mag[b, :, h] = p @ vf, p @ vf.abs()
    return o, mag


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_attention_matches_fp32(dev, shape, dt):
    from lyradiff_amd import ops

    b, sq, sk, h, dh = shape
    g = torch.Generator(device=dev).manual_seed(sq * 1000 + sk)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    if sq == sk:  # parts of one fused tensor
        q, k, v = (1.5 * rnd(b, sq, 3, h, dh)).to(dt).unbind(2)
    else:
        q, (k, v) = (1.5 * rnd(b, sq, h, dh)).to(dt), (1.5 * rnd(b, sk, 2, h, dh)).to(dt).unbind(2)
    got = ops.attention(q, k, v)
    assert got.shape == q.shape and got.is_contiguous()
    want, mag = _reference(q, k, v, dh ** -0.5)
    # u: rounding error of T.  Probabilities rounded to T, summed in fp32, the result rounded to T: 2 u of the sum of |terms|, 3 with room.
    # Absolute part: scores in fp32 over dh products of size ~ 1.5^2 and the exponentials, a few 1e-6; fp16 probabilities under
    # 2^-14 are rounded to a fixed step, 2^-25 for each of at most 1025 keys times |v| ~ 1.2: 4e-5
    u = 2.0 ** -11 if dt is torch.float16 else 2.0 ** -8
    assert ((got.float() - want).abs() <= 3 * u * mag + 5e-5).all()
    assert torch.equal(got, ops.softmax_attention(q, k, v))


@pytest.mark.gpu
@pytest.mark.parametrize("sq,h,dh", [(40, 2, 64), (40, 2, 128), (1408, 24, 128)])  # the three forms of the kernel
def test_attention_leaves_out_keys_of_minus_infinity(dev, sq, h, dh):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(dh + sq)
    q, k, v = (torch.rand(1, n, h, dh, generator=g, device=dev).bfloat16() for n in (sq, 200, 200))
    k[:, :70] = -float("inf")  # the first tile of 64 keys and a part of the second: their scores are -inf for these positive queries
    q.clamp_(min=0.01)
    got = ops.attention(q, k, v)
    assert torch.isfinite(got).all()
    assert torch.allclose(got.float(), ops.attention(q, k[:, 70:].contiguous(), v[:, 70:].contiguous()).float(), rtol=2.0 ** -6, atol=0)
    k[:] = -float("inf")
    assert torch.isnan(ops.attention(q, k, v)).all()  # as softmax of a row of -inf


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-30, 0.5, 0.7, 1.0, 30.0])  # 0.693 * log2(e) = 1
@pytest.mark.parametrize("sq,h,dh", [(40, 2, 64), (40, 2, 128), (1408, 24, 128)])  # the three forms of the kernel
def test_attention_leaves_out_keys_of_minus_infinity_at_every_scale(dev, sq, h, dh, scale):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(dh + sq)
    q, k, v = (torch.rand(1, n, h, dh, generator=g, device=dev).bfloat16() for n in (sq, 264, 264))
    k[:, :136] = -float("inf")  # two tiles of 64 keys and a part of the third
    q.clamp_(min=0.01)
    got = ops.attention(q, k, v, scale)
    assert torch.isfinite(got).all()
    # the same 128 keys in other tiles: probabilities rounded to bf16 on both sides, positive v
    assert torch.allclose(got.float(), ops.attention(q, k[:, 136:].contiguous(), v[:, 136:].contiguous(), scale).float(), rtol=2.0 ** -6, atol=0)
    k[:] = -float("inf")
    assert torch.isnan(ops.attention(q, k, v, scale)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sk", [64, 200])  # one tile; three and a part
@pytest.mark.parametrize("sq,h,dh", [(300, 2, 64), (300, 2, 128), (1408, 24, 128)])  # the three forms of the kernel
def test_attention_sums_its_probabilities_in_32_bits(dev, sq, h, dh, sk, dt):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(sk + sq)
    q, k, v = (torch.zeros(1, n, h, dh, dtype=dt, device=dev) for n in (sq, sk, sk))
    q[..., 0] = (20 * torch.rand(1, sq, h, generator=g, device=dev)).to(dt)
    k[:, 1:, :, 0] = -1  # scores 0, -x, -x, ..., so that the roundings of the probabilities to T all point the same way
    v[:, 0] = 1
    x = q[..., :1].double() * float(torch.tensor(dh ** -0.5))
    want = (1 / (1 + (sk - 1) * torch.exp(-x))).to(dt).expand_as(q)
    # fp32 scores, exponentials and sums: relative errors of about 2^-21, which move a result over a boundary between two numbers of T
    # (2^-12 apart or more) for less than one row in 500; a sum of rounded probabilities moves every third one
    assert (ops.attention(q, k, v) != want).float().mean() < 0.01


@pytest.mark.gpu
@pytest.mark.parametrize("sk", [13, 63, 77, 250])  # the last of one, two and four tiles; 64 keys fill one
@pytest.mark.parametrize("sq,h,dh", [(40, 2, 64), (40, 2, 128), (1408, 24, 128)])  # the three forms of the kernel
def test_attention_keeps_an_infinite_value_of_the_last_key(dev, sq, h, dh, sk):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(sk + sq)
    q, k, v = (torch.randn(2, n, h, dh, generator=g, device=dev).bfloat16() for n in (sq, sk, sk))
    want = ops.attention(q, k, v)
    v[:, -1, :, 0], v[:, -1, :, dh - 1] = float("inf"), -float("inf")
    got = ops.attention(q, k, v)
    assert (got[..., 0] == float("inf")).all() and (got[..., dh - 1] == -float("inf")).all()
    assert torch.equal(got[..., 1:dh - 1], want[..., 1:dh - 1])


@pytest.mark.gpu
def test_attention_of_other_shapes_falls_back(dev):
    from lyradiff_amd import ops

    for dh, dt in ((40, torch.float16), (64, torch.float32), (160, torch.bfloat16)):
        q, k, v = torch.randn(1, 20, 3, 2, dh, device=dev).to(dt).unbind(2)
        assert not ops.attention_supported(q, k, v)
        want, _ = _reference(q, k, v, dh ** -0.5)
        assert (ops.softmax_attention(q, k, v).float() - want).abs().max() < 2e-2
        with pytest.raises(ValueError):
            ops.attention(q, k, v)


@pytest.mark.gpu
def test_attention_follows_the_strides(dev):
    """What the kernel reads in place (parts of wider tokens, a batch repeated by a stride of 0, heads from a wider tensor's start) and
    what it leaves to PyTorch (strides off 16 bytes, also of a single token, heads apart or interleaved, tokens that overlap)."""
    from lyradiff_amd import ops

    h, dh = 3, 64
    w = h * dh
    buf = torch.randn(8 * 40 * 4 * w, generator=torch.Generator(device=dev).manual_seed(5), device=dev).bfloat16()
    make = lambda b, s, row, batch, off=0, head=dh, elem=1: buf.as_strided((b, s, h, dh), (batch, row, head, elem), off)
    dense = lambda b, s: make(b, s, w, s * w)
    cases = [(dense(2, 9), make(2, 40, 4 * w, 160 * w), make(2, 40, 3 * w + 8, 160 * w, 64), True),
             (make(3, 9, w, 0), make(3, 40, w, 0, 8), make(3, 40, 2 * w, 80 * w), True),
             (make(1, 9, w, 3), make(1, 40, w, 5), make(1, 40, w, 7), True),                 # one batch: its stride is of no account
             (dense(2, 9), make(2, 1, w + 3, 8 * w), make(2, 1, 2 * w, 8 * w), False),       # one key, at an odd stride
             (make(2, 1, w + 3, 8 * w), dense(2, 40), dense(2, 40), False),
             (dense(2, 9), make(2, 40, w + 4, 160 * w), dense(2, 40), False),
             (dense(2, 9), dense(2, 40), make(2, 40, w, 40 * w + 2), False),
             (dense(2, 9), dense(2, 40), make(2, 40, w, 40 * w, 4), False),
             (dense(2, 9), make(2, 40, 2 * w, 80 * w, head=2 * dh), dense(2, 40), False),
             (dense(2, 9), make(2, 40, w, 40 * w, head=1, elem=h), dense(2, 40), False),
             (make(2, 9, 8, 9 * w), dense(2, 40), dense(2, 40), False)]
    for i, (q, k, v, taken) in enumerate(cases):
        assert ops.attention_supported(q, k, v) == taken, i
        got = ops.softmax_attention(q, k, v)
        if taken:
            assert torch.equal(got, ops.attention(q.contiguous(), k.contiguous(), v.contiguous())), i
        else:
            assert (got.float() - _reference(q, k, v, dh ** -0.5)[0]).abs().max() < 2e-2, i  # of values up to 4, rounded to bf16
            with pytest.raises(ValueError):
                ops.attention(q, k, v)


@pytest.mark.gpu
@pytest.mark.parametrize("sq,h,dh", [(300, 2, 64), (300, 2, 128), (1408, 24, 128)])  # the three forms of the kernel
def test_attention_on_a_side_stream_and_replayed_from_a_graph(dev, sq, h, dh):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(sq)
    qkv = torch.randn(1, sq, 3, h, dh, generator=g, device=dev).bfloat16()
    static = qkv.clone()
    run = lambda t: ops.softmax_attention(*t.unbind(2))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    want = run(qkv)
    with torch.cuda.stream(side):
        got = run(static)
    side.synchronize()
    assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = run(static)
    for i in range(4):
        new = (qkv * (1.0 + 0.25 * i)).bfloat16()
        want = run(new)
        static.copy_(new)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
        run(qkv)  # eager work between the replays
        torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,sq,h,dh", [(2, 77, 3, 64), (2, 300, 2, 128), (1, 1443, 24, 128)])  # the three forms of the kernel, ragged
def test_attention_codes_are_the_casts_of_its_output(dev, b, sq, h, dh, dt):
    """e4m3 k-panels of both parts and int8 codes: bit for bit the separate quantisers', NaN, saturation and untouched neighbours included."""
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(sq + dh)
    qkv = torch.randn(b, sq, 3, h, dh, generator=g, device=dev).to(dt)
    qkv[0, 5, 2, 0, 7] = float("inf")  # a value: its column saturates
    qkv[-1, 3, 0, h - 1] = float("nan")  # a query: its row is NaN
    q, k, v = qkv.unbind(2)
    o = ops.attention(q, k, v)
    assert o[0, :, 0, 7].isinf().any() and o[-1, 3, h - 1].isnan().all()
    sa, sb = torch.full((1,), 1e-3, device=dev), torch.full((1,), 3e-4, device=dev)
    rows = lambda t: t.reshape(-1, h * dh).contiguous()
    assert torch.equal(ops.attention_codes(q, k, v, fp8_scale=sa), ops.fp8_scale_cast_panels(rows(o), sa))
    for context in (0, 1, 33, sq):
        got, ctx = ops.attention_codes(q, k, v, None, context, sa, sb)
        assert torch.equal(ctx, ops.fp8_scale_cast_panels(rows(o[:, :context]), sb)), context
        assert torch.equal(got, ops.fp8_scale_cast_panels(rows(o[:, context:]), sa)), context
    wide = torch.full((h * dh // 64 + 2, b * sq, 64), 0xAB, dtype=torch.uint8, device=dev)
    ops.attention_codes(q, k, v, fp8_scale=sa, fp8_out=wide[1:-1])
    assert torch.equal(wide[1:-1], ops.fp8_scale_cast_panels(rows(o), sa)) and (wide[0] == 0xAB).all() and (wide[-1] == 0xAB).all()
    pre = 0.5 + torch.rand(h * dh, generator=g, device=dev)
    for scale in (sa, torch.full((1,), 2.0 ** -120, device=dev)):
        assert torch.equal(ops.attention_codes(q, k, v, int8_scale=scale, int8_pre=pre), ops.sq_quant(o.reshape(b, sq, h * dh), pre, scale))
    assert torch.equal(ops.attention_codes(q, k, v, int8_scale=sa), ops.sq_quant(o.reshape(b, sq, h * dh), None, sa))
    with pytest.raises(ValueError):
        ops.attention_codes(q, k, v, None, 1, sa)
    with pytest.raises(ValueError):
        ops.attention_codes(q, k, v)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,s,sc,h,dh", [(1, 97, 0, 24, 128), (1, 40, 33, 3, 64), (2, 21, 21, 5, 128), (2, 9, 4, 1, 64)])
def test_rmsnorm_rope_in_place(dev, b, s, sc, h, dh, dt):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(s + h)
    draw = lambda *shape: torch.randn(*shape, generator=g, device=dev).to(dt)
    qkv, norm, added = draw(b, s, 3 * h * dh), draw(2 * dh), draw(2 * dh)
    for tables in (1, b):
        rope = draw(tables, s, dh // 2, 2, 2)
        want = ops.rmsnorm_rope(qkv[:, sc:].contiguous(), norm, rope, h, qkv[:, :sc].contiguous() if sc else None, added if sc else None)
        got = qkv.clone()
        assert torch.equal(ops.rmsnorm_rope_inplace(got, norm, rope, h, sc, added if sc else None), want)
        assert torch.equal(got.view(b, s, 3, h, dh)[:, :, 2], qkv.view(b, s, 3, h, dh)[:, :, 2])


def test_attention_argument_errors_do_not_reach_the_gpu():
    from lyradiff_amd import lib as L

    lib, one = L.load(), C.c_void_p(16)
    call = lambda **kw: lib.lq_attention(*{**dict(out=one, q=one, qr=384, qb=0, k=one, kr=384, kb=0, v=one, vr=384, vb=0, dt=L.LQ_BF16, b=1, sq=8,
                                                  sk=8, h=3, dh=128, s=1.0, st=None), **kw}.values())
    assert call(dt=L.LQ_F32) == -4
    assert call(dh=96) == -2 and call(sk=0) == -2 and call(kr=376) == -2 and call(sk=1 << 23) == -2
    assert call(s=0.0) == -1 and call(s=-1.0) == -1
    assert call(q=None) == -1 and call(q=C.c_void_p(8)) == -1 and call(qr=388) == -1
    assert call(sq=0) == 0
