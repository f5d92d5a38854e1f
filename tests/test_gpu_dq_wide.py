"""The direct-to-LDS dequantising GEMMs (fake-rule linears and experts) at the edges of their tiles and of
the dispatch, against float64 on the fake-quantized tensors."""
import pytest
import torch

from mindpipe_amd import ops

pytestmark = pytest.mark.gpu

DTYPES = [torch.float16, torch.bfloat16]
# one rounding to the output dtype (half an ulp: 2^-11 / 2^-9 of a value at most, so of the norm too) and fp32
# sums of exact products (K 2^-24 of the sum of magnitudes, a few 1e-5 of the result at these K)
TOL = {torch.float16: 2.0 ** -11 + 5e-5, torch.bfloat16: 2.0 ** -9 + 5e-5}


def _fake(t):
    s = t.abs().amax(-1, keepdim=True).clamp(min=1e-5) / 127
    return (t / s).round() * s


def _weight(shape, dtype, gen):
    q = torch.randint(-127, 128, shape, generator=gen, device="cuda", dtype=torch.int8)
    s = (torch.rand(shape[:-1], generator=gen, device="cuda") * 1e-3 + 5e-4).to(dtype).float()
    return q, s, (q.float() * s.unsqueeze(-1)).to(dtype).double()


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [
    (1, 40, 512), (16, 4097, 640), (17, 8200, 896), (32, 16500, 512),           # a few rows: column tiles, tails, K ranges
    (32, 264, 448), (33, 264, 512), (64, 136, 64), (65, 130, 576),              # the tiled kernel: odd steps, ragged N
    (160, 520, 1024), (161, 392, 320), (192, 136, 256), (224, 264, 128),        # stages by row tiles
    (256, 25000, 192), (257, 12300, 128), (1000, 50000, 64),                    # ragged N, several row slots
    (289, 24842, 448), (1089, 10250, 640),                                      # 256 columns per workgroup, part of a slot
])
def test_linear_edges(dtype, m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m * 7 + n + k)
    q, s, w = _weight((n, k), dtype, gen)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    b = torch.randn(n, generator=gen, device="cuda").to(dtype)
    ref = _fake(x).double() @ w.T
    y = ops.w8a8_linear_fake(x, q, s, None)
    assert y.shape == (m, n) and _rel(y, ref) <= TOL[dtype]
    assert _rel(ops.w8a8_linear_fake(x, q, s, b), ref + b.double()) <= TOL[dtype]
    assert _rel(ops.dq_linear(x, None, q, s, b, dtype), x.double() @ w.T + b.double()) <= TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [8, 24, 2056, 16384, 16392, 40000, 100])
def test_values_equal_codes_times_scale(dtype, k):
    """K of every row-register count, past them, and not a multiple of 8; zero, constant and +-128 rows."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    x = torch.randn(6, k, generator=gen, device="cuda").to(dtype)
    x[1] = 0
    x[2] = 0.37
    x[3, 0], x[4, k - 1] = 9.0, -9.0
    eye_q = torch.eye(k, device="cuda", dtype=torch.int8) if k <= 2056 else None
    q, s = ops.quant_per_token_i8(x, True)
    if eye_q is not None:  # a unit weight returns the activations' values
        y = ops.w8a8_linear_fake(x, eye_q, torch.ones(k, device="cuda"), None)
        assert torch.equal(y, (q.float() * s.float().unsqueeze(-1)).to(dtype))
    else:
        w = torch.randint(-127, 128, (64, k), generator=gen, device="cuda", dtype=torch.int8)
        sw = torch.full((64,), 2.0 ** -10, device="cuda")
        ref = (q.float() * s.float().unsqueeze(-1)).to(dtype).double() @ (w.double() * 2.0 ** -10).T
        y = ops.w8a8_linear_fake(x, w, sw, None)
        assert float((y.double() - ref).norm()) <= TOL[dtype] * float(ref.norm())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(17, 8200, 896), (64, 136, 64), (257, 12300, 128), (6, 64, 16392), (5, 64, 100)])
def test_rows_of_infinities_and_nan(dtype, m, n, k):
    """A row with an infinity (its scale is infinite) or NaN: what the separate quantization gives; the others as without it."""
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    w, sw, wd = _weight((n, k), dtype, gen)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    clean = ops.w8a8_linear_fake(x, w, sw, None)
    x[1, k - 1], x[m - 1, 3], x[3, 0] = float("inf"), float("nan"), float("-inf")
    y = ops.w8a8_linear_fake(x, w, sw, None)
    q, s = ops.quant_per_token_i8(x, True)
    values = (q.float() * s.float().unsqueeze(-1)).to(dtype)
    good = torch.ones(m, dtype=torch.bool, device="cuda")
    good[[1, 3, m - 1]] = False
    assert torch.equal(y[good], clean[good])
    for r in (1, 3, m - 1):
        assert bool(torch.isfinite(y[r]).any()) == bool(torch.isfinite(values[r]).all())
    ref = values[[1, 3, m - 1]].double() @ wd.T
    assert torch.equal(torch.isnan(y[[1, 3, m - 1]]), torch.isnan(ref))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("t,e,top,h,inter", [(1, 4, 1, 64, 64), (37, 8, 2, 192, 320), (300, 4, 2, 128, 576),
                                             (700, 2, 1, 256, 192), (64, 32, 4, 512, 128)])
def test_experts_equal_the_separate_steps(dtype, t, e, top, h, inter):
    """The one-call chain against the four entry points on codes, with an expert no token takes and ids
    outside [0, E): the values between the steps are the same, the sums in another order."""
    gen = torch.Generator(device="cuda").manual_seed(t + e)
    w13, s13, _ = _weight((e, 2 * inter, h), dtype, gen)
    w2, s2, _ = _weight((e, h, inter), dtype, gen)
    x = torch.randn(t, h, generator=gen, device="cuda").to(dtype)
    ids = torch.stack([torch.randperm(e, generator=gen, device="cuda")[:top] for _ in range(t)]).to(torch.int32)
    if e > 2:
        ids[ids == e - 1] = -1
    tw = torch.rand(t, top, generator=gen, device="cuda")
    y = ops.moe_w8a8_forward(x, ids, tw, w13, s13, w2, s2, None, "fake")
    routed, rs, slots, off = ops.moe_permute_quant(x, ids, e, "fake")
    q, s = ops.moe_gmm1_swiglu_quant(routed, rs, w13, s13, off, inter, "fake", dtype)
    ref = ops.moe_unpermute_combine(ops.moe_gmm2(q, s, w2, s2, off, torch.float32, "fake", dtype), slots, tw, dtype, "fake")
    # a sum that lands on the other side of a rounding moves h by an ulp and may flip its code (1 of 127)
    assert _rel(y, ref.double()) <= (2e-3 if dtype == torch.float16 else 8e-3)


@pytest.mark.parametrize("t,e,top,inter,one_call", [(1024, 2, 1, 512, False), (384, 2, 1, 512, False), (382, 2, 1, 512, True),
                                                    (2048, 8, 2, 512, False), (64, 4, 2, 512, True), (1024, 4, 1, 2176, True)])
def test_experts_route(monkeypatch, t, e, top, inter, one_call):
    """Few gate / up workgroups on full chunks of rows: the four entry points; else the one call.  The same values."""
    gen = torch.Generator(device="cuda").manual_seed(t + e)
    w13, s13, _ = _weight((e, 2 * inter, 256), torch.float16, gen)
    w2, s2, _ = _weight((e, 256, inter), torch.float16, gen)
    x = torch.randn(t, 256, generator=gen, device="cuda").half()
    ids = torch.stack([torch.randperm(e, generator=gen, device="cuda")[:top] for _ in range(t)]).to(torch.int32)
    tw = torch.rand(t, top, generator=gen, device="cuda")
    calls, inner = [], ops._moe_fake
    monkeypatch.setattr(ops, "_moe_fake", lambda *a: calls.append(1) or inner(*a))
    y = ops.moe_w8a8_forward(x, ids, tw, w13, s13, w2, s2, None, "fake")
    assert bool(calls) == one_call
    monkeypatch.setattr(ops, "_moe_fake_takes", lambda *a: not one_call)
    assert _rel(ops.moe_w8a8_forward(x, ids, tw, w13, s13, w2, s2, None, "fake"), y.double()) <= 2e-3


def test_linear_op_traces():
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, s, _ = _weight((72, 128), torch.bfloat16, gen)
    x = torch.randn(2, 3, 128, generator=gen, device="cuda").bfloat16()
    torch.library.opcheck(torch.ops.mindpipe_amd_fake.w8a8_linear_fake.default, (x, q, s, None))
    fn = torch.compile(lambda v: ops.w8a8_linear_fake(v, q, s, None), fullgraph=True, backend="aot_eager")
    assert torch.equal(fn(x), ops.w8a8_linear_fake(x, q, s, None))
