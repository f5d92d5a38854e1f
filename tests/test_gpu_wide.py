"""The direct-to-LDS W4A16 and int8 GEMMs at the edges of their tiles, of the K split and of the dispatch: the int8 ones
bit for bit against the exact product with the epilogue's operations, the W4A16 ones against float64."""
import pytest
import torch

from mindpipe_amd import ops

pytestmark = pytest.mark.gpu

DTYPES = [torch.float16, torch.bfloat16]
# one rounding of the output (half an ulp of a value at most) and of every weight where the kernel rounds them (the sum of
# K such errors is at most that share of the result's norm), and fp32 sums
TOL = {torch.float16: 2 * 2.0 ** -11 + 5e-5, torch.bfloat16: 2 * 2.0 ** -9 + 5e-5}


def _gen(*key):
    return torch.Generator(device="cuda").manual_seed(sum(k * p for k, p in zip(key, (1, 1009, 9176, 31))))


def _w4(n, k, dtype, gen, zeros=True):
    packed = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    s = (torch.rand(n, k // 128, generator=gen, device="cuda") * 0.004 + 0.004).to(dtype)
    z = torch.randint(0, 16, (n, k // 128), generator=gen, device="cuda").to(dtype) if zeros else None
    u = ((packed.unsqueeze(-1) >> torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)) & 15).flatten(1).double()
    zz = z.double() if zeros else torch.full_like(s, 8).double()
    w = (u - zz.repeat_interleave(128, 1)) * s.double().repeat_interleave(128, 1)
    return packed, s, z, w


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k,zeros", [
    (65, 12290, 256, True), (96, 12288, 512, False), (130, 12300, 768, True),   # no workspace: 96 tiles and up, ragged N
    (289, 24842, 1280, True), (1089, 10250, 1024, False),                        # 256 columns per workgroup, part of a slot
    (257, 6200, 256, True), (600, 8192, 512, True), (1025, 2568, 1024, False),   # several row slots, one of one row
    (77, 13824, 5120, True), (33, 16392, 8192, False), (200, 4100, 8192, True),  # K split: 2, none and 7 ways
    (256, 4096, 4096, True), (1023, 1032, 4352, True), (64, 8200, 9216, True),
    (2300, 1500, 2048, True), (700, 1540, 4096, False), (3100, 2570, 2048, True),  # 12, 13 and 21 column tiles over the XCDs
    (64, 4096, 512, True), (80, 520, 640, True),                                 # the kernels below the rules
    (300, 6144, 256, True), (128, 12290, 1024, False), (1024, 6150, 768, True),    # the batched and the prefill kernel next to them
    (128, 16384, 2048, True), (128, 12290, 2048, True), (768, 24580, 1024, False),
    (48, 11010, 8192, True), (40, 13830, 8192, False),                             # two ways on few CUs, on most
    (16, 65600, 1280, True), (32, 32800, 2304, False), (16, 32776, 256, True),      # the batched kernel's walk from another step
    (33, 32800, 2304, True),                                                       # three row parts: from the first
])
def test_w4_linear(dtype, m, n, k, zeros):
    gen = _gen(m, n, k)
    packed, s, z, w = _w4(n, k, dtype, gen, zeros)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    b = torch.randn(n, generator=gen, device="cuda").to(dtype)
    ref = x.double() @ w.T
    assert _rel(ops.w4a16_gemm(x, packed, s, z, 128, None), ref) <= TOL[dtype]
    assert _rel(ops.w4a16_gemm(x, packed, s, z, 128, b), ref + b.double()) <= TOL[dtype]


@pytest.mark.parametrize("m,n,k", [(96, 12290, 2048), (40, 13830, 8192), (65, 4100, 16384), (200, 4100, 8192), (289, 4096, 4096),
                                   (512, 4096, 4096), (77, 13824, 5120)])
def test_w4_fractional_zero_points(m, n, k):
    """fp16 rows whose numerics round no weight, with zero points of 4 + 2^-8 in some groups: u - z of 9 to 11 lies between
    two fp16 values, and rounded it would move every product of the row the same way.  The bias takes the sum off, so
    that the output shows the fp32 sums: a few roundings per group of their magnitude, and its own."""
    gen = _gen(m, n, k)
    u = torch.randint(12, 16, (n, k), generator=gen, device="cuda", dtype=torch.int32)
    packed = torch.zeros(n, k // 8, device="cuda", dtype=torch.int32)
    for i in range(8):
        packed |= u[:, i::8] << (4 * i)
    s = torch.full((n, k // 128), 2.0 ** -11, device="cuda").half()
    frac = torch.rand(n, k // 128, generator=gen, device="cuda") < 0.5
    frac[: n // 2, ::2] = False
    z = (4.0 + frac * 2.0 ** -8).half()
    x = torch.randint(1, 4, (1, k), generator=gen, device="cuda").half().expand(m, k).contiguous()
    ref = (x[:1].double() @ ((u.double() - z.double().repeat_interleave(128, 1)) * 2.0 ** -11).T)[0]
    b = -ref.half()
    y = ops.w4a16_gemm(x, packed, s, z, 128, b).double()
    err, left = (y - (ref + b.double())).abs(), (ref + b.double()).abs()
    assert bool((err <= 64 * 2.0 ** -24 * ref + 2.0 ** -11 * left).all()), float((err / ref).max())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n2,k", [(65, 12544, 256), (200, 12304, 512), (300, 6208, 768), (513, 8200, 256), (66, 256, 512),
                                    # half of the CUs and more, K from 1024; the kernels before it next to them
                                    (257, 16640, 1024), (65, 33040, 1024), (700, 11000, 2048), (1025, 6660, 1280), (80, 33040, 768),
                                    (512, 16384, 1024), (1536, 14336, 1024)])
def test_w4_swiglu(dtype, m, n2, k):
    """Gate and up in one kernel against the two launches: the same roundings, sums in another order (an output moves by
    a few ulps where gate, up or silu lands on the other side of one)."""
    gen = _gen(m, n2, k)
    packed, s, z, _ = _w4(n2, k, dtype, gen)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    b = torch.randn(n2, generator=gen, device="cuda").to(dtype)
    y = ops.w4a16_gemm_swiglu(x, packed, s, z, 128, b)
    ref = ops.silu_mul(ops.w4a16_gemm(x, packed, s, z, 128, b))
    assert y.shape == (m, n2 // 2) and _rel(y, ref.double()) <= 2 * TOL[dtype]


@pytest.mark.parametrize("out", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [
    (33, 10300, 256), (64, 10240, 128), (65, 24600, 384), (513, 11010, 256),     # 80 / 96 tiles and up, ragged N
    (289, 24842, 384), (1089, 10250, 384),                                        # 256 columns per workgroup, part of a slot
    (1024, 130, 128), (1025, 520, 640), (1300, 4096, 1280),                       # every M from 1024
    (200, 4100, 8192), (40, 4096, 4096), (1000, 1001, 9216), (64, 8192, 28672),   # K split
    (1100, 40, 256), (5000, 260, 256), (3072, 5120, 256), (700, 1540, 8192),      # 1, 3, 20 and 13 column tiles over the XCDs
    (256, 4096, 4096), (100, 520, 1024),                                          # the kernels below the rules
    (48, 4096, 2048), (640, 4096, 8192), (256, 8200, 8192), (256, 16384, 8192),   # no K split: few steps, the mid-M kernel, one slot
    (128, 33000, 128), (256, 16300, 256), (384, 18400, 256),                      # the tiled kernel's two workgroups per CU
    (5632, 260, 1024), (6144, 1026, 128), (8192, 4104, 4224), (8448, 4100, 4224), # the large-M kernel
    (5633, 260, 256), (7936, 4104, 4224),                                         # and next to it
])
def test_int8_linear_bits(out, m, n, k):
    gen = _gen(m, n, k)
    q = torch.randint(-127, 128, (m, k), generator=gen, device="cuda", dtype=torch.int8)
    w = torch.randint(-127, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
    st, sc = torch.rand(m, generator=gen, device="cuda") * 0.01, torch.rand(n, generator=gen, device="cuda") * 0.01
    b = torch.randn(n, generator=gen, device="cuda").to(out)
    acc = (q.double() @ w.double().T).float()
    ref = ((acc * st[:, None]) * sc[None]) + b.float()
    assert torch.equal(ops.w8a8_gemm(q, st, w, sc, b, out), ref.to(out))
    assert torch.equal(ops.w8a8_gemm(q, st, w, sc, None, out), ((acc * st[:, None]) * sc[None]).to(out))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(96, 12290, 512), (300, 6144, 256), (200, 4100, 8192), (1025, 2568, 1024)])
def test_w4_infinite_rows(dtype, m, n, k):
    """Infinities and NaN in some rows stay in them."""
    gen = _gen(m, n, k)
    packed, s, z, _ = _w4(n, k, dtype, gen)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    clean = ops.w4a16_gemm(x, packed, s, z, 128, None)
    bad = torch.tensor([0, 33, m - 1], device="cuda")
    x[0, 5], x[33, k - 1], x[m - 1, k // 2] = float("inf"), float("nan"), float("-inf")
    y = ops.w4a16_gemm(x, packed, s, z, 128, None)
    good = torch.ones(m, dtype=torch.bool, device="cuda")
    good[bad] = False
    assert not bool(torch.isfinite(y[bad]).any()) and bool(torch.isnan(y[33]).all())
    assert torch.equal(y[good], clean[good])


@pytest.mark.parametrize("m,n,k", [(65, 24600, 384), (200, 4100, 8192), (1025, 520, 640)])
def test_int8_infinite_scales(m, n, k):
    """A row's and a column's scale of infinity or NaN: the product's own values, in fp32."""
    gen = _gen(m, n, k)
    q = torch.randint(-127, 128, (m, k), generator=gen, device="cuda", dtype=torch.int8)
    w = torch.randint(-127, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
    q[3] = 0  # 0 x inf
    st, sc = torch.rand(m, generator=gen, device="cuda") * 0.01, torch.rand(n, generator=gen, device="cuda") * 0.01
    st[3], st[m - 1], sc[n - 1], sc[7] = float("inf"), float("nan"), float("inf"), 3e38
    ref = ((q.double() @ w.double().T).float() * st[:, None]) * sc[None]
    for out in (torch.float32, torch.float16):
        assert torch.equal(ops.w8a8_gemm(q, st, w, sc, None, out).float().nan_to_num(1.5, 2e38, -2e38),
                           ref.to(out).float().nan_to_num(1.5, 2e38, -2e38))


def test_weight_and_workspace_that_the_split_cannot_take():
    """A weight off its 16 bytes, a workspace off them, too short or missing: the kernels without the split, the same
    values."""
    from mindpipe_amd import _lib
    lib, (m, n, k) = _lib.load(), (64, 8200, 4096)
    gen = _gen(m, n, k)
    q = torch.randint(-127, 128, (m, k), generator=gen, device="cuda", dtype=torch.int8)
    buf = torch.randint(-127, 128, (n * k + 16,), generator=gen, device="cuda", dtype=torch.int8)
    st, sc = torch.rand(m, generator=gen, device="cuda") * 0.01, torch.rand(n, generator=gen, device="cuda") * 0.01
    for off in (0, 8, 1):
        w = buf[off:off + n * k].view(n, k)
        ref = (((q.double() @ w.double().T).float() * st[:, None]) * sc[None]).half()
        assert torch.equal(ops.w8a8_gemm(q, st, w, sc, None, torch.float16), ref)
    w = buf[:n * k].view(n, k)
    ref = (((q.double() @ w.double().T).float() * st[:, None]) * sc[None]).half()
    packed, s, z, wd = _w4(n, 2 * k, torch.float16, gen)
    x = torch.randn(m, 2 * k, generator=gen, device="cuda").half()
    need8, need4 = lib.mp_w8a8_gemm_workspace_bytes(m, n, k), lib.mp_w4a16_gemm_workspace_bytes(m, n, 2 * k, 128)
    assert need8 and need4
    ws = torch.zeros(max(need8, need4) + 16, dtype=torch.uint8, device="cuda")
    for ptr, less in ((ws.data_ptr() + 4, 0), (ws.data_ptr(), 1), (None, 0)):
        y = torch.empty(m, n, device="cuda").half()
        assert lib.mp_w8a8_gemm_ws(q.data_ptr(), st.data_ptr(), w.data_ptr(), sc.data_ptr(), None, 0, y.data_ptr(),
                                   ops.MP_F16, m, n, k, ptr, need8 - less, ops._stream()) == 0
        assert torch.equal(y, ref)
        y4 = torch.empty(m, n, device="cuda").half()
        assert lib.mp_w4a16_gemm_ws(x.data_ptr(), m, 2 * k, packed.data_ptr(), n, s.data_ptr(), z.data_ptr(), 128, None,
                                    y4.data_ptr(), ops.MP_F16, ptr, need4 - less, ops._stream()) == 0
        assert _rel(y4, x.double() @ wd.T) <= TOL[torch.float16]
    assert not bool(ws.any())  # none of them wrote to it


@pytest.mark.parametrize("fake", [False, True])
@pytest.mark.parametrize("shape", [(1,), (5, 7), (2, 100), (1500,)])
def test_linear_from_activations_equals_the_two_ops(fake, shape):
    gen = _gen(*shape, 7)
    x = torch.randn(*shape, 256, generator=gen, device="cuda").half()
    w = torch.randint(-127, 128, (264, 256), generator=gen, device="cuda", dtype=torch.int8)
    sc, b = torch.rand(264, generator=gen, device="cuda") * 0.01, torch.randn(264, generator=gen, device="cuda").half()
    q, s = ops.quant_per_token_i8(x, fake)
    ref = ops.w8a8_gemm(q, s.float(), w, sc, b, torch.float16)
    assert torch.equal(ops.w8a8_linear(x, w, sc, b, torch.float16, fake), ref)


@pytest.mark.parametrize("t,e,top,h,inter", [(1, 64, 1, 128, 448), (48, 8, 2, 256, 3136), (700, 8, 2, 3200, 1536),
                                             (300, 2, 1, 12416, 12352), (64, 32, 4, 3072, 896),
                                             # more experts than a wave has lanes, empty ones between, several chunks
                                             (100, 65, 1, 256, 128), (40, 200, 2, 128, 192), (1400, 130, 2, 128, 64),
                                             (2000, 257, 1, 256, 64),
                                             # 64 output columns per workgroup: one group, few tiles, several chunks
                                             (1, 1, 1, 128, 64), (33, 1, 1, 256, 192), (257, 1, 1, 384, 1088), (513, 3, 2, 256, 320)])
def test_int8_experts_bits(t, e, top, h, inter):
    """GEMM1 + SwiGLU + requant and GEMM2 over groups of 0 to 350 rows: GEMM2 bit for bit; the codes up to those that
    exp's last bit decides."""
    gen = _gen(t, e, h, inter)
    w13 = torch.randint(-127, 128, (e, 2 * inter, h), generator=gen, device="cuda", dtype=torch.int8)
    s13 = torch.rand(e, 2 * inter, generator=gen, device="cuda") * 1e-3
    w2 = torch.randint(-127, 128, (e, h, inter), generator=gen, device="cuda", dtype=torch.int8)
    s2 = torch.rand(e, h, generator=gen, device="cuda") * 1e-3
    x = torch.randn(t, h, generator=gen, device="cuda").half()
    ids = torch.stack([torch.randperm(e, generator=gen, device="cuda")[:top] for _ in range(t)]).int()
    if e > 64:  # most of the tokens of the first half go to one expert
        ids[:t // 2, 0] = torch.where((ids[:t // 2, 1:] == e - 3).any(-1), ids[:t // 2, 0], e - 3)
    routed, rs, _, off = ops.moe_permute_quant(x, ids, e)
    q, s = ops.moe_gmm1_swiglu_quant(routed, rs, w13, s13, off, inter)
    y = ops.moe_gmm2(q, s, w2, s2, off)
    differ = 0
    ends = off.tolist()
    for i in range(e):
        a, b = ends[i], ends[i + 1]
        if a == b:
            continue
        gu = ((routed[a:b].double() @ w13[i].double().T).float() * rs[a:b, None]) * s13[i][None]
        g, u = gu[:, :inter], gu[:, inter:]
        hh = g / (1 + torch.exp(-g)) * u
        differ += int(((hh / (hh.abs().amax(-1, keepdim=True) / 127)).round().to(torch.int8) != q[a:b]).sum())
        assert torch.equal(((q[a:b].double() @ w2[i].double().T).float() * s[a:b, None]) * s2[i][None], y[a:b])
    assert differ <= 1e-3 * q.numel()


def test_weights_of_2_gib():
    """Weights past the descriptors of the direct-to-LDS kernel: the large-M kernel, and gate / up on the expert kernel."""
    gen, k, n = _gen(5), 16384, 131096
    w = torch.randint(-127, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
    sc = torch.rand(n, generator=gen, device="cuda") * 1e-3
    q = torch.randint(-127, 128, (1100, k), generator=gen, device="cuda", dtype=torch.int8)
    st = torch.rand(1100, generator=gen, device="cuda") * 0.01
    cols = torch.cat([torch.arange(8, device="cuda"), torch.arange(n - 16, n, device="cuda"),
                      torch.randint(0, n, (40,), generator=gen, device="cuda")])
    y = ops.w8a8_gemm(q, st, w, sc, None, torch.float16)
    acc = (q.double() @ w[cols].double().T).float()
    assert torch.equal(y[:, cols], ((acc * st[:, None]) * sc[cols][None]).half())
    del y
    rows, inter = 40, n // 2
    codes, s = ops.moe_gmm1_swiglu_quant(q[:rows], st[:rows].contiguous(), w.unsqueeze(0), sc.unsqueeze(0),
                                         torch.tensor([0, rows], device="cuda", dtype=torch.int64), inter)
    gu = torch.cat([(q[:rows].double() @ w[i:i + 8192].double().T).float() for i in range(0, n, 8192)], 1)
    gu = (gu * st[:rows, None]) * sc
    hh = gu[:, :inter] / (1 + torch.exp(-gu[:, :inter])) * gu[:, inter:]
    assert torch.allclose(s.view(-1), hh.abs().amax(-1) / 127, rtol=1e-5)
    diff = ((hh / s.view(-1, 1)).round().int() - codes.int()).abs()
    assert int(diff.max()) <= 1 and int((diff != 0).sum()) <= 1e-3 * codes.numel()


@pytest.mark.parametrize("rows,inter", [(1, 63), (3, 1027), (2, 2052), (300, 1030), (2049, 260)])
def test_gate_up_columns(rows, inter):
    """Column counts that vector accesses and the requant's column parts do not divide; codes up to exp's last bit."""
    gen = _gen(rows, inter)
    x = torch.randint(-127, 128, (rows, 256), generator=gen, device="cuda", dtype=torch.int8)
    rs = torch.rand(rows, generator=gen, device="cuda") * 0.01 + 1e-3
    w = torch.randint(-127, 128, (1, 2 * inter, 256), generator=gen, device="cuda", dtype=torch.int8)
    sc = torch.rand(1, 2 * inter, generator=gen, device="cuda") * 1e-3
    off = torch.tensor([0, rows], device="cuda", dtype=torch.int64)
    q, s = ops.moe_gmm1_swiglu_quant(x, rs, w, sc, off, inter)
    gu = ((x.double() @ w[0].double().T).float() * rs[:, None]) * sc
    hh = gu[:, :inter] / (1 + torch.exp(-gu[:, :inter])) * gu[:, inter:]
    amax = hh.abs().amax(-1)
    assert torch.allclose(s.view(-1), amax / 127, rtol=1e-5)
    diff = ((hh / (amax[:, None] / 127)).round().int() - q.int()).abs()
    assert int(diff.max()) <= 1 and int((diff != 0).sum()) <= max(1, 1e-3 * q.numel())


def test_light_ops_refuse_what_the_custom_ops_refuse():
    x = torch.randn(2, 128, device="cuda").half()
    w = torch.randint(-127, 128, (64, 128), device="cuda", dtype=torch.int8)
    sc = torch.ones(64, device="cuda")
    y = ops.w8a8_linear(x.clone().requires_grad_(True), w, sc, None, torch.float16, True)
    with pytest.raises(RuntimeError):
        y.sum().backward()
    with pytest.raises(RuntimeError, match="GPU"):
        ops.quant_per_token_i8(x.cpu())
    fn = torch.compile(lambda v: ops.w8a8_linear(v, w, sc, None, torch.float16, True), fullgraph=True, backend="aot_eager")
    assert torch.equal(fn(x), ops.w8a8_linear(x, w, sc, None, torch.float16, True))
    for op in (torch.ops.mindpipe_amd_light.quant_per_token_i8.default, torch.ops.mindpipe_amd.quant_per_token_i8.default):
        torch.library.opcheck(op, (x, True))
