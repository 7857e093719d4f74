"""The few-row (M <= 16) streaming kernel on the GPU: the edges of its row
counts, column tiles and K chunks, each weight format against its oracle."""
import numpy as np
import pytest
import torch

from conftest import case
from oracle import fp8 as o8
from oracle import int4 as o4
from oracle import int8 as oi
from test_fp8_gpu import check, codes_tensor
from test_w4_gpu import act_values, check_product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e5", [False, True])
@pytest.mark.parametrize("adtype", [torch.bfloat16, torch.float16])
def test_fp8_one_hot_rows(cuda, e5, adtype):
    """One-hot activation rows read every K position of a whole chunk, a
    second one and a 16-element tail back exactly: the K order of A and W."""
    from rdna2_ops.fp8_weight_gemm_v06 import fp8_weight_gemm
    case(f"skinny fp8 one-hot e5={e5} {adtype}")
    codes = np.arange(256, dtype=np.uint8)
    codes = codes[np.isfinite(o8.decode_bits(codes, e5))]
    n, k = 37, 272
    w = codes[(np.arange(n)[:, None] * 7 + np.arange(k)[None, :]) % len(codes)].astype(np.uint8)
    dec = o8.decode_bits(w, e5)
    wt = codes_tensor(w, e5, cuda)
    for k0 in range(0, k, 16):
        a = torch.zeros(16, k, dtype=adtype)
        a[torch.arange(16), k0 + torch.arange(16)] = 1
        y = fp8_weight_gemm(a.to(cuda), wt, method="fused_dot2")
        assert np.array_equal(y.float().cpu().numpy(), dec[:, k0:k0 + 16].T.astype(np.float32)), k0


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 16), (2, 16, 128), (4, 17, 144), (5, 33, 1024), (8, 47, 1040), (9, 48, 2064), (16, 4097, 256),
    (16, 768, 3072), (3, 8208, 384), (7, 12304, 160), (16, 20, 8), (11, 31, 257),
])
@pytest.mark.parametrize("e5,adtype", [(False, torch.bfloat16), (True, torch.float16)])
def test_fp8_shapes(cuda, m, n, k, e5, adtype):
    """Rows, column tiles of one to three, chunks past a wave's first, tails
    and (K % 16 != 0) packed operands; scale and bias; strided activations."""
    from rdna2_ops.fp8_weight_gemm_v06 import fp8_weight_gemm
    case(f"skinny fp8 {m}x{n}x{k} e5={e5} {adtype}")
    rng = np.random.default_rng(m * 1000 + n + k)
    codes = rng.integers(0, 256, (n, k)).astype(np.uint8)
    bad = ~np.isfinite(o8.decode_bits(codes, e5)) | (np.abs(o8.decode_bits(codes, e5)) > 4)
    codes[bad] = 0x30
    a = torch.from_numpy(rng.standard_normal((m, k + 8)).astype(np.float32)).to(adtype)
    scale = torch.from_numpy(rng.uniform(0.5, 2, n).astype(np.float32))
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(adtype)
    ac = a.to(cuda)[:, :k]
    y = fp8_weight_gemm(ac, codes_tensor(codes, e5, cuda), bias=bias.to(cuda), method="fused_dot2",
                        w_scale=scale.to(cuda))
    a64, w64 = a[:, :k].double().numpy(), o8.decode_bits(codes, e5).astype(np.float64)
    s64, b64 = scale.double().numpy(), bias.double().numpy()
    check(y, (a64 @ w64.T) * s64 + b64, (np.abs(a64) @ np.abs(w64).T) * s64 + np.abs(b64), adtype, "skinny fp8")


def test_fp8_values_past_k(cuda):
    """Weight bytes after the last K element of a row (the next row's, here
    NaN codes) do not reach the result."""
    from rdna2_ops.fp8_weight_gemm_v06 import fp8_weight_gemm
    case("skinny fp8 NaN past K")
    n, k, pitch = 24, 144, 256
    store = np.full((n, pitch), 0x7f, np.uint8)
    store[:, :k] = 0x38  # 1.0
    w = codes_tensor(store, False, cuda)[:, :k]
    y = fp8_weight_gemm(torch.ones(3, k, dtype=torch.bfloat16, device=cuda), w, method="fused_dot2")
    assert torch.equal(y.float().cpu(), torch.full((3, n), float(k)))


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 640), (4, 17, 1088), (5, 33, 2176), (8, 4100, 768), (9, 47, 4160), (16, 16, 2048), (16, 8208, 1024),
    (16, 14337, 640), (3, 96, 512),
])
@pytest.mark.parametrize("g", o4.GROUPS)
@pytest.mark.parametrize("sym,order,adtype", [(True, "low", torch.float16), (False, "high", torch.bfloat16)])
def test_int4_shapes(cuda, m, n, k, g, sym, order, adtype):
    """Signed INT4 (nk): row counts, one to four column tiles, an odd number
    of groups and a last chunk of fewer groups, both nibble orders, bias."""
    from rdna2_ops import int4_weight_gemm_v07 as w4
    k = k // g * g
    case(f"skinny int4 {m}x{n}x{k} g{g} sym={sym} {order} {adtype}")
    gen = torch.Generator().manual_seed(m + n + k + g)
    w = torch.randn(n, k, generator=gen) * 0.02
    a = torch.randn(m, k + 8, generator=gen).to(adtype)[:, :k]
    b = (torch.randn(n, generator=gen) * 0.1).to(adtype)
    p = w4.pack_int4(w.to(cuda), group_size=g, symmetric=sym, order=order)
    cen = w4.unpack_int4(p, dtype=torch.int8).cpu().numpy().astype(np.int32)
    s = p.scales.cpu().numpy()
    av = act_values(a)
    y64 = o4.w4a16_linear(av, cen, s, g, act_values(b))
    absmag = o4.w4a16_linear(np.abs(av), np.ones_like(cen), s, g)
    y = w4.int4_linear_a16(a.to(cuda), p, bias=b.to(cuda), method="dot2")
    check_product(y, y64, absmag, adtype, f"skinny int4 {m}x{n}x{k} g{g}")


@pytest.mark.parametrize("m,n,k", [(1, 50, 1152), (2, 33, 14336), (6, 4097, 1152), (16, 40, 14336), (16, 12300, 3200)])
@pytest.mark.parametrize("adtype", [torch.float16, torch.bfloat16])
def test_uint4_shapes(cuda, m, n, k, adtype):
    """uint4 storage with bf16 scales: an odd number of groups (a column's
    scales start in the upper half of a word) and K past the decode kernels'."""
    from rdna2_ops import int4_weight_gemm_v07 as w4
    case(f"skinny uint4 {m}x{n}x{k} {adtype}")
    gen = torch.Generator().manual_seed(m + n + k)
    w = torch.randn(n, k, generator=gen) * 0.02
    a = torch.randn(m, k, generator=gen).to(adtype)
    p = w4.pack_uint4(w.to(cuda), group_size=128)
    cen = w4.unpack_int4(p, dtype=torch.int8).cpu().numpy().astype(np.int32)
    s = p.scales.float().cpu().numpy()
    av = act_values(a)
    y64 = o4.w4a16_linear(av, cen, s, 128)
    absmag = o4.w4a16_linear(np.abs(av), np.ones_like(cen), s, 128)
    y = w4.int4_linear_a16(a.to(cuda), p, method="dot2")
    check_product(y, y64, absmag, adtype, f"skinny uint4 {m}x{n}x{k}")


def test_int4_parameters_past_lds(cuda):
    """More groups than fit next to the rings (group 32, K 32768): the
    kernel without LDS parameters."""
    from rdna2_ops import int4_weight_gemm_v07 as w4
    case("skinny int4 g32 k32768")
    gen = torch.Generator().manual_seed(3)
    n, k, g = 24, 32768, 32
    w = torch.randn(n, k, generator=gen) * 0.02
    a = torch.randn(3, k, generator=gen).to(torch.bfloat16)
    p = w4.pack_int4(w.to(cuda), group_size=g)
    cen = w4.unpack_int4(p, dtype=torch.int8).cpu().numpy().astype(np.int32)
    av, s = act_values(a), p.scales.cpu().numpy()
    y, md = w4.int4_linear_a16(a.to(cuda), p, method="dot2", return_kernel=True)
    assert md["variant"] == "w4a16_skinny"
    check_product(y, o4.w4a16_linear(av, cen, s, g), o4.w4a16_linear(np.abs(av), np.ones_like(cen), s, g),
                  torch.bfloat16, "skinny int4 g32 k32768")


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 16), (2, 17, 144), (8, 33, 1040), (9, 48, 2064), (16, 4097, 256), (16, 768, 3072), (3, 12304, 160),
    (16, 20, 8), (11, 31, 257), (4, 40, 131056),
])
def test_int8_shapes(cuda, m, n, k):
    """int32 sums bit-exact (tails, packed operands, strided rows), and every
    epilogue against the oracle: orders F, FMA and eager, GELU within the
    activation's own bound elsewhere; scalar and per-column scales."""
    from rdna2_ops.int8_gemm import int8_gemm_dequant, int8_matmul
    case(f"skinny int8 {m}x{n}x{k}")
    g = torch.Generator().manual_seed(m * 31 + n * 7 + k)
    a = torch.randint(-128, 128, (m, k + 16), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    sa, sb = torch.rand(m, generator=g) * 0.02 + 0.001, torch.rand(n, generator=g) * 0.02 + 0.001
    bias = torch.randn(n, generator=g)
    acc = oi.int8_matmul(a[:, :k].numpy(), np.ascontiguousarray(w.numpy().T))
    ag, wg, sag, sbg, bg = a.to(cuda)[:, :k], w.to(cuda), sa.to(cuda), sb.to(cuda), bias.to(cuda)
    assert np.array_equal(int8_matmul(ag, wg.T).cpu().numpy(), acc)
    for out, dt in (("f32", torch.float32), ("f16", torch.float16), ("bf16", torch.bfloat16)):
        def same(got, ref):
            return np.array_equal(got.cpu().float().numpy(), np.asarray(oi.round_to(ref, out), np.float32))
        kw = dict(out_dtype=dt)
        assert same(int8_gemm_dequant(ag, wg.T, sag, sbg, bg, **kw),
                    oi.epilogue_f(acc, sa.numpy(), sb.numpy(), bias.numpy(), out=out))
        assert same(int8_gemm_dequant(ag, wg.T, sag, sbg[:1].contiguous(), None, **kw),
                    oi.epilogue_f(acc, sa.numpy(), np.full(n, sb[0].item(), np.float32), None, out=out))
        assert same(int8_gemm_dequant(ag, wg.T, sag, sbg, bg, epilogue_order="eager", **kw),
                    oi.epilogue_e(acc, sa.numpy(), sb.numpy(), bias.numpy(), out=out))
    y, md = int8_gemm_dequant(ag, wg.T, sag, sbg, bg, rounding="fused", return_kernel=True)
    assert md["variant"] == "int8_mfma_16x16x64_skinny" and md["vgpr"] is not None
    scale = (sa.numpy()[:, None] * sb.numpy()[None, :]).astype(np.float32)
    ref = (acc.astype(np.float32).astype(np.float64) * scale + bias.numpy()).astype(np.float32)  # one rounding
    assert np.array_equal(y.cpu().numpy(), ref)


@pytest.mark.parametrize("m,k", [(2, 3072), (16, 1040), (5, 200)])
def test_int8_linear_same_as_wider_batch(cuda, m, k):
    """The W8A8 linear of a few rows equals the same rows of a wider batch
    (the tiled kernels) bit for bit: quantizer, GELU, residual and scale."""
    from rdna2_ops.int8_gemm import w8a8_linear
    case(f"skinny w8a8 {m}x{k}")
    g = torch.Generator().manual_seed(k)
    n = 150
    x = torch.randn(40, k, generator=g).to(torch.float16).to(cuda)
    w = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8).to(cuda)
    ws, b = (torch.rand(n, generator=g) * 0.01).to(cuda), torch.randn(n, generator=g).to(cuda)
    res = torch.randn(40, n, generator=g).to(torch.bfloat16).to(cuda)
    rs = torch.rand(n, generator=g).to(cuda)
    for kw in (dict(), dict(activation="gelu_tanh"), dict(residual=True), dict(activation="gelu_tanh", residual=True)):
        def call(rows):
            extra = dict(kw)
            if extra.pop("residual", False):
                extra.update(residual=res[:rows], residual_scale=rs)
            return w8a8_linear(x[:rows], w, ws, b, **extra)
        assert torch.equal(call(m).view(torch.int16), call(40)[:m].view(torch.int16)), kw
