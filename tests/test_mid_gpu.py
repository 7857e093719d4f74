"""The multi-stage kernel (17 to 2048 rows, K >= 1024) on the GPU: edges of its
row tiles, splits of K and ragged K, each weight format against its oracle."""
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


def _fp8_case(cuda, m, n, k, e5, adtype):
    """The call's metadata, its result held to float64: strided activation rows,
    scale and bias."""
    from rdna2_ops.fp8_weight_gemm_v06 import fp8_weight_gemm
    rng = np.random.default_rng(m * 1000 + n + k)
    codes = rng.integers(0, 256, (n, k)).astype(np.uint8)
    dec = o8.decode_bits(codes, e5)
    codes[~np.isfinite(dec) | (np.abs(dec) > 4)] = 0x30
    a = torch.from_numpy(rng.standard_normal((m, k + 8)).astype(np.float32)).to(adtype)[:, :k]
    scale = torch.from_numpy(rng.uniform(0.5, 2, n).astype(np.float32))
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(adtype)
    md = {}
    y = fp8_weight_gemm(a.to(cuda), codes_tensor(codes, e5, cuda), bias=bias.to(cuda), method="fused_dot2",
                        w_scale=scale.to(cuda), metadata=md)
    a64, w64 = a.double().numpy(), o8.decode_bits(codes, e5).astype(np.float64)
    s64, b64 = scale.double().numpy(), bias.double().numpy()
    check(y, (a64 @ w64.T) * s64 + b64, (np.abs(a64) @ np.abs(w64).T) * s64 + np.abs(b64), adtype, "mid fp8")
    return md


@pytest.mark.parametrize("m,n,k", [
    (17, 130, 1024), (32, 257, 1040), (33, 1, 4096), (64, 300, 12304), (65, 4096, 1152), (200, 1000, 2064),
    (333, 129, 3072), (1000, 700, 1024), (1030, 140, 1536), (40, 50, 1025),
])
@pytest.mark.parametrize("e5,adtype", [(False, torch.bfloat16), (True, torch.float16)])
def test_fp8_shapes(cuda, m, n, k, e5, adtype):
    """32-row tiles, splits, a last stage of a few chunks, packed operands (K %
    16 != 0), strided rows, scale and bias."""
    case(f"mid fp8 {m}x{n}x{k} e5={e5} {adtype}")
    md = _fp8_case(cuda, m, n, k, e5, adtype)
    assert md["variant"] == "fp8w_mid" and md["vgpr"] is not None and md["vgpr_spills"] == 0, md


@pytest.mark.parametrize("m,n,k,rows,split", [
    (300, 515, 1040, 32, False), (17, 130, 2064, 32, True), (333, 3001, 1041, 64, False), (33, 4100, 2064, 64, True),
    (1000, 2049, 1040, 128, False),
])
@pytest.mark.parametrize("e5,adtype", [(False, torch.float16), (True, torch.bfloat16), (False, torch.bfloat16)])
def test_fp8_tiles(cuda, m, n, k, rows, split, e5, adtype):
    """Each tile height, unsplit and split, with ragged rows, columns and K."""
    from rdna2_ops import _lib
    case(f"mid fp8 tile {m}x{n}x{k} e5={e5} {adtype}")
    md = _fp8_case(cuda, m, n, k, e5, adtype)
    assert md["variant"] == "fp8w_mid" and md["vgpr"] is not None and md["vgpr_spills"] == 0, md
    assert md["launched_tile"][0] == rows, md
    assert (_lib.library().qg_row_kernel_choice(_lib.CHOICE_FP8, 0, 0, m, n, k) >> 16 > 1) == split


@pytest.mark.parametrize("m,n,k", [(2049, 1921, 1040), (2049, 2113, 1025), (1500, 3001, 3080)])
@pytest.mark.parametrize("e5,adtype", [(False, torch.bfloat16), (True, torch.float16)])
def test_fp8_smaller_pingpong_grids(cuda, m, n, k, e5, adtype):
    """The ping-pong kernel below 192 tiles of 256 x 192: partial edge tiles,
    odd N, K that is no multiple of the stage (operands packed)."""
    case(f"fp8 ping-pong {m}x{n}x{k} e5={e5} {adtype}")
    md = _fp8_case(cuda, m, n, k, e5, adtype)
    assert md["variant"] == ("fp8w_f16_pingpong" if adtype == torch.float16 else "fp8w_bf16_pingpong"), md


@pytest.mark.parametrize("rows", [32, 64])
def test_fp8_one_hot_rows(cuda, rows):
    """One-hot activation rows read every K position of a stage and of a tail
    back exactly, on both tile heights."""
    from rdna2_ops.fp8_weight_gemm_v06 import fp8_weight_gemm
    case(f"mid fp8 one-hot {rows}")
    codes = np.arange(256, dtype=np.uint8)
    codes = codes[np.isfinite(o8.decode_bits(codes, False))]
    n, k = (4096 if rows == 64 else 64), 1104
    w = codes[(np.arange(n)[:, None] * 7 + np.arange(k)[None, :]) % len(codes)].astype(np.uint8)
    dec, wt = o8.decode_bits(w, False), codes_tensor(w, False, cuda)
    for k0 in range(0, k, 368):
        a = torch.zeros(368, k, dtype=torch.bfloat16)
        a[torch.arange(368), k0 + torch.arange(368)] = 1
        y = fp8_weight_gemm(a.to(cuda), wt, method="fused_dot2")
        assert np.array_equal(y.float().cpu().numpy(), dec[:, k0:k0 + 368].T.astype(np.float32)), k0


def test_fp8_values_past_k(cuda):
    """Weight bytes after the last K element (NaN codes) do not reach the result."""
    from rdna2_ops.fp8_weight_gemm_v06 import fp8_weight_gemm
    case("mid fp8 NaN past K")
    n, k, pitch = 24, 1040, 1280
    store = np.full((n, pitch), 0x7f, np.uint8)
    store[:, :k] = 0x38  # 1.0
    w = codes_tensor(store, False, cuda)[:, :k]
    y = fp8_weight_gemm(torch.ones(20, k, dtype=torch.bfloat16, device=cuda), w, method="fused_dot2")
    assert torch.equal(y.float().cpu(), torch.full((20, n), float(k)))


def _int4_case(cuda, m, n, k, g, sym, order, adtype):
    """The call's metadata, its result held to the exact product of the packed
    weight: signed INT4 (nk), strided activation rows, bias."""
    from rdna2_ops import int4_weight_gemm_v07 as w4
    gen = torch.Generator().manual_seed(m + n + k + g)
    w = torch.randn(n, k, generator=gen) * 0.02
    a = torch.randn(m, k + 8, generator=gen).to(adtype)[:, :k]
    b = (torch.randn(n, generator=gen) * 0.1).to(adtype)
    p = w4.pack_int4(w.to(cuda), group_size=g, symmetric=sym, order=order)
    cen = w4.unpack_int4(p, dtype=torch.int8).cpu().numpy().astype(np.int32)
    av, s = act_values(a), p.scales.cpu().numpy()
    y64 = o4.w4a16_linear(av, cen, s, g, act_values(b))
    y, md = w4.int4_linear_a16(a.to(cuda), p, bias=b.to(cuda), method="dot2", return_kernel=True)
    check_product(y, y64, o4.w4a16_linear(np.abs(av), np.ones_like(cen), s, g), adtype, f"mid int4 {m}x{n}x{k} g{g}")
    return md


@pytest.mark.parametrize("m,n,k", [(17, 130, 1088), (64, 300, 4096), (65, 4100, 1152), (333, 257, 2048),
                                   (700, 1030, 1024), (1024, 1100, 3072)])
@pytest.mark.parametrize("g", o4.GROUPS)
@pytest.mark.parametrize("sym,order,adtype", [(True, "low", torch.float16), (False, "high", torch.bfloat16)])
def test_int4_shapes(cuda, m, n, k, g, sym, order, adtype):
    """Signed INT4 (nk): splits, a last stage of fewer groups, both nibble
    orders, bias; 17 rows of a short K stay on the older kernel, to the same
    bound."""
    k = k // g * g
    case(f"mid int4 {m}x{n}x{k} g{g} sym={sym} {order} {adtype}")
    md = _int4_case(cuda, m, n, k, g, sym, order, adtype)
    assert md["variant"] == ("w4a16_skinny" if m == 17 else "w4a16_mid"), md
    assert md["vgpr"] is not None and md["vgpr_spills"] == 0, md


INT4_TILES = [(65, 33, 1024, 128, 32, False), (33, 33, 2048, 128, 32, True), (333, 3000, 1024, 128, 64, False),
              (33, 2049, 6144, 128, 64, True), (1000, 2049, 1024, 128, 128, False), (300, 1537, 4096, 128, 128, True)]


@pytest.mark.parametrize("m,n,k,g,rows,split", INT4_TILES + [
    (90, 33, 1088, 64, 32, False), (33, 33, 2112, 64, 32, True), (333, 3000, 1088, 64, 64, False),
    (33, 4100, 6144, 64, 64, True), (1000, 2049, 1088, 64, 128, False), (700, 257, 4160, 64, 128, True),
    (90, 700, 1056, 32, 32, False), (33, 33, 2080, 32, 32, True), (333, 3000, 1056, 32, 64, False),
    (33, 2049, 4128, 32, 64, True),
])
@pytest.mark.parametrize("sym,order,adtype", [(False, "low", torch.float16), (True, "high", torch.bfloat16)])
def test_int4_tiles(cuda, m, n, k, g, rows, split, sym, order, adtype):
    """Each tile height of each group size, unsplit and split, with ragged rows,
    columns and (groups below 128) K."""
    case(f"mid int4 tile {m}x{n}x{k} g{g} sym={sym} {order} {adtype}")
    md = _int4_case(cuda, m, n, k, g, sym, order, adtype)
    assert md["variant"] == "w4a16_mid" and md["vgpr"] is not None and md["vgpr_spills"] == 0, md
    assert md["tile"][0] == rows and (md["k_splits"] > 1) == split, md


@pytest.mark.parametrize("m,n,k,rows,split", [(20, 140, 14336, 32, True), (48, 4097, 1152, 32, False),
                                              (96, 520, 4096, 32, True), (512, 1000, 2048, 64, True)]
                         + [(m, n, k, rows, split) for m, n, k, _, rows, split in INT4_TILES])
@pytest.mark.parametrize("adtype", [torch.float16, torch.bfloat16])
def test_uint4_shapes(cuda, m, n, k, rows, split, adtype):
    """uint4 storage (bf16 scales, packed zero points): each tile height,
    unsplit and split."""
    from rdna2_ops import int4_weight_gemm_v07 as w4
    case(f"mid uint4 {m}x{n}x{k} {adtype}")
    gen = torch.Generator().manual_seed(m + n + k)
    w = torch.randn(n, k, generator=gen) * 0.02
    a = torch.randn(m, k, generator=gen).to(adtype)
    p = w4.pack_uint4(w.to(cuda), group_size=128)
    cen = w4.unpack_int4(p, dtype=torch.int8).cpu().numpy().astype(np.int32)
    av, s = act_values(a), p.scales.float().cpu().numpy()
    y, md = w4.int4_linear_a16(a.to(cuda), p, method="dot2", return_kernel=True)
    assert md["variant"] == "w4a16_mid" and md["vgpr"] is not None and md["vgpr_spills"] == 0, md
    assert md["tile"][0] == rows and (md["k_splits"] > 1) == split, md
    check_product(y, o4.w4a16_linear(av, cen, s, 128), o4.w4a16_linear(np.abs(av), np.ones_like(cen), s, 128),
                  adtype, f"mid uint4 {m}x{n}x{k}")


@pytest.mark.parametrize("m,n,k,g", [
    (300, 513, 4096, 32), (100, 140, 1120, 32), (300, 4096, 4096, 64), (100, 300, 1088, 64), (1024, 1030, 2048, 128),
    (100, 260, 4096, 128),
])
@pytest.mark.parametrize("sym,adtype", [(True, torch.float16), (False, torch.bfloat16)])
def test_int4_infinite_activations(cuda, m, n, k, g, sym, adtype):
    """An infinite activation gives what the dequantized weights give: +-inf,
    or NaN where the weight is zero or infinities of both signs meet; sums past
    fp32's range on the way (bf16) stay finite, and the other rows' bits do not
    change."""
    from rdna2_ops import int4_weight_gemm_v07 as w4
    case(f"mid int4 inf {m}x{n}x{k} g{g} sym={sym} {adtype}")
    gen = torch.Generator().manual_seed(m + n + k + g)
    p = w4.pack_int4((torch.randn(n, k, generator=gen) * 0.02).to(cuda), group_size=g, symmetric=sym)
    w = (w4.unpack_int4(p, dtype=torch.int8).double().reshape(n, k // g, g) * p.scales.double()[..., None]).reshape(n, k)
    a = torch.randn(m, k, generator=gen).to(adtype)
    before = w4.w4a16_gemm(a.to(cuda), p)
    rows = {1: {k - 3: float("inf")}, m // 2: {5: -float("inf")}, m - 1: {0: float("inf"), k // 2: float("inf")},
            m - 2: {9: float("inf"), k - 1: -float("inf")}, 7: {11: float("nan")}}
    for r, at in rows.items():
        for c, v in at.items():
            a[r, c] = v
    if adtype == torch.bfloat16:
        rows[3] = None
        a[3] = torch.randn(k, generator=gen).bfloat16() * 2.0 ** 120
    y, md = w4.int4_linear_a16(a.to(cuda), p, method="dot2", return_kernel=True)
    assert md["variant"] == "w4a16_mid", md
    rest = [r for r in range(m) if r not in rows]
    assert torch.equal(y[rest], before[rest])
    for r in rows:
        ref = (a[r].double().to(cuda) * w).sum(-1)
        got = y[r].double()
        assert torch.equal(got.isnan(), ref.isnan()), r
        assert torch.equal(got[got.isinf()], ref[ref.isinf()]) and torch.equal(got.isinf(), ref.isinf()), r
    if adtype == torch.bfloat16:
        assert ((got - ref).abs() <= 1e-2 * ref.square().mean().sqrt() + 2.0 ** -8 * ref.abs()).all()


def test_int4_without_workspace(cuda):
    """A call without the workspace of its partial tiles runs unsplit."""
    from rdna2_ops import _lib
    from rdna2_ops import int4_weight_gemm_v07 as w4
    case("mid int4 no workspace")
    gen = torch.Generator().manual_seed(5)
    m, n, k = 100, 260, 4096
    p = w4.pack_uint4((torch.randn(n, k, generator=gen) * 0.02).to(cuda), group_size=128)
    a = torch.randn(m, k, generator=gen).to(torch.bfloat16).to(cuda)
    lib, P = _lib.library(), _lib.ptr
    assert lib.qg_w4a16_gemm_workspace_bytes(m, n, k, 128, p.flags) > 0
    out = torch.empty(m, n, device=cuda)
    _lib.check(lib.qg_w4a16_gemm(P(a), _lib.BF16, k, m, k, P(p.data), n, 128, p.flags, P(p.scales), _lib.BF16,
                                 P(p.zeros), None, 0, P(out), _lib.F32, None, 0, _lib.stream_of(a)), "qg_w4a16_gemm")
    ref = w4.w4a16_gemm(a, p, out_dtype=torch.float32)
    assert (out - ref).abs().max().item() <= 1e-4 * ref.abs().max().item()  # fp32 sums in another order


@pytest.mark.parametrize("m,n,k,g,room,taken", [
    (1000, 1024, 14336, 32, 2 * 1024 * 14336, True),   # 8 splits planned, which need more: dequant
    (100, 4096, 4096, 32, 2 * 4096 * 4096, True), (100, 4096, 4096, 32, 0, False),
    (300, 4096, 4096, 32, 1 << 20, False),             # parameters of K past LDS, no room to dequantize
    (200, 1000, 1536, 32, 0, True), (300, 8192, 4096, 64, 0, True),  # unsplit
    (300, 8192, 8192, 64, 2 * 8192 * 8192, True), (300, 8192, 8192, 64, 0, False),
    (40, 300, 8192, 64, 0, True), (1024, 4096, 8192, 64, 2 * 4096 * 8192, True),
])
def test_int4_with_less_workspace(cuda, m, n, k, g, room, taken):
    """Less workspace than the query reports: the dequant formulation's 2 n k
    bytes always suffice, without them the call runs unsplit where it can."""
    from rdna2_ops import _lib
    from rdna2_ops import int4_weight_gemm_v07 as w4
    case(f"mid int4 {m}x{n}x{k} g{g} room {room}")
    gen = torch.Generator().manual_seed(m + n + k + g)
    p = w4.pack_int4((torch.randn(n, k, generator=gen) * 0.02).to(cuda), group_size=g)
    a = torch.randn(m, k, generator=gen).to(torch.bfloat16).to(cuda)
    lib, P = _lib.library(), _lib.ptr
    ws = torch.empty(max(room, 256), dtype=torch.uint8, device=cuda)
    out = torch.empty(m, n, device=cuda)
    status = lib.qg_w4a16_gemm(P(a), _lib.BF16, k, m, k, P(p.data), n, g, p.flags, P(p.scales), _lib.F32, P(p.zeros),
                               None, 0, P(out), _lib.F32, P(ws) if room else None, room, _lib.stream_of(a))
    assert (status == 0) == taken, status
    if taken:
        ref = a.double() @ w4.unpack_int4(p, dtype=torch.float32).double().T
        # weights rounded to bf16 at worst: 2^-9 of each product, so of their root sum of squares
        assert (out - ref).norm() <= 2.0 ** -8 * ref.norm()


@pytest.mark.parametrize("m,n,k", [(17, 140, 6160), (64, 300, 12288), (65, 1000, 4096), (130, 257, 6160),
                                   (256, 3072, 8192), (300, 513, 8192)])
def test_int8_split_shapes(cuda, m, n, k):
    """int32 sums of split K bit-exact, and the epilogue orders of the second
    launch; without workspace the tiled kernel gives the same bits."""
    from rdna2_ops import _lib
    from rdna2_ops.int8_gemm import int8_gemm_dequant, int8_matmul
    case(f"mid int8 {m}x{n}x{k}")
    g = torch.Generator().manual_seed(m * 31 + n * 7 + k)
    a = torch.randint(-128, 128, (m, k), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    sa, sb = torch.rand(m, generator=g) * 0.02 + 0.001, torch.rand(n, generator=g) * 0.02 + 0.001
    bias = torch.randn(n, generator=g)
    acc = oi.int8_matmul(a.numpy(), np.ascontiguousarray(w.numpy().T))
    ag, wg, sag, sbg, bg = a.to(cuda), w.to(cuda), sa.to(cuda), sb.to(cuda), bias.to(cuda)
    assert np.array_equal(int8_matmul(ag, wg.T).cpu().numpy(), acc)
    y, md = int8_gemm_dequant(ag, wg.T, sag, sbg, bg, out_dtype=torch.float16, return_kernel=True)
    assert md["variant"] == "int8_mfma_16x16x64_split" and md["k_splits"] > 1 and md["vgpr"] is not None, md
    ref = oi.epilogue_f(acc, sa.numpy(), sb.numpy(), bias.numpy(), out="f16")
    assert np.array_equal(y.float().cpu().numpy(), np.asarray(oi.round_to(ref, "f16"), np.float32))
    y = int8_gemm_dequant(ag, wg.T, sag, sbg, bg, out_dtype=torch.bfloat16, epilogue_order="eager")
    ref = oi.epilogue_e(acc, sa.numpy(), sb.numpy(), bias.numpy(), out="bf16")
    assert np.array_equal(y.float().cpu().numpy(), np.asarray(oi.round_to(ref, "bf16"), np.float32))
    if k % 128 == 0:
        out = torch.empty(m, n, dtype=torch.int32, device=cuda)
        P = _lib.ptr
        _lib.check(_lib.library().qg_int8_gemm(P(ag), k, 1, P(wg), 1, k, m, n, k, None, None, 0, None, 0, P(out),
                                               _lib.I32, 0, None, 0, _lib.stream_of(ag)), "qg_int8_gemm")
        assert np.array_equal(out.cpu().numpy(), acc)
