"""GPU parity: narrow GeMM (layoutA / layoutAB_ContinuousC / layoutABC, soft-FP8) against the
oracle's float64 product on the un-packed weights, rtol = atol = 1e-2, through the C ABI."""
import numpy as np
import pytest
import torch

from muxi_native_layout_kernels_amd import ops
from oracle import gemm as ogemm, layouts
from helpers import randn, pack_a, pack_b, fp8_codes, assert_close, bits

pytestmark = pytest.mark.gpu

RTOL = ATOL = 1e-2


@pytest.mark.parametrize("m", [1, 8, 16, 32, 64])
def test_gemm_layout_a_fp16_config(mlk, m):
    n, k = 11008, 4096
    w = randn((n, k), torch.float16, 0.02, 2025)
    b = randn((m, k), torch.float16, 1.0, 2026 + m)
    c = mlk.gemm_layoutA(pack_a(w).cuda(), b.cuda())
    assert c.shape == (m, n) and c.dtype == torch.float16
    assert_close(c, ogemm.linear_expected(w, b), RTOL, ATOL, "gemm_layoutA M=%d" % m)


@pytest.mark.parametrize("m", [1, 3, 15, 17, 33, 48, 63, 65, 100, 130])
def test_gemm_layout_a_ragged_tokens(mlk, m):
    n, k = 256, 512
    w = randn((n, k), torch.bfloat16, 0.05, 1)
    b = randn((m, k), torch.bfloat16, 1.0, 2)
    c = mlk.gemm_layoutA(pack_a(w).cuda(), b.cuda())
    assert_close(c, ogemm.linear_expected(w, b), RTOL, ATOL, "ragged M=%d" % m)


@pytest.mark.parametrize("p1,p2,p3", [(1, 1, 1), (1, 4, 1), (2, 2, 1), (4, 4, 1), (1, 16, 1), (2, 8, 1), (1, 1, 4),
                                      (2, 4, 3), (4, 2, 8), (1, 2, 64)])
@pytest.mark.parametrize("m", [16, 40, 64])
def test_gemm_launch_parameters(mlk, p1, p2, p3, m):
    n, k = 512, 2048
    w = randn((n, k), torch.bfloat16, 0.02, 3)
    b = randn((m, k), torch.bfloat16, 1.0, 4)
    bias = randn((1, n), torch.bfloat16, 1.0, 5)
    a = pack_a(w).cuda()
    want = ogemm.linear_expected(w, b, 0.75, bias)
    c = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.75, kernelParam1=p1, kernelParam2=p2, kernelParam3=p3,
                                kernelId=1, bias=bias.cuda())
    assert_close(c, want, RTOL, ATOL, "params")
    c2 = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.75, kernelParam1=p1, kernelParam2=p2,
                                 kernelParam3=p3, kernelId=1, bias=bias.cuda())
    assert torch.equal(c, c2), "K split across workgroups must be deterministic and leave its counters clean"


@pytest.mark.parametrize("p1,p3", [(1, 1), (2, 1), (4, 1), (1, 2), (2, 4), (4, 8)])
@pytest.mark.parametrize("m", [16, 33, 48, 64, 100])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gemm_tile_kernel(mlk, p1, p3, m, dtype):
    """kernelId 2: row-shared tile kernel, row-major and native operands, K split across workgroups."""
    n, k = 1024, 2048
    w = randn((n, k), dtype, 0.02, 13)
    b = randn((m, k), dtype, 1.0, 14)
    bias = randn((1, n), dtype, 1.0, 15)
    a = pack_a(w).cuda()
    want = ogemm.linear_expected(w, b, 1.25, bias)
    c = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=1.25, kernelParam1=p1, kernelParam2=1, kernelParam3=p3,
                                kernelId=2, bias=bias.cuda())
    assert_close(c, want, RTOL, ATOL, "tile kernel")
    assert torch.equal(c, mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=1.25, kernelParam1=p1, kernelParam2=1,
                                                  kernelParam3=p3, kernelId=2, bias=bias.cuda()))
    if m % 16 == 0:
        b_nat = mlk.layoutB(b.cuda())
        c_rm = mlk.gemm_layoutAB_ContinuousC_wapper(a, b_nat, n, m, k, alpha=1.25, kernelParam1=p1, kernelParam3=p3,
                                                    kernelId=2, bias=bias.cuda())
        c_nat = mlk.gemm_layoutABC_wapper(a, b_nat, n, m, k, alpha=1.25, kernelParam1=p1, kernelParam3=p3, kernelId=2,
                                          bias=bias.cuda())
        assert torch.equal(c_rm, c) and torch.equal(mlk.reLayoutC(c_nat), c)


def test_gemm_tile_kernel_soft_fp8(mlk):
    n, k, m = 1024, 2048, 40
    codes = fp8_codes((n, k), 21)
    b = randn((m, k), torch.bfloat16, 1.0, 22)
    g = torch.Generator().manual_seed(23)
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float()
    c = mlk.gemm_layoutA_soft_fp8_wapper(pack_a(codes).cuda(), scale.cuda(), b.cuda(), n, m, k, kernelParam1=2,
                                         kernelParam3=2, kernelId=2)
    assert_close(c, ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), b), RTOL, ATOL, "tile fp8")


@pytest.mark.parametrize("kid", [12, 14, 16, 18])
@pytest.mark.parametrize("p1,p2,p3", [(1, 1, 1), (4, 2, 1), (2, 8, 2), (1, 16, 1), (8, 4, 1), (8, 2, 2)])
@pytest.mark.parametrize("m", [1, 7, 16, 40])
def test_gemm_ring_depth_kernel_ids(mlk, kid, p1, p2, p3, m):
    """kernelId 12..18: kernel 1 with 2..8 k tiles in flight per wave.  The summation order does not depend
    on the depth, so the result is bit-equal to kernel 1's; above 16 tokens the ids mean kernel 1."""
    n, k = 512, 1024 + 32 * 5                    # 37 k tiles: fewer than, equal to and more than the ring at some split
    w = randn((n, k), torch.float16, 0.02, 31)
    b = randn((m, k), torch.float16, 1.0, 32)
    a = pack_a(w).cuda()
    c = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, kernelParam1=p1, kernelParam2=p2, kernelParam3=p3, kernelId=kid)
    assert_close(c, ogemm.linear_expected(w, b), RTOL, ATOL, "ring depth id %d" % kid)
    c1 = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, kernelParam1=p1, kernelParam2=p2, kernelParam3=p3, kernelId=1)
    assert torch.equal(c, c1)


def test_gemm_ring_depth_soft_fp8(mlk):
    n, k, m = 512, 1024, 9
    codes = fp8_codes((n, k), 41)
    b = randn((m, k), torch.bfloat16, 1.0, 42)
    g = torch.Generator().manual_seed(43)
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float()
    for kid in (12, 14, 16, 18):
        for p1 in (2, 8):         # eight row groups per wave = one 128-row scale block
            c = mlk.gemm_layoutA_soft_fp8_wapper(pack_a(codes).cuda(), scale.cuda(), b.cuda(), n, m, k, kernelParam1=p1,
                                                 kernelParam2=4, kernelParam3=1, kernelId=kid)
            assert_close(c, ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), b), RTOL, ATOL, "fp8 depth")


@pytest.mark.parametrize("m", [65, 100, 128, 130, 200, 256, 300])
@pytest.mark.parametrize("p1,p3", [(1, 1), (2, 1), (2, 2), (4, 4)])
def test_gemm_tile_kernel_wide_passes(mlk, m, p1, p3):
    """More than 64 tokens with kernelId 2 on row-major operands: passes of up to 128 tokens over the weights."""
    n, k = 512, 1024
    w = randn((n, k), torch.bfloat16, 0.02, 51)
    b = randn((m, k), torch.bfloat16, 1.0, 52)
    bias = randn((1, n), torch.bfloat16, 1.0, 53)
    a = pack_a(w).cuda()
    c = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.5, kernelParam1=p1, kernelParam2=1, kernelParam3=p3,
                                kernelId=2, bias=bias.cuda())
    assert_close(c, ogemm.linear_expected(w, b, 0.5, bias), RTOL, ATOL, "wide passes M=%d" % m)
    c2 = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.5, kernelParam1=p1, kernelParam2=1, kernelParam3=p3,
                                 kernelId=2, bias=bias.cuda())
    assert torch.equal(c, c2)


def test_gemm_wide_default_parameters(mlk):
    """A shape that is in no table, above 64 tokens: the heuristic picks the panel kernel (K % 128 == 0)."""
    n, k, m = 768, 512, 150
    w = randn((n, k), torch.float16, 0.02, 61)
    b = randn((m, k), torch.float16, 1.0, 62)
    c = mlk.gemm_layoutA(pack_a(w).cuda(), b.cuda())
    assert_close(c, ogemm.linear_expected(w, b), RTOL, ATOL, "wide default")
    codes = fp8_codes((n, k), 63)
    g = torch.Generator().manual_seed(64)
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float()
    bb = randn((m, k), torch.bfloat16, 1.0, 65)
    c8 = mlk.gemm_layoutA_linear(pack_a(codes).cuda(), bb.cuda(), scale_matrix=scale.cuda())
    assert_close(c8, ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), bb), RTOL, ATOL, "wide default fp8")


@pytest.mark.parametrize("m", [1, 65, 128, 129, 200, 256, 300, 640])
@pytest.mark.parametrize("n,k,p3", [(512, 256, 1), (272, 384, 1), (272, 384, 3), (1040, 1024, 2), (256, 128, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gemm_panel_kernel(mlk, m, n, k, p3, dtype):
    """kernelId 3: 256-row x 128-token panels with MFMA 32x32x16; ragged token counts, row counts that are not
    a multiple of 256 (or of 32: 272 = 17 row groups), K slices that do not divide the windows evenly, one
    window per slice, more slices than windows."""
    w = randn((n, k), dtype, 0.05, 91)
    b = randn((m, k), dtype, 1.0, 92)
    bias = randn((1, n), dtype, 1.0, 93)
    a = pack_a(w).cuda()
    # (rows, tokens) of a panel: 128 x 128, 256 x 128, 256 x 256, both chosen by the library
    for rg, width in ((2, 1), (4, 1), (4, 2), (1, 4)):
        c = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.5, kernelParam1=rg, kernelParam2=width, kernelParam3=p3,
                                    kernelId=3, bias=bias.cuda())
        assert c.shape == (m, n) and c.dtype == dtype
        assert_close(c, ogemm.linear_expected(w, b, 0.5, bias), RTOL, ATOL, "panel n=%d k=%d M=%d" % (n, k, m))
        c2 = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.5, kernelParam1=rg, kernelParam2=width,
                                     kernelParam3=p3, kernelId=3, bias=bias.cuda())
        assert torch.equal(c, c2)


@pytest.mark.parametrize("m", [100, 256, 385])
@pytest.mark.parametrize("scaled", [False, True])
def test_gemm_panel_kernel_soft_fp8(mlk, m, scaled):
    n, k = 640, 512
    codes = fp8_codes((n, k), 95)
    g = torch.Generator().manual_seed(96)
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float() if scaled else None
    b = randn((m, k), torch.bfloat16, 1.0, 97)
    for p3, rg, width in ((1, 2, 1), (2, 2, 1), (2, 4, 1), (1, 4, 2), (2, 4, 2)):
        c = mlk.gemm_layoutA_soft_fp8_wapper(pack_a(codes).cuda(), None if scale is None else scale.cuda(), b.cuda(),
                                             n, m, k, kernelParam1=rg, kernelParam2=width, kernelParam3=p3, kernelId=3)
        want = ogemm.softfp8_linear_expected(codes.numpy(), None if scale is None else scale.numpy(), b)
        assert_close(c, want, RTOL, ATOL, "panel fp8 M=%d slices=%d width=%d" % (m, p3, width))


@pytest.mark.parametrize("n,m,k,p1,p2,p3", [
    (5504, 1024, 256, 2, 1, 2),      # 43 row tiles x 8 token tiles of 128 x 128: one whole round of 256 panels + 88 sliced
    (5520, 1000, 512, 2, 1, 3),      # ragged rows and tokens, three uneven slices of four windows
    (16640, 1024, 256, 4, 2, 2),     # 65 row tiles x 4 token tiles of 256 x 256: 256 whole + 4 sliced
    (11008, 1024, 128, 4, 1, 2),     # one window: a single slice does all the work
    (5504, 384, 256, 2, 1, 2),       # three token tiles do not divide an XCD's CUs: every panel whole
    (2048, 1024, 256, 2, 1, 2),      # exactly one round: nothing left over, no slices
    (1024, 200, 512, 4, 1, 4),       # less than a round: every panel sliced, as with kernelId 3
    (5504, 1152, 256, 2, 1, 2),      # nine token tiles, one and a half rounds: whole, the fold would cost more
    (16640, 1100, 256, 4, 2, 2),     # the same with 256 x 256 panels and a ragged last token tile
    (7424, 640, 8192, 2, 1, 4),      # five token tiles, 290 panels of a long K: four slices save more than they cost
])
def test_gemm_panel_kernel_last_round_slices(mlk, n, m, k, p1, p2, p3):
    """kernelId 5: the panel kernel with K slices only on the panels left over after whole rounds of one panel per
    CU; bit-equal on a second run, and equal to the oracle like kernelId 3."""
    dtype = torch.bfloat16
    w = randn((n, k), dtype, 0.05, 191)
    b = randn((m, k), dtype, 1.0, 192)
    bias = randn((1, n), dtype, 1.0, 193)
    a = pack_a(w).cuda()
    c = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.5, kernelParam1=p1, kernelParam2=p2, kernelParam3=p3,
                                kernelId=5, bias=bias.cuda())
    assert c.shape == (m, n) and c.dtype == dtype
    assert_close(c, ogemm.linear_expected(w, b, 0.5, bias), RTOL, ATOL, "panel, last round sliced n=%d M=%d" % (n, m))
    c2 = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.5, kernelParam1=p1, kernelParam2=p2, kernelParam3=p3,
                                 kernelId=5, bias=bias.cuda())
    assert torch.equal(c, c2)


def test_gemm_panel_kernel_last_round_slices_soft_fp8(mlk):
    n, k, m = 5504, 512, 1024
    codes = fp8_codes((n, k), 195)
    g = torch.Generator().manual_seed(196)
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float()
    b = randn((m, k), torch.bfloat16, 1.0, 197)
    c = mlk.gemm_layoutA_soft_fp8_wapper(pack_a(codes).cuda(), scale.cuda(), b.cuda(), n, m, k, kernelParam1=2,
                                         kernelParam2=1, kernelParam3=2, kernelId=5)
    assert_close(c, ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), b), RTOL, ATOL, "panel fp8, last round sliced")


@pytest.mark.parametrize("fp8", [False, True])
def test_gemm_panel_kernel_band_and_chunk_mapping(mlk, fp8):
    """256 x 256 panels computed whole: the workgroup ids walk bands of eight groups of row tiles in chunks of four token
    tiles.  73 row tiles = ten groups (a band of eight and one of two, the last group with one row tile) and six token
    tiles (a chunk of four and one of two, the last tile ragged): every output element is checked."""
    n, k, m = 18560, 256, 1300
    b = randn((m, k), torch.bfloat16, 1.0, 292)
    if fp8:
        codes = fp8_codes((n, k), 293)
        g = torch.Generator().manual_seed(294)
        scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float()
        c = mlk.gemm_layoutA_soft_fp8_wapper(pack_a(codes).cuda(), scale.cuda(), b.cuda(), n, m, k, kernelParam1=4,
                                             kernelParam2=2, kernelParam3=1, kernelId=3)
        want = ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), b)
    else:
        w = randn((n, k), torch.bfloat16, 0.05, 291)
        bias = randn((1, n), torch.bfloat16, 1.0, 295)
        c = mlk.gemm_layoutA_wapper(pack_a(w).cuda(), b.cuda(), n, m, k, alpha=0.5, kernelParam1=4, kernelParam2=2,
                                    kernelParam3=1, kernelId=3, bias=bias.cuda())
        want = ogemm.linear_expected(w, b, 0.5, bias)
    assert c.shape == (m, n)
    assert_close(c, want, RTOL, ATOL, "band / chunk mapping fp8=%s" % fp8)


@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("m", [1, 64, 65, 257, 320, 321, 384, 385, 448, 449, 512])
def test_gemm_panel_kernel_columns_of_the_last_token_tile(mlk, kind, m):
    """256 x 256 panels computed whole: the last token tile multiplies 64, 128, 192 or 256 columns, whichever cover it; row
    groups past N in the last row tile."""
    n, k = 640, 256
    dtype = torch.float16 if kind == "fp16" else torch.bfloat16
    b = randn((m, k), dtype, 1.0, 301)
    params = dict(kernelParam1=4, kernelParam2=2, kernelParam3=1, kernelId=3)
    if kind == "fp8":
        codes = fp8_codes((n, k), 302)
        g = torch.Generator().manual_seed(303)
        scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float()
        c = mlk.gemm_layoutA_soft_fp8_wapper(pack_a(codes).cuda(), scale.cuda(), b.cuda(), n, m, k, **params)
        want = ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), b)
    else:
        w = randn((n, k), dtype, 0.05, 304)
        bias = randn((1, n), dtype, 1.0, 305)
        c = mlk.gemm_layoutA_wapper(pack_a(w).cuda(), b.cuda(), n, m, k, alpha=0.5, bias=bias.cuda(), **params)
        want = ogemm.linear_expected(w, b, 0.5, bias)
    assert c.shape == (m, n)
    assert_close(c, want, RTOL, ATOL, "last token tile %s M=%d" % (kind, m))


@pytest.mark.parametrize("kind,n,m,k,p1,p2,p3,whole", [
    ("fp8", 4608, 800, 7168, 2, 1, 4, False),    # 252 panels, but 35 of them on half of the XCDs: a second round for three
    ("fp8", 4608, 2112, 7168, 4, 1, 4, True),    # 256 x 128 panels, two per CU when whole
    ("fp8", 4608, 1856, 7168, 4, 1, 2, True),
    ("bf16", 4608, 800, 7168, 2, 1, 4, False),
    ("bf16", 11008, 2100, 4096, 4, 2, 2, True),
])
def test_gemm_panel_kernel_id5_slices_where_it_pays(mlk, kind, n, m, k, p1, p2, p3, whole):
    """Token tiles that do not divide an XCD's CUs, several rounds: which of the two orders of summation kernelId 5 takes (both
    measured) shows in the bits."""
    g = torch.Generator(device="cuda").manual_seed(411)
    b = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn((n, k), generator=g, device="cuda")
    if kind == "fp8":
        a = mlk.pack_layout_a((w * 16).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))
        scale = (torch.rand((n // 128, k // 128), generator=g, device="cuda") + 0.5) * (k ** -0.5 / 16)
    else:
        a, scale = mlk.pack_layout_a((w * k ** -0.5).to(torch.bfloat16)), None

    def run(kernel_id, slices):
        kw = dict(kernelParam1=p1, kernelParam2=p2, kernelParam3=slices, kernelId=kernel_id)
        if kind == "fp8":
            return mlk.gemm_layoutA_soft_fp8_wapper(a, scale, b, n, m, k, **kw)
        return mlk.gemm_layoutA_wapper(a, b, n, m, k, **kw)
    orders = {True: run(3, 1), False: run(3, p3)}
    assert not torch.equal(orders[True], orders[False]), "the two orders of summation cannot be told apart"
    assert_close(orders[True], orders[False].double().cpu().numpy(), RTOL, ATOL, "whole and sliced panels")
    assert torch.equal(run(5, p3), orders[whole])


def test_gemm_panel_kernel_id5_off_16_bytes_stays_sliced(mlk):
    """Soft-FP8 panels of 256 x 128, eleven token tiles: computed whole by the loop that loads straight into LDS, but sliced by the
    loop that loads through registers when the activations do not lie on 16 bytes."""
    n, m, k = 4608, 1281, 512
    codes = fp8_codes((n, k), 401)
    g = torch.Generator().manual_seed(402)
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float().cuda()
    a, b = pack_a(codes).cuda(), randn((m, k), torch.bfloat16, 1.0, 403).cuda()
    flat = torch.empty(m * k + 8, dtype=b.dtype, device="cuda")
    flat[1:1 + m * k] = b.view(-1)
    shifted = flat[1:1 + m * k].view(m, k)
    assert shifted.data_ptr() % 16 and shifted.is_contiguous()

    def run(x, kernel_id, slices):
        return mlk.gemm_layoutA_soft_fp8_wapper(a, scale, x, n, m, k, kernelParam1=4, kernelParam2=1, kernelParam3=slices,
                                                kernelId=kernel_id)
    whole, sliced = run(b, 3, 1), run(b, 3, 2)
    assert not torch.equal(whole, sliced), "the two orders of summation cannot be told apart"
    assert torch.equal(run(b, 5, 2), whole)
    assert torch.equal(run(shifted, 5, 2), sliced)


def test_gemm_panel_kernel_is_the_wide_default(mlk):
    """Above 64 tokens unscanned shapes run the eight-wave panels; the rule of thumb for shapes that the library has no plan for names the
    older panel kernel, which computes the same, but for a K that is no multiple of 128, which keeps the row-shared kernel and which
    the panel kernel refuses when asked for by id."""
    from muxi_native_layout_kernels_amd import arg_selector, ops
    # 4224 rows: a weight shape that no packaged table holds
    assert arg_selector.selector("layoutA_gemm").get_args((4224, 300, 1024))[0] == 3
    assert arg_selector.selector("layoutA_soft_fp8_gemm").get_args((4224, 300, 1024))[0] == 3
    assert arg_selector.selector("layoutA_gemm").get_args((4224, 300, 1088))[0] == 2
    assert arg_selector.selector("layout_gemm").get_args((4224, 304, 1024))[0] == 2       # native operands
    n, k, m = 4224, 1024, 300
    assert ops._gemm_args("layoutA_gemm", n, m, k, 1)[0] == 8 and ops._gemm_args("layoutA_soft_fp8_gemm", n, m, k, 2)[0] == 8
    w = randn((n, k), torch.bfloat16, 0.02, 98)
    b = randn((m, k), torch.bfloat16, 1.0, 99)
    c = mlk.gemm_layoutA_linear(pack_a(w).cuda(), b.cuda())
    assert_close(c, ogemm.linear_expected(w, b), RTOL, ATOL, "panel default")
    _, p1, p2, p3 = arg_selector.selector("layoutA_gemm").get_args((n, m, k))
    c = mlk.gemm_layoutA_wapper(pack_a(w).cuda(), b.cuda(), n, m, k, kernelParam1=p1, kernelParam2=p2, kernelParam3=p3, kernelId=3)
    assert_close(c, ogemm.linear_expected(w, b), RTOL, ATOL, "kernel 3")
    with pytest.raises(RuntimeError, match="K % 128"):
        mlk.gemm_layoutA_wapper(pack_a(w[:, :960].contiguous()).cuda(), b[:, :960].contiguous().cuda(), n, m, 960,
                                kernelParam1=1, kernelParam2=1, kernelParam3=1, kernelId=3)
    with pytest.raises(RuntimeError, match="row-major"):
        mlk.gemm_layoutABC_wapper(pack_a(w).cuda(), mlk.layoutB(b[:288].contiguous().cuda()), n, 288, k, kernelParam1=1,
                                  kernelParam2=1, kernelParam3=1, kernelId=3)


@pytest.mark.parametrize("n", [16 * 300, 16 * 384, 16 * 688, 16 * 768, 16 * 1000])
@pytest.mark.parametrize("m", [1, 7, 16, 32, 40, 48, 57, 64])
def test_gemm_balanced_rows_kernel(mlk, n, m):
    """kernelId 4: one workgroup per CU, the row groups dealt out evenly (one to four per workgroup, uneven
    deals included).  From three token blocks on the activations of a k window are shared through LDS; shapes
    it does not take run as kernel 1."""
    k = 256
    w = randn((n, k), torch.bfloat16, 0.05, 71)
    b = randn((m, k), torch.bfloat16, 1.0, 72)
    bias = randn((1, n), torch.bfloat16, 1.0, 73)
    a = pack_a(w).cuda()
    for p2 in (1, 2, 8):
        c = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=2.0, kernelParam1=1, kernelParam2=p2, kernelParam3=1,
                                    kernelId=4, bias=bias.cuda())
        assert_close(c, ogemm.linear_expected(w, b, 2.0, bias), RTOL, ATOL, "balanced rows n=%d m=%d" % (n, m))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k", [192, 1024, 1152, 4096])
@pytest.mark.parametrize("m", [20, 32, 33, 48, 50, 64])
def test_gemm_balanced_rows_kernel_shared_windows(mlk, dtype, k, m):
    """kernelId 4 at two (eight waves), three and four token blocks over short and long K: K = 192 (six k tiles, no whole
    windows: the plain wave kernel takes it), 1024 and 4096 (the unrolled loop with its lead-in), 1152 (36 k
    tiles: nine windows, an odd tail), on 688 row groups (three and two per workgroup on 256 CUs); twice, and the
    two runs must agree bit for bit."""
    n = 16 * 688
    w = randn((n, k), dtype, 0.02, 74)
    b = randn((m, k), dtype, 1.0, 75)
    bias = randn((1, n), dtype, 1.0, 76)
    a = pack_a(w).cuda()
    for p2 in (8, 4, 2):
        c = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.5, kernelParam1=1, kernelParam2=p2, kernelParam3=1,
                                    kernelId=4, bias=bias.cuda())
        assert_close(c, ogemm.linear_expected(w, b, 0.5, bias), RTOL, ATOL, "balanced shared k=%d m=%d p2=%d" % (k, m, p2))
        c2 = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, alpha=0.5, kernelParam1=1, kernelParam2=p2, kernelParam3=1,
                                     kernelId=4, bias=bias.cuda())
        assert torch.equal(c, c2)


@pytest.mark.parametrize("n", [11008, 12288, 4736, 18432, 22016, 28672, 32768])
@pytest.mark.parametrize("m", [20, 32, 40, 64])
def test_gemm_balanced_rows_kernel_soft_fp8(mlk, n, m):
    """kernelId 4 with soft-FP8 weights from two token blocks on (eight waves share staged windows): two to eight
    row groups per workgroup (on 256 CUs: three or two for 11008 rows, five or four for 18432, six or five for 22016,
    seven for 28672, eight for 32768) that start anywhere, so they straddle two 128-row blocks of scales; every block
    has its own random scale.  With two waves at two token blocks the id means kernel 1."""
    k = 1024
    codes = fp8_codes((n, k), 91)
    g = torch.Generator().manual_seed(92)
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float()
    b = randn((m, k), torch.bfloat16, 1.0, 93)
    a = pack_a(codes).cuda()
    want = ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), b)
    for p2 in (8, 4, 2):
        c = mlk.gemm_layoutA_soft_fp8_wapper(a, scale.cuda(), b.cuda(), n, m, k, kernelParam1=1, kernelParam2=p2,
                                             kernelParam3=1, kernelId=4)
        assert_close(c, want, RTOL, ATOL, "balanced fp8 n=%d m=%d p2=%d" % (n, m, p2))


def test_gemm_balanced_rows_fallbacks(mlk):
    """Soft-FP8 weights at one token block and native operands are outside kernel 4: the id then means kernel 1."""
    n, k, m = 16 * 300, 512, 16
    codes = fp8_codes((n - n % 128, k), 81)
    n8 = codes.shape[0]
    g = torch.Generator().manual_seed(82)
    scale = (torch.rand((n8 // 128, k // 128), generator=g) * 0.02 + 0.001).float()
    b = randn((m, k), torch.bfloat16, 1.0, 83)
    c = mlk.gemm_layoutA_soft_fp8_wapper(pack_a(codes).cuda(), scale.cuda(), b.cuda(), n8, m, k, kernelParam1=1,
                                         kernelParam2=4, kernelParam3=1, kernelId=4)
    assert_close(c, ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), b), RTOL, ATOL, "kernel 4 on fp8")
    w = randn((n, k), torch.float16, 0.05, 84)
    bh = randn((m, k), torch.float16, 1.0, 85)
    a = pack_a(w).cuda()
    c_rm = mlk.gemm_layoutAB_ContinuousC_wapper(a, mlk.layoutB(bh.cuda()), n, m, k, kernelParam1=1, kernelParam2=4,
                                                kernelParam3=1, kernelId=4)
    assert_close(c_rm, ogemm.linear_expected(w, bh), RTOL, ATOL, "kernel 4 on native B")


def test_gemm_special_cases(mlk):
    n = k = 256
    eye = torch.eye(n, dtype=torch.float16)
    b = randn((32, k), torch.float16, 1.0, 6)
    assert torch.equal(mlk.gemm_layoutA(pack_a(eye).cuda(), b.cuda()).cpu(), b)
    bias = randn((1, n), torch.float16, 1.0, 7)
    c0 = mlk.gemm_layoutA(pack_a(eye).cuda(), b.cuda(), alpha=0.0, bias=bias.cuda())
    assert torch.equal(c0.cpu(), bias.expand(32, n))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m", [32, 48, 64])
def test_native_chain_balanced_rows_kernel(mlk, dtype, m):
    """kernelId 4 on layout-B activations from two token blocks on (eight and four waves share staged windows):
    layout-C output + reLayoutC equals the row-major output bit for bit, the layout-C tensor equals the oracle's
    relayout of it, and both match the oracle; 688 and 512 row groups (three / two and two per workgroup)."""
    for n, k in ((16 * 688, 1024), (8192, 512)):
        w = randn((n, k), dtype, 0.02, 18)
        b = randn((m, k), dtype, 1.0, 19)
        a, b_nat = pack_a(w).cuda(), mlk.layoutB(b.cuda())
        for p2 in (8, 4):
            c_rm = mlk.gemm_layoutAB_ContinuousC_wapper(a, b_nat, n, m, k, kernelParam1=1, kernelParam2=p2, kernelParam3=1,
                                                        kernelId=4)
            c_nat = mlk.gemm_layoutABC_wapper(a, b_nat, n, m, k, kernelParam1=1, kernelParam2=p2, kernelParam3=1,
                                              kernelId=4)
            assert torch.equal(mlk.reLayoutC(c_nat), c_rm)
            assert torch.equal(c_nat.cpu().view(torch.int16), ogemm.layout_c_of(c_rm.cpu()).view(torch.int16))
            assert_close(c_rm, ogemm.linear_expected(w, b), RTOL, ATOL, "native balanced n=%d m=%d p2=%d" % (n, m, p2))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_native_chain_bit_exact(mlk, dtype):
    """layoutB -> gemm_layoutABC -> reLayoutC equals gemm_layoutAB_ContinuousC bit for bit (same launch
    parameters, hence same accumulation order), and both match the oracle."""
    n, k, m = 1024, 2048, 32
    w = randn((n, k), dtype, 0.02, 8)
    b = randn((m, k), dtype, 1.0, 9)
    a = pack_a(w).cuda()
    b_nat = mlk.layoutB(b.cuda())
    assert np.array_equal(bits(b_nat.cpu()), layouts.pack_layout_b(bits(b)))
    for (p1, p2, p3) in [(1, 4, 1), (2, 2, 2)]:
        c_nat = mlk.gemm_layoutABC_wapper(a, b_nat, n, m, k, kernelParam1=p1, kernelParam2=p2, kernelParam3=p3)
        assert c_nat.shape == (n // 32, m // 16, 4, 16, 8)
        c_rm = mlk.gemm_layoutAB_ContinuousC_wapper(a, b_nat, n, m, k, kernelParam1=p1, kernelParam2=p2,
                                                    kernelParam3=p3)
        assert torch.equal(mlk.reLayoutC(c_nat), c_rm)
        # layout-C of the result is layout-B of the row-major result
        assert np.array_equal(bits(c_nat.cpu()), layouts.pack_layout_c(bits(c_rm.cpu())))
        c_a = mlk.gemm_layoutA_wapper(a, b.cuda(), n, m, k, kernelParam1=p1, kernelParam2=p2, kernelParam3=p3)
        assert torch.equal(c_a, c_rm)
        assert_close(c_rm, ogemm.linear_expected(w, b), RTOL, ATOL, "native chain")


def test_native_chain_config(mlk):
    n = k = 8192
    m = 32
    w = randn((n, k), torch.bfloat16, 0.02, 2025)
    b = randn((m, k), torch.bfloat16, 1.0, 2026)
    a = pack_a(w).cuda()
    b_nat = mlk.layoutB(b.cuda())
    c_nat = mlk.gemm_layoutABC(a, b_nat)
    c = mlk.reLayoutC(c_nat)
    assert_close(c, ogemm.linear_expected(w, b), RTOL, ATOL, "ABC 8192")
    # the native output is layout-C of the row-major one (oracle permutation, bit for bit)
    assert torch.equal(c_nat.cpu(), ogemm.layout_c_of(c.cpu()))
    # chain a second product on the native output: C1 is the layout-B operand of the next layer
    w2 = randn((256, n), torch.bfloat16, 0.02, 2027)
    c2 = mlk.reLayoutC(mlk.gemm_layoutABC(pack_a(w2).cuda(), c_nat))
    assert_close(c2, ogemm.linear_expected(w2, c.cpu()), RTOL, ATOL, "chained")


@pytest.mark.parametrize("n,k,kid", [(8704, 512, 1), (9728, 256, 1), (640, 1152, 1)])
def test_native_chain_planned(mlk, n, k, kid):
    """Sixteen tokens in layout B on weight shapes that no table holds: launch parameters of a kernel that takes them (the first of these shapes
    has kernel 4 with row-major activations), both outputs."""
    from muxi_native_layout_kernels_amd import ops
    m = 16
    w, x = randn((n, k), torch.bfloat16, k ** -0.5, 23), randn((m, k), torch.bfloat16, 1.0, 24)
    assert ops._gemm_args("layout_gemm", n, m, k, 1, 1)[0] == kid
    a, xb = pack_a(w).cuda(), mlk.layoutB(x.cuda())
    c = mlk.gemm_layoutAB_ContinuousC(a, xb)
    assert_close(c, ogemm.linear_expected(w, x), RTOL, ATOL, "planned")
    assert torch.equal(mlk.reLayoutC(mlk.gemm_layoutABC(a, xb)), c)


@pytest.mark.parametrize("m", [1, 4, 16, 33])
@pytest.mark.parametrize("scaled", [False, True])
def test_gemm_soft_fp8(mlk, m, scaled):
    n, k = 1024, 2048
    codes = fp8_codes((n, k), 2025)
    b = randn((m, k), torch.bfloat16, 1.0, 2026)
    g = torch.Generator().manual_seed(3)
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float() if scaled else \
        torch.ones((n // 128, k // 128))
    c = mlk.gemm_layoutA_soft_fp8(pack_a(codes).cuda(), scale.cuda(), b.cuda())
    assert_close(c, ogemm.softfp8_linear_expected(codes.numpy(), scale.numpy(), b), RTOL, ATOL, "soft-fp8 gemm")
    c2 = mlk.gemm_layoutA_linear(pack_a(codes).cuda(), b.cuda(), scale_matrix=scale.cuda())
    assert torch.equal(c, c2)


@pytest.mark.parametrize("m", [4, 16])
@pytest.mark.parametrize("scaled", [False, True])
def test_gemm_soft_fp8_config(mlk, m, scaled):
    """The third benchmark configuration at its full shape through the shipped table rows, with unit scales and
    with an arbitrary fp32 scale per 128 x 128 block (the general widening path, which is what the bench times)."""
    n, k = 28672, 8192
    codes = fp8_codes((n, k), 2025)
    b = randn((m, k), torch.bfloat16, 1.0, 2026)
    if scaled:
        g = torch.Generator().manual_seed(2027)
        scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 0.001).float()
    else:
        scale = torch.ones((n // 128, k // 128))
    c = mlk.gemm_layoutA_soft_fp8(pack_a(codes).cuda(), scale.cuda(), b.cuda())
    # float64 product in row chunks to bound host memory
    from oracle import softfp8
    got = c.cpu()
    for r0 in range(0, n, 4096):
        wchunk = softfp8.dequant_weight_f32(codes[r0:r0 + 4096].numpy(), scale[r0 // 128:(r0 + 4096) // 128].numpy() if scaled else None)
        assert_close(got[:, r0:r0 + 4096], ogemm.linear_expected(wchunk, b), RTOL, ATOL, "soft-fp8 config")


def test_gemm_errors(mlk):
    a = torch.zeros(8, 16, 16, 8, dtype=torch.bfloat16, device="cuda")   # 128 x 128
    b = torch.zeros(16, 128, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="same k"):
        mlk.gemm_layoutA(a, torch.zeros(16, 256, dtype=torch.bfloat16, device="cuda"))
    with pytest.raises(RuntimeError, match="2D"):
        mlk.gemm_layoutA(a, b.view(1, 16, 128))
    with pytest.raises(RuntimeError, match="m % 128"):
        mlk.gemm_layoutA(torch.zeros(4, 16, 16, 8, dtype=torch.bfloat16, device="cuda"), b)
    with pytest.raises(RuntimeError, match="5D"):
        mlk.gemm_layoutABC(a, b)
    with pytest.raises(RuntimeError, match="data type"):
        mlk.gemm_layoutA(a, b.half())
    assert mlk.gemm_layoutA(a, b).shape == (16, 128)


def test_gemm_repeated_calls_take_the_launch_plan_and_keep_the_checks(mlk):
    """Second calls with the same shapes run from the launch plan: same results as the first, K-split workspace
    included, and the per-call checks (contiguity, beta) still raise."""
    n, k, m = 1024, 2048, 24
    w = randn((n, k), torch.float16, 0.02, 51)
    a = pack_a(w).cuda()
    b1, b2 = randn((m, k), torch.float16, 1.0, 52).cuda(), randn((m, k), torch.float16, 1.0, 53).cuda()
    c1 = mlk.gemm_layoutA(a, b1)
    c2 = mlk.gemm_layoutA(a, b2)                                  # planned
    c1b = mlk.gemm_layoutA(a, b1)                                 # planned
    assert torch.equal(c1, c1b)
    assert_close(c2, ogemm.linear_expected(w, b2.cpu()), RTOL, ATOL, "planned call")
    bn = mlk.layoutB(randn((32, k), torch.float16, 1.0, 54).cuda())
    for fn in (mlk.gemm_layoutABC, mlk.gemm_layoutAB_ContinuousC):
        assert torch.equal(fn(a, bn), fn(a, bn))
    assert torch.equal(mlk.reLayoutC(mlk.gemm_layoutABC(a, bn)), mlk.gemm_layoutAB_ContinuousC(a, bn))
    with pytest.raises(RuntimeError, match="beta"):
        mlk.gemm_layoutA(a, b1, beta=2)
    wide = torch.zeros((m, 2 * k), dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError, match="contiguous"):
        mlk.gemm_layoutA(a, wide[:, ::2])


@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("p1,p2", [(p1, p2) for p1 in (2, 4) for p2 in (1, 2, 3, 4)])
@pytest.mark.parametrize("n,m,k,p3,native", [
    (128, 1, 128, 1, False),           # the smallest call: one panel, four slabs
    (272, 65, 384, 1, False),          # rows that end inside a panel, a token tile of one token
    (400, 130, 640, 3, False),         # ten k windows in three slices
    (528, 257, 1152, 64, False),       # k windows dealt to as many workgroups: runs that end inside a panel
    (1040, 192, 2048, 16, False),      # two windows per slice
    (416, 80, 384, 1, True),           # the same remainders in native layouts: whole,
    (544, 272, 1152, 64, True),        # dealt,
    (416, 144, 640, 3, True),          # sliced, the last token tile narrower than the others
    (1056, 192, 2048, 16, True),
    (160, 48, 512, 4, True),           # slots of 48 tokens
])
def test_gemm_eight_wave_panels(mlk, kind, p1, p2, n, m, k, p3, native):
    """kernelId 8 in every panel shape: remainders of rows, tokens and k, whole, sliced and dealt; row-major operands against the
    oracle, layout-B activations and layout-C output against the row-major run, whose sums have the same order."""
    dtype = torch.float16 if kind == "fp16" else torch.bfloat16
    x = randn((m, k), dtype, 1.0, 31)
    bias = randn((1, n), dtype, 1.0, 32)
    kw = dict(alpha=0.5, bias=bias.cuda(), kernelParam1=p1, kernelParam2=p2, kernelParam3=p3, kernelId=8)
    if kind == "fp8":
        w = fp8_codes((n, k), 33)
        scale = (torch.rand(((n + 127) // 128, k // 128), generator=torch.Generator().manual_seed(34)) * 0.02 + 0.001).float()
        a, scale_dev = pack_a(w).cuda(), scale.cuda()
        c = mlk.gemm_layoutA_soft_fp8_wapper(a, scale_dev, x.cuda(), n, m, k, **kw)
        want = ogemm.softfp8_linear_expected(w, scale, x, 0.5, bias)
        assert_close(c, want, RTOL, ATOL, "soft-FP8 panels")
        if native:                     # no Python entry point takes this pair, the C one does
            for c_mode, row_major in ((0, lambda c: c), (1, mlk.reLayoutC)):
                got = ops._gemm_call(a, scale_dev, mlk.layoutB(x.cuda()), n, m, k, 0.5, 0, kw["bias"], 1, c_mode, 8, p1, p2, p3, "gemm")
                assert torch.equal(row_major(got), c)
        return
    w = randn((n, k), dtype, k ** -0.5, 33)
    a = pack_a(w).cuda()
    c = mlk.gemm_layoutA_wapper(a, x.cuda(), n, m, k, **kw)
    assert_close(c, ogemm.linear_expected(w, x, 0.5, bias), RTOL, ATOL, "panels")
    if native:
        xb = mlk.layoutB(x.cuda())
        assert torch.equal(mlk.gemm_layoutAB_ContinuousC_wapper(a, xb, n, m, k, **kw), c)
        assert torch.equal(mlk.reLayoutC(mlk.gemm_layoutABC_wapper(a, xb, n, m, k, **kw)), c)


@pytest.mark.parametrize("kind", ["fp16", "fp8"])
@pytest.mark.parametrize("p1,p2", [(p1, p2) for p1 in (2, 4) for p2 in (1, 2, 3, 4)])
@pytest.mark.parametrize("k,p3", [(128, 2), (256, 1), (384, 2), (640, 1), (768, 5), (896, 1), (1152, 1), (1664, 3), (1920, 1)])
def test_gemm_eight_wave_rings(mlk, kind, p1, p2, k, p3):
    """kernelId 8 on full panels: K, and slices of it, shorter than the rings of every shape (two to five pairs of k32 slabs), as long, and
    longer by every remainder.  The weights of neighbouring slabs differ in scale, so that a slab multiplied twice or by its
    neighbour's tokens shows; whole numbers, so that sums of up to 2^24 have one value in any order.  Activations row-major and in layout B."""
    n, m = 64 * p1, 64 * p2
    g = torch.Generator().manual_seed(36)
    x = torch.randint(-3, 4, (m, k), generator=g).to(torch.float16 if kind == "fp16" else torch.bfloat16)
    w = torch.randint(-2, 3, (n, k), generator=g) * (1 + torch.arange(k) // 32 % 3)
    want = x.double() @ w.double().t()
    kw = dict(kernelParam1=p1, kernelParam2=p2, kernelParam3=p3, kernelId=8)
    if kind == "fp8":
        # one scale per 128 x 128 block, powers of two: widened exactly
        scale = torch.exp2(torch.randint(-2, 3, ((n + 127) // 128, k // 128), generator=g).float())
        want = x.double() @ (w * scale.repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)).double().t()
        a = pack_a(w.float().to(torch.float8_e4m3fn).view(torch.uint8)).cuda()
        scale = scale.cuda()
        c = mlk.gemm_layoutA_soft_fp8_wapper(a, scale, x.cuda(), n, m, k, **kw)
    else:
        a, scale = pack_a(w.to(x.dtype)).cuda(), None
        c = mlk.gemm_layoutA_wapper(a, x.cuda(), n, m, k, **kw)
    want = want.float().to(x.dtype)
    assert torch.equal(c.cpu(), want)
    c = ops._gemm_call(a, scale, mlk.layoutB(x.cuda()), n, m, k, 1, 0, None, 1, 0, 8, p1, p2, p3, "gemm")
    assert torch.equal(c.cpu(), want)


@pytest.mark.parametrize("kind,native", [("bf16", False), ("bf16", True), ("fp8", False)])
@pytest.mark.parametrize("n,m,k,p1,p2,p3,first", [
    (384, 1488, 256, 2, 2, 1, True),       # three row tiles, twelve token tiles, the last one short
    (1040, 1600, 384, 2, 4, 2, True),      # nine row tiles, the last one ragged, in slices
    (400, 2832, 256, 4, 1, 3, True),       # two row tiles, 45 token tiles, more slices than windows of some
    (640, 1504, 640, 2, 3, 1, True),
    (640, 144, 640, 2, 3, 1, False),       # one token tile: either order is the same
    (128, 1040, 128, 2, 1, 2, False),      # one row tile
])
def test_gemm_eight_wave_row_tiles_first(mlk, kind, native, n, m, k, p1, p2, p3, first):
    """One line of panels with more activations than weights: the row tiles of a token tile side by side.  Whole numbers, one value in
    any order of the sums."""
    weights, tokens = n * (1 if kind == "fp8" else 2), 2 * m
    row_tiles, token_tiles = -(-n // (64 * p1)), -(-m // (64 * p2))
    assert row_tiles * token_tiles <= 256                      # one line
    # the rule of p8_rows_first() in csrc/mlk_panel.hip
    assert first == (tokens > weights and tokens + weights * min(8, token_tiles) < weights + tokens * min(8, row_tiles))
    g = torch.Generator().manual_seed(37)
    x = torch.randint(-3, 4, (m, k), generator=g).to(torch.bfloat16)
    w = torch.randint(-2, 3, (n, k), generator=g)
    want = (x.double() @ w.double().t()).float().to(x.dtype)
    kw = dict(kernelParam1=p1, kernelParam2=p2, kernelParam3=p3, kernelId=8)
    if kind == "fp8":
        scale = torch.ones((n + 127) // 128, k // 128)
        a = pack_a(w.float().to(torch.float8_e4m3fn).view(torch.uint8)).cuda()
        c = mlk.gemm_layoutA_soft_fp8_wapper(a, scale.cuda(), x.cuda(), n, m, k, **kw)
    elif native:
        c = mlk.gemm_layoutAB_ContinuousC_wapper(pack_a(w.to(x.dtype)).cuda(), mlk.layoutB(x.cuda()), n, m, k, **kw)
    else:
        c = mlk.gemm_layoutA_wapper(pack_a(w.to(x.dtype)).cuda(), x.cuda(), n, m, k, **kw)
    assert torch.equal(c.cpu(), want)


@pytest.mark.parametrize("kind", ["bf16", "fp8"])
@pytest.mark.parametrize("n,m,k,p1,p2", [(4352, 4100, 256, 4, 4), (2304, 1984, 256, 2, 1), (8448, 1000, 128, 2, 2)])
def test_gemm_eight_wave_panels_several_rounds(mlk, kind, n, m, k, p1, p2):
    """More panels than CUs: the bands' order of the panels, and the panels left over after whole rounds dealt or sliced."""
    g = torch.Generator(device="cuda").manual_seed(35)
    w = torch.randn((n, k), generator=g, device="cuda") * k ** -0.5
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    kw = dict(kernelParam1=p1, kernelParam2=p2, kernelId=8)
    if kind == "fp8":
        codes = (w * 256).clamp_(-448, 448).to(torch.float8_e4m3fn)
        # powers of two: the widened weight is the bf16 that the reference multiplies
        scale = torch.exp2(torch.randint(-9, -6, (n // 128, k // 128), generator=g, device="cuda").float())
        a, w = mlk.pack_layout_a(codes.view(torch.uint8)), codes.float() * scale.repeat_interleave(128, 0).repeat_interleave(128, 1)
    else:
        a, w = mlk.pack_layout_a(w.to(torch.bfloat16)), w.to(torch.bfloat16).float()
    want = (x.float() @ w.t()).double().cpu().numpy()
    for p3 in (1, 2, 64):
        if kind == "fp8":
            c = mlk.gemm_layoutA_soft_fp8_wapper(a, scale, x, n, m, k, kernelParam3=p3, **kw)
        else:
            c = mlk.gemm_layoutA_wapper(a, x, n, m, k, kernelParam3=p3, **kw)
        assert_close(c, want, RTOL, ATOL, "several rounds, p3 = %d" % p3)


@pytest.mark.parametrize("kid", [3, 5])
@pytest.mark.parametrize("n,m,k,p3", [
    (256, 256, 4096, 63), (256, 256, 4096, 64),     # one panel, as many k windows as slices
    (512, 300, 8192, 64),                           # four panels, two windows a slice
    (256, 256, 1024, 64),                           # fewer windows than slices
])
def test_gemm_panel_ids_3_and_5_take_64_slices(mlk, kid, n, m, k, p3):
    """p3 = 64 is a slice count of kernel ids 3 and 5 like any other (kernel id 8 gives it a meaning of its own): panels of 256 x 256
    run on the workspace that mlk_gemm_workspace_bytes() answers, and nothing behind it is written."""
    from muxi_native_layout_kernels_amd import _lib
    from muxi_native_layout_kernels_amd.ops import _stream
    lib = _lib.load()
    w, x = randn((n, k), torch.bfloat16, k ** -0.5, 41), randn((m, k), torch.bfloat16, 1.0, 42)
    a, b, c = pack_a(w).cuda(), x.cuda(), torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    size = lib.mlk_gemm_workspace_bytes(m, n, 4, p3)
    ws = torch.full((size + 4096,), 0xAB, dtype=torch.uint8, device="cuda")
    ws[:lib.mlk_gemm_counter_bytes()].zero_()
    _lib.check(lib.mlk_gemm_layout_a(a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, 1, 1, 0, 0, 1.0, None, None, kid, 4, 2, p3,
                                     ws.data_ptr(), size, _stream()), "gemm")
    assert_close(c, ogemm.linear_expected(w, x), RTOL, ATOL, "p3 = %d" % p3)
    assert (ws[size:] == 0xAB).all()


@pytest.mark.parametrize("m,p1,p2,p3", [(1, 2, 1, 3), (16, 2, 1, 6), (33, 2, 1, 6), (48, 4, 1, 5), (40, 2, 2, 4), (64, 2, 1, 7)])
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_gemm_eight_wave_slices_fit_the_workspace_of_the_other_ids(mlk, kind, m, p1, p2, p3):
    """Up to 64 tokens the K slices of kernel id 8 run on what mlk_gemm_workspace_bytes() answers, as those of every row of the
    tables do, and write nothing behind what mlk_gemm_panel_workspace_bytes() says."""
    from muxi_native_layout_kernels_amd import _lib
    from muxi_native_layout_kernels_amd.ops import _stream
    lib = _lib.load()
    n, k = 512, 1152
    x = randn((m, k), torch.bfloat16, 1.0, 46)
    if kind == "fp8":
        w = fp8_codes((n, k), 47)
        scale = (torch.rand((n // 128, k // 128), generator=torch.Generator().manual_seed(48)) * 0.02 + 0.001).float()
        want, sc = ogemm.softfp8_linear_expected(w.numpy(), scale.numpy(), x), scale.cuda()
    else:
        w = randn((n, k), torch.bfloat16, k ** -0.5, 47)
        want, sc = ogemm.linear_expected(w, x), None
    a, b, c = pack_a(w).cuda(), x.cuda(), torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    size, need = lib.mlk_gemm_workspace_bytes(m, n, p1, p3), lib.mlk_gemm_panel_workspace_bytes(m, n, k, p1, p2, p3)
    assert need <= size
    ws = torch.full((size + 4096,), 0xAB, dtype=torch.uint8, device="cuda")
    _lib.check(lib.mlk_gemm_layout_a(a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, 2 if kind == "fp8" else 1, 1, 0, 0, 1.0, None,
                                     None if sc is None else sc.data_ptr(), 8, p1, p2, p3, ws.data_ptr(), size, _stream()), "gemm")
    assert_close(c, want, RTOL, ATOL, "m = %d" % m)
    assert (ws[need:] == 0xAB).all()


@pytest.mark.parametrize("kid,p3", [(3, 1), (3, 2), (5, 2)])
@pytest.mark.parametrize("kind", ["fp16", "fp8"])
@pytest.mark.parametrize("n,m,k", [(256, 300, 512), (2304, 520, 256)])
def test_gemm_panel_ids_3_and_5_off_16_bytes(mlk, n, m, k, kind, kid, p3):
    """Weights, activations or both off 16 bytes: panels of 128 tokens through registers, also where 256 were asked for."""
    dtype = torch.float16 if kind == "fp16" else torch.bfloat16
    x = randn((m, k), dtype, 1.0, 43)
    if kind == "fp8":
        w = fp8_codes((n, k), 44)
        scale = (torch.rand((n // 128, k // 128), generator=torch.Generator().manual_seed(45)) * 0.02 + 0.001).float()
        want = ogemm.softfp8_linear_expected(w.numpy(), scale.numpy(), x)
    else:
        w = randn((n, k), dtype, k ** -0.5, 44)
        want = ogemm.linear_expected(w, x)

    def shifted(t):
        at = 1 if t.element_size() == 2 else 8
        flat = torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")
        flat[at:at + t.numel()] = t.reshape(-1)
        out = flat[at:at + t.numel()].view(t.shape)
        assert out.data_ptr() % 16 and out.is_contiguous()
        return out
    a, b = pack_a(w).cuda(), x.cuda()
    kw = dict(kernelParam1=4, kernelParam2=2, kernelParam3=p3, kernelId=kid)
    for aa, bb in ((a, shifted(b)), (shifted(a), b), (shifted(a), shifted(b))):
        c = mlk.gemm_layoutA_soft_fp8_wapper(aa, scale.cuda(), bb, n, m, k, **kw) if kind == "fp8" else \
            mlk.gemm_layoutA_wapper(aa, bb, n, m, k, **kw)
        assert_close(c, want, RTOL, ATOL, "off 16 bytes")


@pytest.mark.parametrize("native", [False, True])
def test_gemm_eight_wave_panels_off_16_bytes(mlk, native):
    """Operands that do not lie on 16 bytes run the kernels that load through registers."""
    n, m, k = 640, 80, 512
    w, x = randn((n, k), torch.bfloat16, 0.05, 36), randn((m, k), torch.bfloat16, 1.0, 37)
    a = pack_a(w).cuda()
    b = pack_b(x).cuda() if native else x.cuda()
    flat = torch.empty(m * k + 8, dtype=b.dtype, device="cuda")
    flat[1:1 + m * k] = b.view(-1)
    shifted = flat[1:1 + m * k].view(b.shape)
    assert shifted.data_ptr() % 16
    c = mlk.gemm_layoutAB_ContinuousC(a, shifted) if native else mlk.gemm_layoutA(a, shifted)
    assert_close(c, ogemm.linear_expected(w, x), RTOL, ATOL, "off 16 bytes")


@pytest.mark.parametrize("native", [0, 1, 2])
@pytest.mark.parametrize("n,m,k,split", [(512, 112, 8192, True), (512, 32, 8192, True), (4352, 64, 512, False), (8448, 1040, 256, False)])
def test_gemm_eight_wave_panels_off_16_bytes_fill_the_chip(mlk, n, m, k, split, native):
    """Off 16 bytes a call for the eight-wave panels gets launch parameters for the kernels that take it: K slices where it has few
    rows (they write partial sums into the workspace), row-major, with layout-B activations and with layout-C output too."""
    from muxi_native_layout_kernels_amd import _lib
    from muxi_native_layout_kernels_amd.ops import _stream
    lib = _lib.load()
    w, x = randn((n, k), torch.bfloat16, k ** -0.5, 49), randn((m, k), torch.bfloat16, 1.0, 50)
    a, b = pack_a(w).cuda(), pack_b(x).cuda() if native else x.cuda()
    flat = torch.empty(m * k + 8, dtype=b.dtype, device="cuda")
    flat[1:1 + m * k] = b.view(-1)
    c = torch.empty((n // 32, m // 16, 4, 16, 8) if native == 2 else (m, n), dtype=b.dtype, device="cuda")
    counters = lib.mlk_gemm_counter_bytes()
    for size in (counters + (4 << 20), 0):
        ws = torch.full((size + 4096,), 0xAB, dtype=torch.uint8, device="cuda")
        ws[:counters if size else 0].zero_()
        _lib.check(lib.mlk_gemm_layout_a(a.data_ptr(), flat.data_ptr() + 2, c.data_ptr(), m, n, k, 1, 1, int(native > 0), int(native == 2),
                                         1.0, None, None, 8, 4, 2, 1, ws.data_ptr() if size else None, size, _stream()), "gemm")
        assert_close(mlk.reLayoutC(c) if native == 2 else c, ogemm.linear_expected(w, x), RTOL, ATOL, "off 16 bytes")
        assert bool((ws[counters:size] != 0xAB).any()) == (split and size > 0)
        assert (ws[size:] == 0xAB).all() and not ws[:counters if size else 0].any()


@pytest.mark.parametrize("native", [False, True])
@pytest.mark.parametrize("n,m,k,dealt", [(512, 112, 4096, False), (512, 48, 4096, False), (2304, 1984, 256, True)])
def test_gemm_without_room_for_scratch_runs_in_one_slice(mlk, monkeypatch, n, m, k, dealt, native):
    """A card without room for the scratch of K slices or dealt panels: the call runs whole panels (or one slice) on its first pass and from
    the launch plan, and takes the slices again once there is room."""
    from muxi_native_layout_kernels_amd import ops
    w, x = randn((n, k), torch.bfloat16, k ** -0.5, 56), randn((m, k), torch.bfloat16, 1.0, 57)
    a, b = pack_a(w).cuda(), pack_b(x).cuda() if native else x.cuda()
    kid, p1, p2, p3 = (8, 2, 1, 64) if dealt else \
        ops._gemm_args("continuous_gemm" if native else "layoutA_gemm", n, m, k, 1, int(native))
    assert p3 > 1

    def run(slices):
        fn = mlk.gemm_layoutAB_ContinuousC_wapper if native else mlk.gemm_layoutA_wapper
        return fn(a, b, n, m, k, kernelParam1=p1, kernelParam2=p2, kernelParam3=slices, kernelId=kid)

    def call():
        return run(p3) if dealt else (mlk.gemm_layoutAB_ContinuousC if native else mlk.gemm_layoutA)(a, b)
    whole = run(1)

    def full(device, stream, nbytes, prefix_bytes=0):
        raise torch.OutOfMemoryError("no room for %d bytes" % nbytes)
    with monkeypatch.context() as patch:
        patch.setattr(ops._gemm_pool, "get", full)
        for _ in range(2):
            assert torch.equal(call(), whole)
    want = ogemm.linear_expected(w, x)
    assert_close(whole, want, RTOL, ATOL, "no scratch")
    split = call()
    assert_close(split, want, RTOL, ATOL, "scratch")
    assert not torch.equal(split, whole), "the two orders of summation cannot be told apart"


def test_gemm_eight_wave_panels_replayed_from_a_graph(mlk):
    """The second launch of a sliced product under capture: every replay equals the eager result."""
    n, m, k = 1024, 100, 4096
    w, x = randn((n, k), torch.bfloat16, 0.02, 38), randn((m, k), torch.bfloat16, 1.0, 39).cuda()
    a = pack_a(w).cuda()
    want = mlk.gemm_layoutA(a, x)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        mlk.gemm_layoutA(a, x)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            c = mlk.gemm_layoutA(a, x)
    for _ in range(3):
        c.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want)
        assert torch.equal(mlk.gemm_layoutA(a, x), want)
