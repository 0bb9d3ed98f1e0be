"""Outputs whose bytes leave past the L2s, on either side of each rule's lines in sizes and channel counts, against ordinary
stores of the same values: an output pointer off the 16-byte grid, the plain kernel, calls short of the line, or torch's own
pooling.  The values themselves are compared with the oracle elsewhere."""
import pytest
import torch

from gpu_util import say
from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu


def off_grid(shape, dtype):
    """An uninitialised output one byte past the grid, and the bytes around it, which have to stay."""
    n = 1
    for d in shape:
        n *= d
    flat = torch.full((n + 64,), 77, dtype=dtype, device="cuda")
    return flat[1:n + 1].view(shape), [flat[:1], flat[n + 1:]]


@pytest.mark.parametrize("b,h,w,ic,oc,k,groups,post", [
    (10, 56, 53, 24, 56, 1, 1, "none"),       # channels off the grid: never past the L2s
    (10, 56, 53, 24, 64, 1, 1, "relu"),       # pointwise: a block of 64 channels
    (30, 56, 53, 20, 24, 1, 1, "relu"),       # eight channels a lane
    (17, 41, 57, 64, 80, 1, 1, "add"),        # a last block of 16 channels
    (17, 41, 57, 64, 96, 1, 1, "silu"),
    (5, 41, 57, 128, 80, 1, 1, "silu"),       # 0.93 MB behind SiLU and 65 to 128 channels: ordinary
    (6, 41, 57, 128, 80, 1, 1, "silu"),       # 1.1 MB
    (27, 56, 57, 24, 144, 1, 1, "relu"),      # parts of lines, 12.4 MB
    (28, 56, 57, 24, 144, 1, 1, "relu"),      # 12.9 MB, past 12 MiB: ordinary stores
    (28, 56, 57, 24, 144, 1, 1, "silu"),      # ... but behind SiLU
    (34, 56, 57, 24, 192, 1, 1, "relu"),      # whole lines, 20.8 MB
    (35, 56, 57, 24, 192, 1, 1, "relu"),      # 21.5 MB, past 20 MiB: ordinary
    (27, 56, 57, 24, 256, 1, 1, "relu"),      # ... but where a pixel's channel blocks are one CU's
    (18, 56, 57, 256, 384, 1, 1, "relu"),     # ... or the layer is wide
    (16, 41, 37, 64, 64, 3, 1, "relu"),       # halo tiles
    (16, 41, 37, 64, 80, 3, 1, "add"),
    (27, 56, 57, 64, 96, 3, 1, "relu"),       # lines of several blocks, 8.3 MB
    (28, 56, 57, 64, 96, 3, 1, "relu"),       # 8.6 MB, past 8 MiB: ordinary
    (24, 56, 57, 60, 60, 3, 60, "relu"),      # depthwise, 4.6 MB: ordinary below 4.5 MiB
    (25, 56, 57, 60, 60, 3, 60, "relu"),      # 4.8 MB
    (25, 56, 57, 60, 60, 5, 60, "silu"),      # ... ordinary under a larger window
    (25, 56, 57, 60, 60, 7, 60, "relu"),
    (25, 56, 57, 60, 60, 3, 60, "silu"),
    (54, 56, 57, 96, 96, 5, 96, "relu"),      # 16.5 MB
    (55, 56, 57, 96, 96, 5, 96, "relu"),      # 16.9 MB, past 16 MiB: ordinary
    (30, 56, 57, 66, 66, 3, 66, "relu"),      # off the 4-channel grid
    (16, 29, 31, 256, 272, 3, 1, "relu"),     # implicit GEMM
    (20, 61, 67, 3, 24, 3, 1, "relu"),        # images, of any size
    (3, 61, 67, 3, 64, 7, 1, "relu"),
    (3, 61, 67, 3, 64, 7, 1, "silu"),         # but SiLU behind 7 x 7 short of 1 MiB
    (5, 61, 67, 3, 64, 7, 1, "silu"),
    (20, 61, 67, 1, 48, 3, 1, "relu"),        # byte runs, 3.9 MB
    (10, 61, 67, 1, 48, 3, 1, "relu"),        # 2.0 MB, short of 2 MiB: ordinary
    (27, 56, 57, 24, 592, 1, 1, "silu"),      # parts of lines behind SiLU past 48 MiB: ordinary
])
@pytest.mark.parametrize("out_signed", [False, True])
def test_conv(b, h, w, ic, oc, k, groups, post, out_signed):
    say("conv", b, h, w, ic, oc, k, groups, post, out_signed)
    gen = torch.Generator("cuda").manual_seed(b + oc)
    x = torch.randint(0, 256, (b, h, w, ic), generator=gen, device="cuda").to(torch.uint8)
    wq = torch.randint(-127, 128, (oc, k, k, ic // groups), generator=gen, device="cuda").to(torch.int8)
    ws = torch.rand(oc, generator=gen, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(oc, generator=gen, device="cuda") * 0.1
    accum = torch.randint(0, 256, (b, h, w, oc), generator=gen, device="cuda").to(torch.uint8) if post == "add" else None
    g = cabi.conv_geom(tuple(x.shape), tuple(wq.shape), (1, 1), (k // 2, k // 2), (1, 1), groups)
    pw = cabi.PackedConv2d(wq, g)
    scale, zp = (ic // groups * k * k) ** 0.5 / 400, 0 if out_signed else 100
    dtype = torch.int8 if out_signed else torch.uint8

    def run(out):
        return cabi.conv2d_fused(x, pw, g, 0.03, 128, ws, bias, scale, zp, accum=accum, accum_scale=0.02, accum_zp=100,
                                 activation="relu" if post == "add" else post, out_signed=out_signed, out=out)

    plain, around = off_grid((b, h, w, oc), dtype)
    run(plain)
    assert all(bool((a == 77).all()) for a in around)
    on_grid = run(torch.full((b, h, w, oc), 77, dtype=dtype, device="cuda"))
    assert torch.equal(on_grid, plain)
    assert on_grid.unique().numel() > 50


@pytest.mark.parametrize("m,k,n", [
    (700, 1024, 2304), (1000, 512, 1600), (1000, 512, 1610), (384, 768, 3072),   # tiles that are never large
    (1000, 512, 1000), (517, 1008, 2048), (130, 640, 130),                       # all of K in LDS
    (4133, 1024, 1040), (2048, 128, 2048), (401, 4096, 4096), (5000, 1024, 4096),
])
def test_products(m, k, n):
    say("product", m, k, n)
    gen = torch.Generator("cuda").manual_seed(m + n)
    x = torch.randint(0, 256, (m, k), generator=gen, device="cuda").to(torch.uint8)
    pw = cabi.PackedLinear(torch.randint(-127, 128, (n, k), generator=gen, device="cuda").to(torch.int8))
    ws = torch.rand(n, generator=gen, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(n, generator=gen, device="cuda")
    plain, around = off_grid((m, n), torch.uint8)
    outs = [cabi.linear(x, pw, 0.05, 128, ws, bias, k ** 0.5 / 100, 100, out=out)
            for out in (plain, torch.full((m, n), 77, dtype=torch.uint8, device="cuda"))]
    assert all(bool((a == 77).all()) for a in around)
    assert torch.equal(*outs)
    assert plain.unique().numel() > 100


# Products whose tiles may write outputs of any size: past the L2s up to 24 MiB, where channels lie on the 64-byte grid up to
# 52 MiB (256 x 256 tiles there at any size), against the plain kernel, which has ordinary stores only.
@pytest.mark.parametrize("n,rows", [(272, (92521, 92522)), (4096, (13312, 13313))])
@pytest.mark.parametrize("cfg,k", [(1, 384), (2, 384), (3, 384), (7, 384), (17, 384), (20, 384), (1, 64), (2, 64)])
@pytest.mark.parametrize("x_signed", [False, True])
def test_products_on_either_side_of_the_lines(n, rows, cfg, k, x_signed):
    lo, hi, dt = (-128, 128, torch.int8) if x_signed else (0, 256, torch.uint8)
    gen = torch.Generator("cuda").manual_seed(n + k)
    pw = cabi.PackedLinear(torch.randint(-127, 128, (n, k), generator=gen, device="cuda").to(torch.int8))
    ws = torch.rand(n, generator=gen, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(n, generator=gen, device="cuda")
    for m in rows:
        x = torch.randint(lo, hi, (m, k), generator=gen, device="cuda").to(dt)
        for pitch in {n, 272 if n == 272 else 4160}:   # rows of a wider output as well
            say("product", m, n, k, cfg, x_signed, pitch)
            outs = []
            for pin in (9, cfg):
                y = torch.full((m, pitch), 77, dtype=dt, device="cuda")
                cabi.force_linear_config(pin)
                try:
                    outs.append(cabi.linear(x, pw, 0.05, 3, ws, bias, k ** 0.5 / 100, 10 if x_signed else 100, out=y[:, :n]))
                finally:
                    cabi.force_linear_config(-1)
                assert bool((y[:, n:] == 77).all())
            assert torch.equal(*outs)
            assert outs[0].unique().numel() > 100


# Implicit GEMMs likewise: two images past the line (ordinary stores), each by itself below it.
@pytest.mark.parametrize("h,w,ic,oc,tile", [
    (217, 214, 288, 272, (0, 1)), (217, 214, 288, 272, (128, 1)), (217, 214, 288, 272, (256, 1)),
    (653, 653, 144, 64, (128, 1)),                                       # whole lines
    (513, 512, 32, 48, (0, 0)), (397, 397, 32, 80, (0, 0)),              # the k order walked, 256 x 64 and 128 x 128
])
def test_implicit_gemm_on_either_side_of_the_lines(h, w, ic, oc, tile):
    say("implicit GEMM", h, w, ic, oc, tile)
    gen = torch.Generator("cuda").manual_seed(oc + ic)
    x = torch.randint(0, 256, (2, h, w, ic), generator=gen, device="cuda").to(torch.uint8)
    wq = torch.randint(-127, 128, (oc, 1, 1, ic), generator=gen, device="cuda").to(torch.int8)
    ws = torch.rand(oc, generator=gen, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(oc, generator=gen, device="cuda") * 0.1

    def run(xs):
        g = cabi.conv_geom(tuple(xs.shape), tuple(wq.shape), (1, 1), (0, 0), (1, 1), 1)
        cabi.force_conv_path(2)
        cabi.force_conv_tile(*tile)
        try:
            return cabi.conv2d(xs, cabi.PackedConv2d(wq, g), g, 0.03, 60, ws, bias, ic ** 0.5 / 400, 100)
        finally:
            cabi.force_conv_path(-1)
            cabi.force_conv_tile(0, 0)

    whole = run(x)
    for i in range(2):
        assert torch.equal(whole[i:i + 1], run(x[i:i + 1].contiguous()))
    assert whole.unique().numel() > 100


# 28 Mi codes and more (per tensor short of 96 Mi) leave past the L2s: the whole against runs of rows short of that.
@pytest.mark.parametrize("rows,cols", [(7168, 4096), (7167, 4096), (4100, 8196), (28001, 1050), (24575, 4096), (24576, 4096)])
def test_quantize(rows, cols):
    say("quantize", rows, cols)
    gen = torch.Generator("cuda").manual_seed(rows)
    x = torch.randn(rows, cols, device="cuda", generator=gen)
    scales = x.abs().amax(1) / 127
    zps = torch.randint(-5, 6, (rows,), generator=gen, device="cuda")

    def codes(lo, hi):
        xs, sc, zp = x[lo:hi], scales[lo:hi].clone(), zps[lo:hi].clone()   # (whole rows: contiguous, on the grid of the whole)
        return (cabi.quantize_per_tensor(xs, 0.03, 5, True), cabi.quantize_per_channel(xs, sc.double(), zp, 0, True),
                cabi.quantize_per_channel_float_qparams(xs, sc, zp.float() + 0.25, 0, True))

    whole, step = codes(0, rows), 3000
    for lo in range(0, rows, step):
        for a, few in zip(whole, codes(lo, min(lo + step, rows))):
            assert torch.equal(a[lo:lo + step], few), lo
    assert all(a.unique().numel() > 100 for a in whole)


# Up to 3 MiB of maxima on the 16-channel grid (2.6, 3.1 and 3.0 MB); 3.4 MB and off that grid by ordinary stores.
@pytest.mark.parametrize("b,c", [(9, 48), (11, 48), (8, 64), (9, 64), (9, 56)])
@pytest.mark.parametrize("dtype", [torch.quint8, torch.qint8])
def test_max_pool(b, c, dtype):
    say("max pool", b, c, dtype)
    gen = torch.Generator("cuda").manual_seed(c)
    x = torch.randn(b, 147, 159, c, device="cuda", generator=gen).permute(0, 3, 1, 2)
    q = torch.quantize_per_tensor(x, 6.0 / 255, 128 if dtype == torch.quint8 else 0, dtype)
    expected = torch.nn.functional.max_pool2d(q.int_repr().float(), 3, 2, 1)
    assert torch.equal(torch.nn.functional.max_pool2d(q, 3, 2, 1).int_repr().float(), expected)
