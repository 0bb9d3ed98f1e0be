"""Outputs large enough that their bytes leave past the L2s, against the same images (rows) in calls too small for that: the
same bytes.  Either side of each line in sizes and channel counts; what the small calls give is compared with the oracle
elsewhere."""
import pytest
import torch

import torch_musa_amd  # noqa: F401  (registers the operators)
from gpu_util import say

pytestmark = pytest.mark.gpu
OPS = torch.ops.quantized


def feature_map(gen, b, h, w, c):
    x = torch.relu(torch.randn(b, h, w, c, device="cuda", generator=gen)).permute(0, 3, 1, 2)
    return torch.quantize_per_tensor(x, 4.0 / 255, 0, torch.quint8)


def weight(gen, *shape):
    w = torch.randn(*shape, device="cuda", generator=gen)
    scales = w.abs().flatten(1).amax(1).double() / 127
    return torch.quantize_per_channel(w, scales, torch.zeros(shape[0], dtype=torch.long, device="cuda"), 0, torch.qint8)


@pytest.mark.parametrize("b,h,w,ic,oc,k,groups,post", [
    (10, 56, 53, 24, 56, 1, 1, ""),          # 1.7 MB, channels off the grid
    (10, 56, 53, 24, 64, 1, 1, "relu"),      # 1.9 MB, a block of 64 channels
    (30, 56, 53, 20, 24, 1, 1, "relu"),      # 2.1 MB, eight channels a lane
    (17, 41, 57, 64, 80, 1, 1, "add"),       # a last block of 16 channels
    (17, 41, 57, 64, 96, 1, 1, "silu"),
    (33, 56, 57, 24, 208, 1, 1, "relu"),     # past 20 MB, channel blocks on several CUs
    (27, 56, 57, 24, 256, 1, 1, "relu"),     # past 20 MB, on one
    (16, 41, 37, 64, 64, 3, 1, "relu"),      # halo tiles
    (16, 41, 37, 64, 80, 3, 1, "add"),
    (33, 56, 57, 64, 96, 3, 1, "relu"),      # past 8 MB, lines of several blocks
    (30, 56, 57, 60, 60, 3, 60, "relu"),     # depthwise, 5.7 MB
    (30, 56, 57, 66, 66, 3, 66, "relu"),     # off the 4-channel grid
    (16, 29, 31, 256, 272, 3, 1, "relu"),    # implicit GEMM
    (20, 61, 67, 3, 24, 3, 1, "relu"),       # images
    (3, 61, 67, 3, 64, 7, 1, "relu"),
    (20, 61, 67, 1, 48, 3, 1, "relu"),       # byte runs
])
def test_conv(b, h, w, ic, oc, k, groups, post):
    say("conv", b, h, w, ic, oc, k, groups, post)
    gen = torch.Generator("cuda").manual_seed(b + oc)
    x, accum = feature_map(gen, b, h, w, ic), feature_map(gen, b, h, w, oc)
    packed = OPS.conv2d_prepack(weight(gen, oc, ic // groups, k, k), torch.randn(oc, device="cuda", generator=gen),
                                [1, 1], [k // 2, k // 2], [1, 1], groups)
    scale = 8 * (ic // groups * k * k) ** 0.5 / 255

    def run(lo, hi):
        xs = x[lo:hi]
        if post == "add":
            return OPS.conv2d_add_relu(xs, accum[lo:hi], packed, scale, 3).int_repr()
        op = {"": OPS.conv2d, "relu": OPS.conv2d_relu, "silu": OPS.conv2d_silu}[post]
        return op(xs, packed, scale, 3).int_repr()

    whole = run(0, b)
    for i in range(b):
        assert torch.equal(whole[i:i + 1], run(i, i + 1)), i
    assert whole.unique().numel() > 50


# Products whose tiles may write outputs of any size: past the L2s up to 24 MiB, where channels lie on the 64-byte grid up to
# 52 MiB (256 x 256 tiles there at any size), against the plain kernel, which has ordinary stores only.
@pytest.mark.parametrize("n,rows", [(272, (92521, 92522)), (4096, (13312, 13313))])
@pytest.mark.parametrize("cfg,k", [(1, 384), (2, 384), (3, 384), (7, 384), (17, 384), (20, 384), (1, 64), (2, 64)])
@pytest.mark.parametrize("x_signed", [False, True])
def test_products_on_either_side_of_the_lines(n, rows, cfg, k, x_signed):
    from torch_musa_amd import cabi
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
    from torch_musa_amd import cabi
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


@pytest.mark.parametrize("rows,cols,axis", [(7168, 4096, 0), (7167, 4096, 0), (4100, 8196, 0), (28001, 1050, 0)])
def test_quantize(rows, cols, axis):
    say("quantize", rows, cols)
    gen = torch.Generator("cuda").manual_seed(rows)
    x = torch.randn(rows, cols, device="cuda", generator=gen)
    scales = x.abs().amax(1).double() / 127
    zps = torch.zeros(rows, dtype=torch.long, device="cuda")
    whole, channels = torch.quantize_per_tensor(x, 0.03, 5, torch.qint8), torch.quantize_per_channel(x, scales, zps, axis, torch.qint8)
    step = 3001
    for lo in range(0, rows, step):
        part = x[lo:lo + step].contiguous()
        assert torch.equal(whole.int_repr()[lo:lo + step], torch.quantize_per_tensor(part, 0.03, 5, torch.qint8).int_repr())
        few = torch.quantize_per_channel(part, scales[lo:lo + step].contiguous(), zps[lo:lo + step].contiguous(), axis, torch.qint8)
        assert torch.equal(channels.int_repr()[lo:lo + step], few.int_repr())


@pytest.mark.parametrize("c", [48, 56])
def test_max_pool(c):
    gen = torch.Generator("cuda").manual_seed(c)
    x = feature_map(gen, 9, 147, 159, c)  # 2.6 and 3.1 MB of maxima in all
    whole = torch.nn.functional.max_pool2d(x, 3, 2, 1).int_repr()
    for i in range(9):
        assert torch.equal(whole[i:i + 1], torch.nn.functional.max_pool2d(x[i:i + 1], 3, 2, 1).int_repr())
