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


@pytest.mark.parametrize("m,k,n", [
    (1000, 512, 1600),    # 1.6 MB: tiles
    (1000, 512, 1568),    # just below
    (1000, 512, 1610),    # off the 16-channel grid
    (700, 1024, 2304),
    (4133, 1024, 1040),   # a last row tile and a last 16 channels
    (5000, 1024, 4096),   # persistent
    (2048, 128, 2048),    # one or two stages
    (401, 4096, 4096),
])
def test_linear(m, k, n):
    say("linear", m, k, n)
    gen = torch.Generator("cuda").manual_seed(m + n)
    x = torch.quantize_per_tensor(torch.randn(m, k, device="cuda", generator=gen), 8.0 / 255, 128, torch.quint8)
    packed = OPS.linear_prepack(weight(gen, n, k), torch.randn(n, device="cuda", generator=gen))
    scale = 8 * k ** 0.5 / 255
    whole = OPS.linear(x, packed, scale, 128).int_repr()
    step = max(1, (1 << 20) // n)
    for lo in range(0, m, step):
        assert torch.equal(whole[lo:lo + step], OPS.linear(x[lo:lo + step], packed, scale, 128).int_repr()), lo
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
