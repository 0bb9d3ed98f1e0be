"""The native call paths of torch.ops.quantized.*: the same results, errors and hooks as PyTorch's own callable
(`packet._op`), on CPU tensors."""
import pytest
import torch
import torch_musa_amd  # noqa: F401  (installs them)

OPS = torch.ops.quantized


def _operands(name):
    torch.manual_seed(3)
    x = torch.quantize_per_tensor(torch.randn(5, 16), 0.05, 120, torch.quint8)
    if name.startswith("linear"):
        w = torch.quantize_per_tensor(torch.randn(7, 16), 0.02, 0, torch.qint8)
        packed = OPS.linear_prepack(w, torch.randn(7))
        return (torch.randn(5, 16), packed) if "dynamic" in name else (x, packed, 0.1, 99)
    if name.startswith("conv"):
        one = name.startswith("conv1d")
        shape, w_shape = ((2, 6, 9), (4, 6, 3)) if one else ((2, 6, 9, 8), (4, 6, 3, 3))
        w = torch.quantize_per_tensor(torch.randn(w_shape), 0.02, 0, torch.qint8)
        n = 1 if one else 2
        prepack = OPS.conv1d_prepack if one else OPS.conv2d_prepack
        xc = torch.quantize_per_tensor(torch.randn(shape), 0.05, 120, torch.quint8)
        return xc, prepack(w, torch.randn(4), [1] * n, [1] * n, [1] * n, 1), 0.2, 101
    return x, torch.quantize_per_tensor(torch.randn(5, 16), 0.03, 7, torch.quint8), 0.08, 128


@pytest.mark.parametrize("name", ["linear", "linear_relu", "linear_dynamic", "linear_relu_dynamic", "conv2d",
                                  "conv2d_relu", "conv1d", "conv1d_relu", "add", "add_relu"])
def test_same_results_errors_and_hooks(name):
    packet, args = getattr(OPS, name), _operands(name)
    assert isinstance(packet, torch._ops.OpOverloadPacket) and packet.__name__ == name
    plain = (lambda t: t.int_repr()) if args[0].is_quantized else (lambda t: t)
    want = plain(packet._op(*args))
    assert torch.equal(plain(packet(*args)), want)
    schema = (packet.new if name.startswith("conv2d") else packet.default)._schema
    names = [a.name for a in schema.arguments]
    assert torch.equal(plain(packet(args[0], **dict(zip(names[1:], args[1:])))), want)
    for bad in (args[:1], args + (1, 2, 3, 4, 5), (args[0], "w") + args[2:], (1.5,) + args[1:]):
        with pytest.raises(RuntimeError) as got:
            packet(*bad)
        with pytest.raises(RuntimeError) as own:
            packet._op(*bad)
        assert str(got.value).splitlines()[0] == str(own.value).splitlines()[0]

    seen = []

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Mode():
        assert torch.equal(plain(packet(*args)), want)
    assert len(seen) > 0
