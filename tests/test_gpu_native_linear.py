"""A quantized layer's forward through the extension module: the same bits as the library's entry points give, the general path where
an input is not what the module takes, and no call of its own where a mode or a transform looks on."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from ajllm_amd import QuantLinear, _lib, quant, w4a16_matmul, w8a16_matmul

pytestmark = pytest.mark.gpu


def _layer(scheme, n, k, cuda):
    g = torch.Generator(device=cuda).manual_seed(n + k)
    return QuantLinear.from_weight(torch.randn((n, k), generator=g, device=cuda) * 0.02, scheme)


def _x(cuda, *shape):
    return torch.randn(shape, generator=torch.Generator(device=cuda).manual_seed(3), device=cuda).to(torch.bfloat16)


@pytest.fixture
def calls(monkeypatch):
    """The general path's products: how often, and what it made."""
    made = []
    plain = quant._matmul
    monkeypatch.setattr(quant, "_matmul", lambda *a: made.append(a) or plain(*a))
    return made


@pytest.mark.parametrize("out", [None, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(256,), (1, 256), (2, 3, 256), (16, 256), (17, 256), (5, 0, 256), (130, 256)])
@pytest.mark.parametrize("scheme", ["w4a16_g128", "w8a16"])
def test_same_bits_as_the_entry_points(cuda, calls, scheme, shape, out):
    layer, x = _layer(scheme, 1024, 256, cuda), _x(cuda, *shape)
    got = layer(x, out_dtype=out)
    assert len(calls) == (1 if x.numel() == 0 else 0)
    matmul = w4a16_matmul if scheme == "w4a16_g128" else w8a16_matmul
    want = matmul(x.reshape(-1, 256), layer.wq, layer.meta, out or torch.bfloat16).view(*shape[:-1], 1024)
    assert got.dtype == (out or torch.bfloat16) and got.shape == want.shape and torch.equal(got, want)
    assert got.is_contiguous() and not got.requires_grad


@pytest.mark.parametrize("scheme", ["w4a16_g128", "w8a16"])
def test_ragged_outputs(cuda, calls, scheme):
    """A number of outputs off the 16-row tiles: a view of the padded result, for every number of dimensions."""
    layer = _layer(scheme, 1000, 256, cuda)
    matmul = w4a16_matmul if scheme == "w4a16_g128" else w8a16_matmul
    for shape in ((256,), (4, 256), (2, 3, 256), (40, 256)):
        x = _x(cuda, *shape)
        got = layer(x)
        assert not calls
        want = matmul(x.reshape(-1, 256), layer.wq, layer.meta)[:, :1000]
        calls.clear()
        assert torch.equal(got, want.reshape(*shape[:-1], 1000)) and got.stride()[-1] == 1
        assert len(shape) < 2 or got.stride()[-2] == 1008


def test_long_k_with_scratch(cuda, calls):
    layer, x = _layer("w8a16", 4096, 14336, cuda), _x(cuda, 37, 14336)
    assert _lib.load().ajq_matmul_scratch_bytes(37, 4096, 14336, 0) > 0
    got = layer(x)
    assert not calls
    assert torch.equal(got, w8a16_matmul(x, layer.wq, layer.meta))


def test_anything_else_takes_the_general_path(cuda, calls):
    layer, x = _layer("w4a16_g128", 1024, 256, cuda), _x(cuda, 4, 256)
    want = layer(x)
    assert not calls
    wide = _x(cuda, 4, 512)[:, ::2]
    assert torch.equal(layer(wide), layer(wide.contiguous())) and len(calls) == 1
    assert torch.equal(layer(x.float(), out_dtype=torch.bfloat16), want) and len(calls) == 2
    assert torch.equal(layer(x, out_dtype=torch.float64), want.double()) and len(calls) == 3

    class Mine(torch.Tensor):
        pass

    assert torch.equal(layer(x.as_subclass(Mine)).as_subclass(torch.Tensor), want) and len(calls) == 4

    class Watching(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Watching():
        assert torch.equal(layer(x), want)
    assert len(calls) == 5
    with pytest.raises((ValueError, RuntimeError)):
        layer(_x(cuda, 4, 128))
    with pytest.raises(ValueError):
        layer(x.cpu())
    with pytest.raises(RuntimeError):
        torch.func.vmap(layer)(x[:, None])
    with pytest.raises(RuntimeError, match="named tensors"):
        layer(x.rename("rows", "columns"))


def test_without_the_module(cuda, calls, monkeypatch):
    layer, x = _layer("w4a16_g128", 1000, 256, cuda), _x(cuda, 2, 3, 256)
    want = layer(x)
    assert not calls
    monkeypatch.setattr(quant, "_linear", quant._leave)
    got = layer(x)
    assert len(calls) == 1 and torch.equal(got, want) and got.stride() == want.stride()


def test_on_a_stream_and_in_a_graph(cuda):
    layer, x = _layer("w8a16", 4096, 14336, cuda), _x(cuda, 37, 14336)
    want = layer(x)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        assert torch.equal(layer(x), want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = layer(x)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
