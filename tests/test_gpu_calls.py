"""GPU: the launchers' native per-call path (csrc/torch_calls.cpp) against
the general path (the functional gemv_rows / gemv_group / gemv_narrow calls):
the same bits for every form of activation, bias and output it takes, and the
general path's answer or refusal for every form it does not."""

import numpy as np
import pytest

from oracle import radix_oracle as O
from tests.helpers import finite_bits, oracle_dict

pytestmark = pytest.mark.gpu

C = 2048


def _tensors(cuda, rows, profile="sip"):
    from drinkme_amd import swap

    rng = np.random.default_rng(sum(rows))
    return [swap.to_device_radix(oracle_dict(finite_bits(rng, (R, C), spread=True), profile), cuda) for R in rows]


def _activations(cuda):
    """(name, x, taken): plain forms, and forms the native path leaves alone."""
    import torch

    gen = torch.Generator(device=cuda).manual_seed(3)
    base = torch.randn(8, C, generator=gen, device=cuda)
    for dtype in (torch.bfloat16, torch.float32):
        b = base.to(dtype)
        yield f"row {dtype}", b[0], True
        yield f"leading dimensions {dtype}", b[:6].view(2, 3, C), True
        yield f"eight rows {dtype}", b, True
        yield f"offset by one element {dtype}", torch.cat([b[0, :1], b.reshape(-1)])[1:].view(8, C)[:3], True
        yield f"transposed {dtype}", b.t().contiguous().t()[:4], False
        yield f"every other row {dtype}", b[::2], False
        yield f"expanded {dtype}", b[:1].expand(3, C), False


def test_rows_and_groups_equal_the_general_path(cuda):
    import torch

    from drinkme_amd import _native, radix_ops

    ps = _tensors(cuda, (1027, 64))
    one, many = radix_ops.RowsLauncher(ps[0]), radix_ops.GroupLauncher(ps)
    biases = {None: [None, None]}
    for d in (torch.bfloat16, torch.float32):
        biases[d] = [torch.randn(p["R"], device=cuda).to(d) for p in ps]
    one(torch.zeros(1, C, device=cuda))  # (builds the descriptors)
    many(torch.zeros(1, C, device=cuda))
    for name, x, taken in _activations(cuda):
        print(f"case calls {name}", flush=True)
        rows = x.reshape(-1, C)
        native = _native.calls().rows(one._live[1], ps[0], x, None, torch.float32, 1027, C, x.device.index,
                                      radix_ops._stream(x.device))
        assert (native is not None) == taken, name
        for bs in biases.values():
            for out in (torch.bfloat16, torch.float32):
                y = one(x, bs[0], out)
                assert y.dtype == out and y.shape == (*x.shape[:-1], 1027)
                assert torch.equal(y.reshape(-1, 1027), radix_ops.gemv_rows(ps[0], rows, bs[0], out)), name
                for got, want in zip(many(x, bs, out), radix_ops.gemv_group(ps, rows, bs, out)):
                    assert got.shape[:-1] == x.shape[:-1] and torch.equal(got.reshape(want.shape), want), name


def test_refusals_and_moved_buffers_keep_the_general_paths_answers(cuda):
    import torch

    from drinkme_amd import radix_ops

    p, = _tensors(cuda, (128,))
    one, many = radix_ops.RowsLauncher(p), radix_ops.GroupLauncher([p])
    x = torch.randn(2, C, device=cuda)
    want = one(x)
    for call in (one, many):
        with pytest.raises(ValueError):
            call(x[:, :-1].contiguous())
        with pytest.raises(ValueError, match="outside 1..8"):
            call(torch.zeros(9, C, device=cuda))
        with pytest.raises(ValueError, match="outside 1..8"):
            call(x[:0])
        with pytest.raises(ValueError, match="device"):
            call(x.cpu())
        with pytest.raises(TypeError, match="bf16 or fp32"):
            call(x.half())
    with pytest.raises(ValueError, match="bias"):
        one(x, torch.zeros(127, device=cuda))
    with pytest.raises(TypeError, match="output"):
        one(x, None, torch.float16)
    for key in ("rx_data", "rx_offsets", "rx_palette"):
        p[key] = p[key].clone()  # other buffers in the dict: the descriptors follow
        assert torch.equal(one(x), want) and torch.equal(many(x, None, torch.float32)[0], want), key


def test_narrow_equals_the_general_path(cuda):
    import torch

    from drinkme_amd import radix_ops, swap

    for bias in (False, True):
        lin = torch.nn.Linear(C, 48, bias=bias, device=cuda, dtype=torch.bfloat16)
        mod = swap.NarrowLinear.adopt(lin)
        b = lin.bias
        for name, x, taken in _activations(cuda):
            print(f"case calls narrow {name}", flush=True)
            with torch.no_grad():
                assert (radix_ops.narrow_rows(lin.weight, x, b) is not None) == taken, name
                y = mod(x)
                want = radix_ops.gemv_narrow(lin.weight, x.reshape(-1, C), b)
            assert y.shape == (*x.shape[:-1], 48) and torch.equal(y.reshape(-1, 48), want), name
        with torch.no_grad():
            x9 = torch.randn(9, C, device=cuda, dtype=torch.bfloat16)
            assert torch.equal(mod(x9), torch.nn.functional.linear(x9, lin.weight, b))


def test_without_the_extension_the_general_path_gives_the_same(cuda, monkeypatch):
    import torch

    from drinkme_amd import _native, radix_ops, swap

    p, = _tensors(cuda, (257,))
    one, many = radix_ops.RowsLauncher(p), radix_ops.GroupLauncher([p, p])
    lin = torch.nn.Linear(C, 48, bias=True, device=cuda, dtype=torch.bfloat16)
    mod = swap.NarrowLinear.adopt(lin)
    x = torch.randn(3, C, device=cuda).to(torch.bfloat16)
    with torch.no_grad():
        def passes():
            return [one(x), *many(x), mod(x)]

        passes()  # (builds the descriptors)
        want = passes()
        monkeypatch.setattr(_native, "_calls", None)
        for got, y in zip(passes(), want):
            assert got.shape == y.shape and torch.equal(got, y)
