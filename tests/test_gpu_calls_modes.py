"""GPU: what the launchers' native per-call path (csrc/torch_calls.cpp) must
leave to the general path or pass on to torch: function modes, tensor
subclasses, vmap, dispatch modes, and streams other than the first call's."""

import numpy as np
import pytest

from tests.helpers import finite_bits, oracle_dict

pytestmark = pytest.mark.gpu

C = 2048


@pytest.fixture(scope="module")
def launch(cuda):
    """[(name, call(x) -> tensor, native(x) -> tensor or None)] for one
    Linear, a group and a raw narrow Linear, each called once before."""
    import torch

    from drinkme_amd import _native, radix_ops, swap

    rng = np.random.default_rng(11)
    p, q = (swap.to_device_radix(oracle_dict(finite_bits(rng, (R, C), spread=True), "sip"), cuda) for R in (130, 66))
    one, many = radix_ops.RowsLauncher(p), radix_ops.GroupLauncher([p, q])
    lin = torch.nn.Linear(C, 48, bias=False, device=cuda, dtype=torch.bfloat16).requires_grad_(False)
    mod = swap.NarrowLinear.adopt(lin)
    native, stream = _native.calls(), lambda: radix_ops._stream(cuda)

    def rows(x):
        return native.rows(one._live[1], p, x, None, torch.float32, 130, C, 0, stream())

    def group(x):
        return native.group(many._live[2], [p, q], x, 0, 0, torch.bfloat16, (130, 66), C, 0, stream())

    calls = [("rows", one, rows), ("group", lambda x: torch.cat(many(x), -1), group),
             ("narrow", mod, lambda x: radix_ops.narrow_rows(lin.weight, x, None))]
    for _, call, _ in calls:
        call(torch.zeros(1, C, device=cuda, dtype=torch.bfloat16))
    return calls


def _x(cuda, seed=0):
    import torch

    gen = torch.Generator(device=cuda).manual_seed(seed)
    return torch.randn(3, C, generator=gen, device=cuda).to(torch.bfloat16)


def test_function_modes_and_subclasses_go_the_general_way(cuda, launch):
    import torch
    from torch.overrides import TorchFunctionMode

    class Seen(TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    x = _x(cuda)
    for name, call, native in launch:
        print(f"case calls modes {name}", flush=True)
        want = call(x)
        seen = Seen()
        with seen:
            assert native(x) is None, name
            assert torch.equal(call(x), want), name
        assert "empty" in seen.names, name  # (the mode saw the output made)
        sub = x.as_subclass(Sub)
        assert native(sub) is None, name
        assert torch.equal(call(sub).as_subclass(torch.Tensor), want), name


def test_vmap_is_refused_and_dispatch_modes_see_the_output(cuda, launch):
    import torch
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.made = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.made += "empty" in str(func)
            return func(*args, **(kwargs or {}))

    x = _x(cuda)
    for name, call, native in launch:
        print(f"case calls dispatch {name}", flush=True)
        want = call(x)
        seen = Seen()
        with seen:
            got = call(x)
        assert seen.made >= 1 and torch.equal(got, want), name
        with pytest.raises(RuntimeError):  # a batched tensor has no address
            torch.vmap(call)(x[:, None])


def test_other_streams_and_threads_after_the_first_call(cuda, launch):
    """Each call runs on its caller's current stream: its input is produced
    there, late, and its output is read there. The same launcher from four
    threads with a stream each."""
    import threading

    import torch

    for name, call, _ in launch:
        print(f"case calls streams {name}", flush=True)
        xs = [_x(cuda, s) for s in range(4)]
        want = [call(x) for x in xs]
        torch.cuda.synchronize()
        got, errors = [None] * 4, []

        def work(i):
            try:
                with torch.no_grad(), torch.cuda.stream(torch.cuda.Stream(device=cuda)):
                    for _ in range(20):
                        x = torch.zeros_like(xs[i])
                        big = torch.randn(2048, 2048, device=cuda)
                        for _ in range(4):
                            big = big @ big * 1e-2
                        x.copy_(xs[i])  # (after the products: a launch on another stream would read zeros)
                        y = call(x)
                        if not torch.equal(y, want[i]):
                            raise AssertionError(f"{name}: thread {i} read another stream's data")
                    torch.cuda.current_stream().synchronize()
                got[i] = True
            except BaseException as e:  # noqa: BLE001 (handed to the main thread)
                errors.append(e)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors[0]
        assert all(got)
