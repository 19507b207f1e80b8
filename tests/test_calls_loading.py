"""CPU: the launchers without the extension of their per-call path
(lib/dmx_calls.so): where it is not built, or built for another torch, one
warning names why and the launchers take their general path, which launches
the same kernels through the C ABI."""

import types
import warnings

import pytest
import torch

from drinkme_amd import _native, radix_ops


@pytest.fixture
def unloaded(monkeypatch):
    monkeypatch.setattr(_native, "_calls", _native._UNLOADED)
    return monkeypatch


def _runtime(rows, cols):
    buf = {"rx_data": torch.zeros(8, dtype=torch.int32), "rx_offsets": torch.zeros(8, dtype=torch.int32),
           "rx_palette": torch.zeros(2, dtype=torch.int32)}
    return {**buf, "R": rows, "C": cols, "codec": "radix"}


def test_a_missing_extension_is_none_with_one_warning(unloaded, tmp_path):
    unloaded.setattr(_native, "CALLS", str(tmp_path / "dmx_calls.so"))
    with pytest.warns(RuntimeWarning, match="not built"):
        assert _native.calls() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _native.calls() is None


def test_an_extension_for_another_torch_is_none(unloaded):
    import drinkme_amd

    class Loader:
        def __init__(self, *_):
            pass

        def create_module(self, spec):
            return types.ModuleType("dmx_calls")

        def exec_module(self, module):
            module.torch_version = "0.0.1"

    unloaded.setattr(_native.importlib.machinery, "ExtensionFileLoader", Loader)
    unloaded.setattr(_native, "CALLS", drinkme_amd.__file__)  # (a file that exists)
    with pytest.warns(RuntimeWarning, match="built for torch 0.0.1"):
        assert _native.calls() is None


def test_the_built_extension_is_for_this_torch(unloaded):
    assert _native.calls().torch_version == torch.__version__


def test_the_launchers_take_their_general_path_without_it(unloaded):
    """Seen by the general path's own refusals: the native path raises none."""
    unloaded.setattr(_native, "_calls", None)
    x = torch.zeros(9, 64)
    one, many = radix_ops.RowsLauncher(_runtime(32, 64)), radix_ops.GroupLauncher([_runtime(32, 64)])
    one._live, many._live = (None, 0), (None, None, 0, (32,))  # as after a first call
    for call in (one, many):
        with pytest.raises(ValueError, match="outside 1..8"):
            call(x)
    assert radix_ops.narrow_rows(torch.zeros(32, 64, dtype=torch.bfloat16), x, None) is None
