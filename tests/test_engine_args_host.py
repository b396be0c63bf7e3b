"""The engine's argument marshalling on the CPU: what reaches the library's
calls, recorded by a stand-in for it."""
import struct

import pytest
import torch

from adapterslotsplusplus_amd import _lib, engine as engine_mod
from adapterslotsplusplus_amd.engine import WarpPipeEngine


class RecordingLib:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return _lib.WP_OK

        return call


@pytest.fixture
def eng(monkeypatch):
    """An engine over CPU tensors (device index -1) and the recording library."""
    monkeypatch.setattr(engine_mod, "_raw_stream", lambda dev: 0)
    e = WarpPipeEngine.__new__(WarpPipeEngine)
    e._lib, e._handle, e._dev_index, e._ranks = RecordingLib(), None, -1, {8: True}
    return e


def slices(n, T=3, L=2, d=16, o=12, r=8):
    dt = torch.float16
    return (torch.zeros(T, n * o, dtype=dt), torch.zeros(T, d, dtype=dt),
            [torch.zeros(L, 1, r, d, dtype=dt) for _ in range(n)], [torch.zeros(L, 1, o, r, dtype=dt) for _ in range(n)])


@pytest.mark.parametrize("wrap", [list, tuple, iter, lambda v: (w for w in v)], ids=["list", "tuple", "iter", "generator"])
def test_nslice_takes_any_iterable_of_weights(eng, wrap):
    y, x, was, wbs = slices(3)
    assert eng.add_lora_packed_nslice(y, x, wrap(was), wrap(wbs), 0.5, [12, 12, 12])
    name, args = eng._lib.calls[-1]
    assert name == "wp_add_lora_nslice" and args[3] == 3
    assert struct.unpack("3q", args[6]) == tuple(w.data_ptr() for w in wbs)


def test_offsets_reach_the_library_one_per_slice(eng):
    """The library reads one offset per slice: those not given are 0, and more
    than the slices are refused."""
    y, x, was, wbs = slices(3)
    for given in ([], [4], [0, 12], [0, 12, 24]):
        assert eng.add_lora_slices(y, x, was[0], wbs, 0.5, given)
        name, args = eng._lib.calls[-1]
        assert name == "wp_add_lora" and args[6] == 3
        assert struct.unpack("3i", args[10]) == tuple((given + [0, 0, 0])[:3])
    with pytest.raises(IndexError):
        eng.add_lora_slices(y, x, was[0], wbs, 0.5, [0, 12, 24, 36])
    with pytest.raises(IndexError):
        eng.add_lora_packed_nslice(y, x, was, wbs, 0.5, [12, 12, 12, 12])
