"""The tensor-level entry points' own bookkeeping (flour_amd/ops.py), with the library's calls
recorded instead of launched: no GPU needed."""
from __future__ import annotations

import ctypes
import gc
import weakref

import pytest
import torch

from flour_amd import ops


class RecordingLib:
    """Stands in for libflour_hip.so: sizes as the argument says, launches recorded."""

    def __init__(self, nbytes: int):
        self.nbytes, self.calls = nbytes, []

    def flour_hip_paged_decode_workspace_size(self, *args) -> int:
        ctypes.cast(args[-1], ctypes.POINTER(ctypes.c_size_t))[0] = self.nbytes
        return 0

    def flour_hip_paged_decode(self, *args) -> int:
        self.calls.append(args)
        return 0


@pytest.fixture
def recorded(monkeypatch):
    rec = RecordingLib(4096)
    monkeypatch.setattr(ops, "lib", lambda: rec)
    monkeypatch.setattr(ops, "_need_cuda", lambda *ts: None)
    monkeypatch.setattr(ops, "_stream", lambda: ctypes.c_void_p(0))
    monkeypatch.setattr(ops, "_default_ws", {})
    return rec


def decode_args(dtype, max_ctx, D=64):
    q = torch.zeros(2, 8, D, dtype=dtype)
    pool = torch.zeros(8, 16 * 64, D, dtype=dtype)
    return (q, pool, pool, torch.zeros(2, 64, dtype=torch.int32),
            torch.zeros(2, dtype=torch.int32), 0.125, max_ctx)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("then", ["grow", "drop"])
def test_prepared_decode_owns_its_workspace(recorded, dtype, then):
    """A prepared step launches with the address of its workspace's buffer: the buffer lives as long
    as the step does, also when another call makes the workspace grow or when it is dropped."""
    ws = ops.Workspace("cpu")
    args = decode_args(dtype, 1000)
    step = ops.prepare_paged_decode(*args, torch.empty_like(args[0]), ws)
    buf = weakref.ref(ws.buf)
    address = ws.buf.data_ptr()
    if then == "grow":
        ws.get(1 << 20)
    else:
        del ws
    gc.collect()
    assert buf() is not None and buf().data_ptr() == address
    step()
    assert recorded.calls[-1][-3].value == address
    del step
    gc.collect()
    assert buf() is None


@pytest.mark.parametrize("max_ctx", [1, 128, 255, 256, 257, 4096])
def test_fp32_decode_without_a_workspace_shares_none(recorded, max_ctx):
    """Two fp32 steps without a workspace argument never get the same scratch, whatever rule the
    library has for the length from which it uses one: their own, or none."""
    args = decode_args(torch.float32, max_ctx)
    held = []
    for _ in range(2):
        ops.paged_decode(*args)
        *_, address, nbytes, _ = recorded.calls[-1]
        held.append((address.value or 0, nbytes))
    assert not ops._default_ws
    for address, nbytes in held:
        assert (address == 0) == (nbytes == 0)


def test_16_bit_decode_without_a_workspace_reuses_the_default(recorded):
    args = decode_args(torch.bfloat16, 300)
    for _ in range(2):
        ops.paged_decode(*args)
    a, b = (call[-3].value for call in recorded.calls)
    assert a == b == ops._default_ws[0].buf.data_ptr()
