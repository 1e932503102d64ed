"""Host-side parts of the Python mirror that need no GPU: pinned slots of scalar results, shapes."""
import numpy as np
import pytest


class _Stream:
    def __init__(self, fail=False):
        self.waits, self.fail = 0, fail

    def synchronize(self):
        self.waits += 1
        if self.fail:
            raise RuntimeError("stream error")


@pytest.fixture()
def slots(rk, monkeypatch):
    """The module with one slot of ordinary memory and a stream that can be told to fail or to be capturing."""
    from amdgpu_jl_amd import array
    words = np.zeros(array.SLOT_BYTES, dtype=np.uint8)
    slot = (words.ctypes.data, words, None)
    state = dict(stream=_Stream(), capturing=False)
    monkeypatch.setattr(array, "_free_slots", [slot])
    monkeypatch.setattr(array, "_parked_slots", [])
    monkeypatch.setattr(array, "check_waits", lambda: None)
    monkeypatch.setattr(array, "stream_ptr", lambda: 0)
    monkeypatch.setattr(array.torch.cuda, "current_stream", lambda *a: state["stream"])
    monkeypatch.setattr(array.torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    return array, slot, state


def test_a_slot_is_read_after_the_wait(slots):
    array, slot, state = slots
    got = array.take_slot()
    assert got is slot and array._free_slots == []

    def call(*args):
        assert args == (slot[0], 3, 0) and state["stream"].waits == 0
        slot[1][0] = 7
        return 0
    array.fill_slot(got, call, "call", (slot[0], 3))
    assert got[1][0] == 7 and state["stream"].waits == 1
    array.give_slot(got)
    assert array._free_slots == [slot] and array._parked_slots == []


@pytest.mark.parametrize("where", ["launch", "status", "wait"])
@pytest.mark.parametrize("error", [ValueError, KeyboardInterrupt])
def test_an_interrupted_fetch_waits_before_the_slot_is_used_again(slots, monkeypatch, where, error):
    array, slot, state = slots

    def stop(*args):
        assert state["stream"].waits == 0
        raise error()
    if where == "wait":
        monkeypatch.setattr(array, "check_waits", stop)
    if where == "status":
        error = array.L.RKError
    call = {"launch": stop, "status": lambda *a: array.L.RK_ERR_WORKSPACE, "wait": lambda *a: 0}[where]
    with pytest.raises(error):
        array.fill_slot(array.take_slot(), call, "call", ())
    assert state["stream"].waits == 1
    assert array._free_slots == [slot] and array._parked_slots == []


@pytest.mark.parametrize("why", ["capturing", "failed wait"])
def test_a_slot_that_may_still_be_written_is_parked(slots, why):
    array, slot, state = slots
    state.update(capturing=why == "capturing", stream=_Stream(fail=True))
    with pytest.raises(RuntimeError, match="stream error"):
        array.fill_slot(array.take_slot(), lambda *a: 0, "call", ())
    assert array._free_slots == [] and array._parked_slots == [slot]
    assert state["stream"].waits == (1 if why == "capturing" else 2)


def test_reshape_counts_the_elements_of_the_dims_it_makes(rk):
    """The check is on the whole numbers that become the result's dims, whatever type they come in."""
    import torch
    from amdgpu_jl_amd import _lib as L
    x = rk.ROCArray(buf=torch.zeros(20, dtype=torch.uint8), dims=(5,), dtype=np.float32)
    assert x.reshape(5, 1).dims == x.reshape((np.int32(5), 1.0)).dims == (5, 1)
    for dims in ((2.5, 2), (4,), (5, 2)):
        with pytest.raises(L.DimensionMismatch):
            x.reshape(*dims)
    y = rk.ROCArray(buf=torch.zeros(16, dtype=torch.uint8), dims=(4,), dtype=np.float32)
    assert y.reshape(2.5, 2).dims == (2, 2)


@pytest.mark.parametrize("words,written,waits", [(1, [0], 0), (0b1101, [0, 2, 3], 0), (0b1101, [0, 3], 1), (1, [], 1), (0, [0], 1)])
def test_a_slot_is_read_when_its_words_are_there(slots, monkeypatch, words, written, waits):
    """The stream is waited for only if a word of the result is missing after the time that the words are waited for; words
    that are no part of the result, and what an earlier call has left, do not count."""
    array, slot, state = slots
    monkeypatch.setattr(array, "_WAIT_US", 50)
    slot[1][:] = 9

    def call(*args):
        for i in written:
            slot[1][8 * i] ^= 0xff                       # a byte of a word is enough
        return 0
    array.fill_slot(array.take_slot(), call, "call", (), words=words)
    assert state["stream"].waits == waits


def test_wait_words_sees_what_another_thread_writes(rk):
    import threading
    from amdgpu_jl_amd import _lib as L
    w = np.full(4, 5, dtype=np.uint64)
    later = threading.Timer(0.05, lambda: w.__setitem__(2, 6))
    later.start()
    assert L.lib.rk_wait_words(w.ctypes.data, 0b100, 5, 20_000_000) == 1          # (the interpreter is not held meanwhile)
    later.join()
    assert L.lib.rk_wait_words(w.ctypes.data, 0b110, 5, 1000) == 0
    assert L.lib.rk_wait_words(w.ctypes.data, 0, 5, 0) == 1 and L.lib.rk_wait_words(None, 1, 5, 0) == 1
