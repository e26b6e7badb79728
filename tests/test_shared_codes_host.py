"""Host logic of the activation codes that sibling projections share (no GPU):
``MixedLinear._prompt_forward`` against a stand-in for the foreign call, whose
"quantizer" writes the input's first value at the head of the codes and whose
"GEMM" writes the head of the codes it is given to the output's first value."""
from __future__ import annotations

import ctypes
from types import SimpleNamespace

import pytest
import torch

from test_host_logic import _cpu_pack
from tilequant_amd import mixed_linear as ml
from tilequant_amd.mixed_linear import MixedLinear

CFG = SimpleNamespace(dtype_out="bf16")
ROWS, COLS = 100, 192


class _Library:
    """Stands in for the foreign calls; ``before`` runs ahead of the launches
    and returns the call's code."""

    def __init__(self):
        self.quantized = []
        self.before = lambda: 0

    def tq_prompt_forward(self, ref):
        d = ref._obj
        rc = self.before()
        if rc:
            return rc
        self.quantized.append(bool(d.quantize))
        if d.quantize:
            ctypes.memmove(d.x_blocked, d.x, 2)
        ctypes.memmove(d.out, d.x_blocked, 2)
        return 0

    @staticmethod
    def tq_stream_capture_id(stream):
        return 0

    @staticmethod
    def tq_error_string(code):
        return b"forced by the test"


@pytest.fixture
def library(monkeypatch):
    lib = _Library()
    monkeypatch.setattr(ml.nat, "lib", lambda: lib)
    monkeypatch.setattr(ml.nat, "require_device", lambda *tensors: None)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 0)
    monkeypatch.setattr(ml, "_SHARED_QUANT", {})
    return lib


def _siblings(count=2):
    return [MixedLinear(_cpu_pack(128, COLS, 0.3, seed)[0], None, CFG) for seed in range(count)]


def _input(value):
    return torch.full((ROWS, COLS), float(value), dtype=torch.bfloat16)


def _call(lin, x):
    return float(lin._prompt_forward(x, x)[0, 0])


def test_siblings_share_one_quantization(library):
    a, b = _siblings()
    x = _input(2)
    with torch.inference_mode():
        assert [_call(a, x), _call(b, x), _call(a, x)] == [2, 2, 2]
    assert library.quantized == [True, False, True]      # a consumer asking twice starts a new pass


def test_codes_of_a_failed_call_are_not_shared(library, monkeypatch):
    a, b = _siblings()
    x = _input(3)
    with torch.inference_mode():
        library.before = lambda: 2
        with pytest.raises(RuntimeError, match="forced"):
            _call(a, x)
        library.before = lambda: 0
        assert _call(b, x) == 3

        real = torch.empty

        def no_room_for_the_output(size, *args, **kwargs):
            if tuple(size) == (ROWS, 128):
                raise torch.OutOfMemoryError("forced by the test")
            return real(size, *args, **kwargs)

        y = _input(4)
        monkeypatch.setattr(torch, "empty", no_room_for_the_output)
        with pytest.raises(torch.OutOfMemoryError):
            _call(a, y)
        monkeypatch.setattr(torch, "empty", real)
        assert _call(b, y) == 4
    assert library.quantized == [True, True]


def test_codes_are_not_shared_before_their_launch(library):
    """A second thread on the same stream, with the same input, while the first
    is inside the foreign call and has launched nothing yet."""
    a, b = _siblings()
    x, seen = _input(5), []

    def other_thread():
        library.before = lambda: 0
        seen.append(_call(b, x))
        return 0

    with torch.inference_mode():
        library.before = other_thread
        assert _call(a, x) == 5
    assert seen == [5] and library.quantized == [True, True]


@pytest.mark.parametrize("inside", [True, False])
def test_an_input_changed_in_place_is_quantized_again(library, inside):
    """Tensors made under inference mode have no version counter: an in-place
    change between two siblings cannot be seen, so their codes are not shared."""
    a, b = _siblings()
    with torch.inference_mode(inside):
        x = _input(2)
    with torch.inference_mode():
        assert x.is_inference() == inside
        assert _call(a, x) == 2
        x.mul_(2)
        assert _call(b, x) == 4
    assert library.quantized == [True, True]


def test_codes_do_not_cross_a_graph_capture(library, monkeypatch):
    """Codes of an eager call are not taken inside a capture (its graph would
    hold no quantization), nor those of a capture outside it or in another
    one (its launches are only recorded); siblings of one capture share."""
    now = [0]
    monkeypatch.setattr(ml.nat, "capture_id", lambda stream: now[0])
    a, b = _siblings()
    with torch.inference_mode():
        for first, second in ((0, 7), (7, 0), (7, 9), (7, 7), (None, None)):
            with torch.inference_mode(False):
                x = _input(2)
            library.quantized.clear()
            now[0] = first
            _call(a, x)
            now[0] = second
            _call(b, x)
            assert library.quantized == [True, first != second or first is None], (first, second)


def test_group_outputs_do_not_cross_a_graph_capture(library, monkeypatch):
    now, calls = [0], []
    monkeypatch.setattr(ml.nat, "capture_id", lambda stream: now[0])
    group = ml.MixedLinearGroup(_siblings())
    group.linear.forward = lambda x: calls.append(now[0]) or torch.zeros(ROWS, 256)
    x = _input(2)
    for first, second, want in ((0, 0, [0]), (0, 7, [0, 7]), (7, 0, [7, 0]), (7, 9, [7, 9]), (7, 7, [7]),
                                (None, None, [None, None])):
        calls.clear()
        group.reset_pending()
        now[0] = first
        group.output_for(x, 0)
        now[0] = second
        group.output_for(x, 1)
        assert calls == want


def test_a_lookup_never_returns_another_inputs_value():
    """Threads on one stream share a memo: another thread's put between a
    lookup's checks and its result must not reach the lookup's caller."""
    memo, x, other = ml.ServeOnce(), torch.zeros(2), torch.ones(2)

    class Key:
        def __eq__(self, rhs):
            memo.put(other, "key of the other", "a", "codes of the other")
            return True

        def __ne__(self, rhs):
            return not self == rhs

    memo.put(x, Key(), "a", "codes of x")
    assert memo.take(x, "key", "b") in (None, "codes of x")
    memo.put(x, "key", "a", "codes of x")
    assert memo.take(x, "key", "b") == "codes of x"


def test_a_memo_copies_empty():
    import copy
    import pickle

    memo, x = ml.ServeOnce(consumers=3), torch.zeros(2)
    memo.put(x, "key", "a", "codes of x")
    for other in (copy.deepcopy(memo), pickle.loads(pickle.dumps(memo))):
        assert other.consumers == 3 and other.take(x, "key", "b") is None
    # as modules saved by earlier versions hold it: one state entry per field
    old = ml.ServeOnce.__new__(ml.ServeOnce)
    old.__setstate__((None, {"consumers": 2, "_source": None, "_key": None, "_taken": frozenset(), "_value": None}))
    assert old.consumers == 2 and old.take(x, "key", "b") is None
    assert memo.take(x, "key", "b") == "codes of x"


def test_an_outgrown_absmax_workspace_stays_alive(monkeypatch):
    """A captured graph holds the partial-max workspace by address: a larger
    input replaces the buffer, the old one is kept."""
    import gc
    import weakref

    from tilequant_amd import quantize_activation as qa

    need = [100]
    monkeypatch.setattr(qa.nat, "lib", lambda: SimpleNamespace(tq_act_absmax_workspace_elems=lambda n, k: need[0]))
    monkeypatch.setattr(qa.nat, "stream_handle", lambda device: 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(qa, "_WORKSPACE", {})
    monkeypatch.setattr(qa, "_RETIRED", [], raising=False)
    x = torch.zeros(2, 64)
    first = qa._absmax_workspace(x, 600, 64)
    assert qa._absmax_workspace(x, 600, 64) is first
    need[0], alive = first.numel() + 1, weakref.ref(first)
    del first
    assert qa._absmax_workspace(x, 20000, 64).numel() >= need[0]
    gc.collect()
    assert alive() is not None
