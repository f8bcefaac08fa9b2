"""The torch-level call over device sizes, without a GPU: the host side of _call_device with the library
and the stream replaced by stand-ins on the CPU."""
import types

import pytest
import torch


class _Stream:
    cuda_stream = 0

    def __init__(self):
        self.waits = 0

    def synchronize(self):
        self.waits += 1


def _run(pkg, monkeypatch, call):
    """_call_device over CPU tensors with `call` as gg_call_device_lens; returns the stream."""
    stream, pinned, empty = _Stream(), [], torch.empty

    def empty_without_pinning(*shape, pin_memory=False, **kw):
        t = empty(*shape, **kw)
        if pin_memory:
            pinned.append(t)
        return t

    lib = types.SimpleNamespace(gg_call_device_lens=call, gg_check_status=lambda p: pkg.GG_OK)
    monkeypatch.setattr(pkg, "load_library", lambda: lib)
    monkeypatch.setattr(pkg, "last_error", lambda: "refused")
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *_: stream)
    monkeypatch.setattr(torch, "empty", empty_without_pinning)
    cpu = {"device": "cpu"}
    x, w, out = torch.zeros((4, 8), **cpu), torch.zeros((1, 8, 8), **cpu), torch.zeros((4, 8), **cpu)
    try:
        pkg._call_device(pkg.OP_FORWARD, pkg.DType.BF16, pkg.DType.BF16, 8, 8, torch.tensor([4], **cpu), None, 4, x, w, out)
    finally:
        assert [t.device.type for t in pinned] == ["cpu"]
    return stream


def test_waits_once_before_the_status_is_read(pkg, monkeypatch):
    assert _run(pkg, monkeypatch, lambda *a: pkg.GG_OK).waits == 1


@pytest.mark.parametrize("failure", ["status", "interrupt"])
def test_a_failing_call_waits_before_its_status_is_freed(pkg, monkeypatch, failure):
    """A kernel that the call enqueued before it failed still writes the pinned status: the stream is waited
    for before the status goes back to torch's host allocator, which would give it to the next caller."""
    stream = []

    def call(*a):
        stream.append(torch.cuda.current_stream())
        if failure == "interrupt":
            raise KeyboardInterrupt
        return pkg.GG_ERR_HIP

    with pytest.raises(KeyboardInterrupt if failure == "interrupt" else pkg.GGError):
        _run(pkg, monkeypatch, call)
    assert stream[0].waits == 1


def test_status_is_host_memory_whatever_the_default_device(pkg, monkeypatch):
    with torch.device("meta"):
        torch.empty(1)  # torch lists the functions that take a default device on first use: before the stand-ins
        assert _run(pkg, monkeypatch, lambda *a: pkg.GG_OK).waits == 1
