"""What Device.dispatch hands to boot_dispatch: handles and offsets of every binding form, as the
ABI's arrays (CPU only: the native entries are replaced by a recorder)."""
import ctypes
import struct

import numpy as np
import pytest

from bootstrap_hip import HipError, KernelArgs
from bootstrap_hip.native import SIGNATURES, Binding, Device, GpuBuffer


@pytest.fixture
def recorder():
    calls = []

    def entry(name, result=1):
        def record(*arguments):
            calls.append((name, arguments))
            return result
        return record

    device = Device.__new__(Device)
    device.handle, device._context = 0x1000, ctypes.c_void_p(0x1000)
    device._entries = (entry("dispatch"), entry("noalloc"))
    device.calls, device.entry = calls, entry
    yield device
    device.handle = 0


def unpack(packed, count):
    return list(struct.unpack(f"{count}Q", packed))


@pytest.mark.parametrize("count", [0, 1, 11, 31, 40])
def test_bindings_are_packed_in_order(recorder, count):
    buffers = [GpuBuffer(recorder, 0x7f0000000000 + 16 * i, 1 << 20) for i in range(count)]
    recorder.dispatch("k", KernelArgs(M=3), 64, 256, *buffers)
    mixed = [b if i % 2 else b.at(i * 8) for i, b in enumerate(buffers)]
    recorder.dispatch2d("k2", KernelArgs(), 64, 2, 128, *mixed, noalloc=True)
    (first, a), (second, m) = recorder.calls
    assert (first, second) == ("dispatch", "noalloc")
    assert a[0].value == 0x1000 and a[1] == b"k" and m[1] == b"k2"
    assert unpack(a[2], count) == unpack(m[2], count) == [b.handle for b in buffers]
    assert a[3] is None or unpack(a[3], count) == [0] * count
    if count:
        assert unpack(m[3], count) == [0 if i % 2 else i * 8 for i in range(count)]
    assert a[4] == m[4] == count and a[6] == 64
    assert a[7:13] == (64, 1, 1, 256, 1, 1) and m[7:13] == (64, 2, 1, 128, 1, 1)
    assert a[13] is None and a[14].value == 0


@pytest.mark.parametrize("offset,expected", [(-4, 2 ** 64 - 4), (2 ** 64 + 8, 8), (np.int64(24), 24)])
def test_offsets_convert_as_uint64(recorder, offset, expected):
    buffer = GpuBuffer(recorder, 0x7f0000000000, 1 << 20)
    recorder.dispatch("k", KernelArgs(), 64, 256, buffer, Binding(buffer, offset))
    assert unpack(recorder.calls[0][1][3], 2) == [0, expected]


def test_a_failed_dispatch_raises_with_the_context_error(recorder):
    recorder._entries = (recorder.entry("dispatch", 0), None)

    class Lib:
        @staticmethod
        def boot_error(handle):
            return b"no such kernel"
    recorder.lib = Lib
    with pytest.raises(HipError, match="no such kernel"):
        recorder.dispatch("k", KernelArgs(), 64, 256)


@pytest.fixture
def native():
    """A device whose entries are C function pointers (into Python), typed and untyped as the library's."""
    device = Device.__new__(Device)
    device.handle, device._context, device.calls = 0x1000, ctypes.c_void_p(0x1000), []

    class Untyped(ctypes._CFuncPtr):
        _flags_, _restype_ = ctypes._FUNCFLAG_CDECL, ctypes.c_int

    class Lib:
        pass
    device.lib, device.kept, entries = Lib, [], []
    for name in ("boot_dispatch", "boot_dispatch_noalloc"):
        result, types = SIGNATURES[name]
        typed = ctypes.CFUNCTYPE(result, *types)(lambda *a, name=name: device.calls.append((name, a)) or 1)
        device.kept.append(typed)
        pointer = Untyped(ctypes.cast(typed, ctypes.c_void_p).value)
        entries.append(pointer)
        bound = Untyped(ctypes.cast(typed, ctypes.c_void_p).value)
        bound.argtypes = types
        setattr(Lib, name, staticmethod(bound))
    device._entries = tuple(entries)
    yield device
    device.handle = 0


@pytest.mark.parametrize("value,expected", [
    (64, 64), (np.int64(64), 64), (np.uint32(64), 64), (np.int32(64), 64), (True, 1), (0, 0), (2 ** 32 - 1, 2 ** 32 - 1),
    (-1, 2 ** 32 - 1), (2 ** 32 + 64, 64), (2 ** 70 + 64, 64), (ctypes.c_uint32(64), 64)])
def test_thread_counts_convert_as_uint32(native, value, expected):
    buffer = GpuBuffer(native, 0x7f0000000000, 1 << 20)
    native.dispatch("k", KernelArgs(), value, 256, buffer)
    native.dispatch("k", KernelArgs(), 64, value, buffer)
    native.dispatch2d("k", KernelArgs(), 64, value, 256, buffer.at(8), noalloc=True)
    assert [name for name, _ in native.calls] == ["boot_dispatch", "boot_dispatch", "boot_dispatch_noalloc"]
    assert [a[7:13] for _, a in native.calls] == [(expected, 1, 1, 256, 1, 1), (64, 1, 1, expected, 1, 1),
                                                  (64, expected, 1, 256, 1, 1)]
    assert all(a[0] == 0x1000 and a[1] == b"k" and a[4] == 1 and a[6] == 64 and a[13] is None and a[14] == 0
               for _, a in native.calls)


@pytest.mark.parametrize("value", [1.5, "64", None, ctypes.c_double(64.0), b"64"])
def test_thread_counts_of_other_types_are_refused(native, value):
    with pytest.raises(ctypes.ArgumentError):
        native.dispatch("k", KernelArgs(), value, 256)
    with pytest.raises(ctypes.ArgumentError):
        native.dispatch2d("k", KernelArgs(), 64, 1, value)
    assert native.calls == []


@pytest.mark.parametrize("noalloc,name", [(False, "boot_dispatch"), (None, "boot_dispatch"), (0, "boot_dispatch"),
                                          (True, "boot_dispatch_noalloc"), (2, "boot_dispatch_noalloc"),
                                          (np.bool_(True), "boot_dispatch_noalloc"), ("yes", "boot_dispatch_noalloc")])
def test_noalloc_takes_truth_values(native, noalloc, name):
    native.dispatch("k", KernelArgs(), 64, 256, noalloc=noalloc)
    assert [called for called, _ in native.calls] == [name]
