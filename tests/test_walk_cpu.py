"""The host walk (csrc/walk.cpp) where no GPU is needed."""
import struct

from lpmm import _native


def _program_header_types(path):
    with open(path, "rb") as f:
        head = f.read(64)
        assert head[:5] == b"\x7fELF\x02"
        offset, = struct.unpack_from("<Q", head, 32)
        size, count = struct.unpack_from("<HH", head, 54)
        f.seek(offset)
        table = f.read(size * count)
    return [struct.unpack_from("<I", table, i * size)[0] for i in range(count)]


def test_the_module_has_no_thread_local_storage():
    """PT_TLS: a module with thread-local storage that is loaded late slows down every thread-local access of the
    process, torch's own among them."""
    types = _program_header_types(_native.walk().__file__)
    assert 1 in types and 7 not in types  # PT_LOAD, PT_TLS
