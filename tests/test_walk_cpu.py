"""The host walk (csrc/walk.cpp) where no GPU is needed."""
import struct
import sys

import pytest
import torch

import lpmm
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


@pytest.mark.parametrize("group_size", [None, 0, 1 << 40])
def test_a_group_size_that_nothing_reads(group_size):
    """Rank-1 scales for both moments: the group size is not read, and may be anything."""
    p = torch.nn.Parameter(torch.zeros(70, 61))
    opt = lpmm.optim.AdamW([p], qconfig=dict(QUANT=dict(M=dict(SCALE_TYPE=dict(DEFAULT="rank1"), GROUP_SIZE=group_size),
                                                        SQM=dict(SCALE_TYPE=dict(DEFAULT="rank1")))))
    assert opt.step() is None
    assert lpmm.optim.adamw._Routes(*map(opt.get_qmetadata_by_state_name, ("exp_avg", "exp_avg_sq"))).m_group == 0


def test_steps_without_the_module(monkeypatch):
    """Where the module does not load (another version of torch or Python), one warning is given and the Python loops take
    every tensor: SGD on tensors in host memory, which needs no library at all."""
    monkeypatch.setattr(_native, "_walk", None)
    monkeypatch.setattr(lpmm, "_walk", None, raising=False)
    monkeypatch.delattr(lpmm, "_walk")
    monkeypatch.setitem(sys.modules, "lpmm._walk", None)
    p, q = (torch.nn.Parameter(torch.arange(1.0, 8.0)) for _ in range(2))
    ours, torchs = lpmm.optim.SGD([p], lr=0.1, momentum=0.9), torch.optim.SGD([q], lr=0.1, momentum=0.9)
    with pytest.warns(RuntimeWarning, match="_walk.so does not load") as warned:
        for step in range(3):
            p.grad, q.grad = torch.full((7,), 1.0 + step), torch.full((7,), 1.0 + step)
            ours.step()
            torchs.step()
    assert len(warned) == 1 and torch.allclose(p, q)
    assert lpmm.optim.AdamW([torch.nn.Parameter(torch.zeros(3))]).step() is None


def test_a_tensors_hash_is_its_address():
    """The walk looks states up with it (hash_of), and dictionaries keep what it is given."""
    for t in (torch.zeros(3), torch.nn.Parameter(torch.zeros(3)), torch.nn.Parameter(torch.zeros(0))):
        assert hash(t) == id(t)
