"""Buffers set in one launch (mui_fill_buffers, muillm_ext.fill_buffers)."""
import pytest
import torch

from muillm_amd import _lib, muillm_ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 5, 64, 65, 130])
@pytest.mark.parametrize("words", [1, 2, 3, 1023, 1024, 70001])
def test_every_word_and_nothing_else(count, words):
    """Odd counts of words, buffers 16 bytes apart from a 16-byte boundary or 8, more buffers than one launch takes."""
    guard, room = 7, words + 9 + (words & 1)
    pool = torch.full((count * room + 2 * guard,), guard, dtype=torch.int64, device="cuda")
    views = [pool[guard + i * room + (i & 1):][:max(1, words - i % 3)] for i in range(count)]
    muillm_ext.fill_buffers(views, [-5 * (1 << 33) + i for i in range(count)])
    want = torch.full_like(pool, guard)
    for i, v in enumerate(views):
        want[v.storage_offset():v.storage_offset() + v.numel()] = -5 * (1 << 33) + i
    assert torch.equal(pool, want)


def test_what_the_kernel_does_not_take():
    odd = torch.ones(3, dtype=torch.float16, device="cuda")
    strided = torch.ones(4, 6, device="cuda")
    host, empty = torch.ones(5), torch.ones(0, device="cuda")
    whole = torch.ones(64, dtype=torch.bfloat16, device="cuda")
    muillm_ext.fill_buffers([odd, strided[:, :4], host, empty, whole])
    assert not odd.any() and not strided[:, :4].any() and strided[:, 4:].all() and not host.any() and not whole.any()
    muillm_ext.fill_buffers([strided], [3])
    assert bool((strided == 3).all())


def test_refused_arguments():
    import ctypes

    lib, t = _lib.load(), torch.zeros(4, dtype=torch.int64, device="cuda")
    one = lambda ty, v: (ty * 1)(v)
    call = lambda at, n, count=1: lib.mui_fill_buffers(0, count, one(ctypes.c_void_p, at), one(ctypes.c_size_t, n), one(ctypes.c_int64, 1))
    assert call(t.data_ptr() + 4, 8) == call(t.data_ptr(), 12) == _lib_alignment()
    assert call(None, 8) == call(t.data_ptr(), 8, -1) == -1
    assert call(t.data_ptr(), 0) == call(None, 0) == 0 and not t.any()


def _lib_alignment():
    return next(c for c in range(-1, -10, -1) if "align" in _lib.status_string(c))
