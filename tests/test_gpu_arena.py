"""A context's device memory (prg::Arena, by its symbols): what it holds beyond
the buffers in use, over buffers that grow."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


class _Arena:
    """An empty prg::Arena: its members are empty when all bytes are zero."""

    def __init__(self, prg):
        self.lib = prg.lib()
        self.at = C.create_string_buffer(512)
        self.take_ = self.lib._ZN3prg5Arena4takeEm
        self.take_.restype = C.c_void_p
        self.give_ = self.lib._ZN3prg5Arena4giveEPvm
        self.lib.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t)] * 2
        self.start = self.free()

    def take(self, n):
        return self.take_(self.at, C.c_size_t(n))

    def give(self, p, n):
        self.give_(self.at, C.c_void_p(p), C.c_size_t(n))

    def free(self):
        a, b = C.c_size_t(), C.c_size_t()
        assert self.lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    def held(self):
        return self.start - self.free()

    def close(self):
        self.lib._ZN3prg5ArenaD1Ev(self.at)


def test_outgrown_large_buffers_go_back(prg):
    """Eight buffers of 1 to 2.4 GiB, each outgrown in turn by a third: the
    memory held is that of the buffers in use (allocations round up to 2 MiB)."""
    a = _Arena(prg)
    sizes = [(1024 + 200 * k) * MIB + 512 * k for k in range(8)]
    live = [a.take(n) for n in sizes]
    for step in range(3):
        for k in range(len(sizes)):
            a.give(live[k], sizes[k])
            sizes[k] += sizes[k] // 3
            live[k] = a.take(sizes[k])
            held = a.held()
            assert held <= sum(sizes) + 2 * MIB * len(sizes), (step, k, held / MIB, sum(sizes) / MIB)
    for p, n in zip(live, sizes):
        a.give(p, n)
    assert a.held() <= 2 * MIB
    a.close()


def test_small_buffers_share_and_are_used_again(prg):
    """Buffers under the line share allocations; parts given back are handed
    out again, whole and apart from those in use."""
    a = _Arena(prg)
    sizes = [1, 511, 513, 3 * MIB + 7, 40 * MIB, 200 * MIB, 1000, 5]
    for _ in range(4):
        parts = [(a.take(n), n) for n in sizes]
        spans = sorted((p, p + n) for p, n in parts)
        assert all(p % 512 == 0 for p, _ in spans)
        assert all(e <= q for (_, e), (q, _) in zip(spans, spans[1:]))
        if _ == 0:
            held = a.held()
        assert a.held() == held
        for p, n in parts[::2] + parts[1::2]:
            a.give(p, n)
    a.close()
    assert a.held() <= 2 * MIB
