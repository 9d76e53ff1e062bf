"""gw_run_noalloc makes no HIP allocation: the entries of the library's own jump
table for the allocating calls are replaced by ones that count, in a context
whose pinned buffers no other run has filled. Cells of one and of several pieces;
the records are gw_run's."""
import ctypes as C
import struct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CALLS = ("hipMalloc", "hipHostMalloc", "hipFree", "hipHostFree", "hipEventCreate", "hipEventCreateWithFlags",
         "hipStreamCreateWithFlags")


def _jump_slots(path):
    """{symbol: offset of its jump slot} of an ELF64 library, from its section .rela.plt."""
    data = open(path, "rb").read()
    shoff, = struct.unpack_from("<Q", data, 0x28)
    shentsize, shnum, shstrndx = struct.unpack_from("<HHH", data, 0x3A)
    sections = [struct.unpack_from("<IIQQQQIIQQ", data, shoff + k * shentsize) for k in range(shnum)]
    names = sections[shstrndx][4]
    by_name = {data[names + s[0]:data.index(b"\0", names + s[0])].decode(): s for s in sections}
    sym, strs, rela = by_name[".dynsym"][4], by_name[".dynstr"][4], by_name[".rela.plt"]
    out = {}
    for at in range(rela[4], rela[4] + rela[5], 24):
        offset, info, _ = struct.unpack_from("<QQq", data, at)
        name = strs + struct.unpack_from("<I", data, sym + 24 * (info >> 32))[0]
        out[data[name:data.index(b"\0", name)].decode()] = offset
    return out


class _Counted:
    """While open, counts the library's calls of CALLS by name."""

    def __init__(self, path):
        base = min(int(ln.split("-")[0], 16) for ln in open("/proc/self/maps") if ln.rstrip().endswith(path))
        slots = _jump_slots(path)
        self.count, self.keep = {}, []
        for name in CALLS:
            slot = C.c_uint64.from_address(base + slots[name])
            real = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_size_t, C.c_uint)(slot.value)

            def counted(a, b, c, name=name, real=real):
                self.count[name] = self.count.get(name, 0) + 1
                return real(a, b, c)

            fn = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_size_t, C.c_uint)(counted)
            self.keep.append((slot, slot.value, fn))

    def __enter__(self):
        self.count.clear()
        for slot, _, fn in self.keep:
            slot.value = C.cast(fn, C.c_void_p).value
        return self.count

    def __exit__(self, *_):
        for slot, real, _ in self.keep:
            slot.value = real


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32_local"])
@pytest.mark.parametrize("n", [50, 16_384, 16_385, 70_001])
def test_a_run_without_allocations(gwcapi, precision, n):
    ctx = gwcapi.Context(0)
    counted = _Counted(gwcapi.LIB_PATH)
    p, crus, ist = gwcapi.Params.default(), gwcapi.rest_state(n, 4), np.full(60, 100.0)
    args = (ctx, p, n, 1e-3, 60, ist, 20, None, crus, 5, 0, precision)
    with counted as count:
        got = [gwcapi.run(*args, noalloc=True) for _ in range(2)]
        assert count == {}
        want = gwcapi.run(*args)
        assert count["hipMalloc"] == 1 and count["hipFree"] == 1
    for k, v in want.items():
        for g in got:
            assert np.array_equal(g[k], v), k
    ctx.close()
