"""Decode kernels start on multiples of 64 KB in the built library, so that
their place in the instruction cache does not move with the other kernels."""
import struct

from zeromoe_amd import _lib

EM_AMDGPU = 224


def kernels(data):
    """(name, address) of the functions in every AMDGPU code object of the file."""
    at = data.find(b"\x7fELF\x02\x01", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU:
            shoff, = struct.unpack_from("<Q", data, at + 40)
            shentsize, shnum = struct.unpack_from("<HH", data, at + 58)
            sec = [struct.unpack_from("<IIQQQQIIQQ", data, at + shoff + i * shentsize) for i in range(shnum)]
            for s in sec:
                if s[1] != 11:  # SHT_DYNSYM
                    continue
                strs = at + sec[s[6]][4]
                for i in range(s[5] // s[9]):
                    name, info, _, _, value, _ = struct.unpack_from("<IBBHQQ", data, at + s[4] + i * s[9])
                    if info & 15 == 2:
                        yield data[strs + name:data.index(b"\0", strs + name)].decode(), value
        at = data.find(b"\x7fELF\x02\x01", at + 1)


def test_decode_kernels_start_on_64k():
    found = [k for k in kernels(open(_lib.LIB_PATH, "rb").read()) if "k_moe_decode" in k[0]]
    assert len(found) >= 30
    assert not [k for k in found if k[1] % 65536]
