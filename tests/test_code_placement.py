"""The code object inside libbrik.so has its .text at the address that the build asks for, whatever the metadata
before it takes (build.py, TEXT_ADDR): where the decode kernels lie moves a decoder layer by 1 %."""
import struct

from brimkern_amd import build, capi


def test_text_address():
    blob = open(capi.LIB_PATH, "rb").read()
    at = blob.index(b"\x7fELF", 4096)               # the embedded code object, after the library's own header
    elf = blob[at:]
    assert struct.unpack_from("<H", elf, 18)[0] == 224          # EM_AMDGPU
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum, shstrndx = struct.unpack_from("<HHH", elf, 58)
    sections = [struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize) for i in range(shnum)]
    names = sections[shstrndx][4]
    address = {elf[names + s[0]:elf.index(b"\0", names + s[0])].decode(): s[3] for s in sections}
    assert address[".text"] == build.TEXT_ADDR
