"""Host cost of a launch, read from the built library: a kernel that reads
gridDim or blockDim takes 14 hidden arguments (248 bytes) that the runtime
fills at every launch.  The dense GEMV, whose shortest calls the host bounds,
takes its grid size as an ordinary argument instead."""
import struct

import msgpack

import q4mi


def kernels(path):
    """{kernel symbol: argument kinds} of the gfx950 code objects in a
    library (clang offload bundles, the AMDGPU metadata note of each)."""
    data = open(path, "rb").read()
    magic, out, at = b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    while (at := data.find(magic, at)) >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            target, p = data[p + 24:p + 24 + idlen], p + 24 + idlen
            if b"gfx950" in target and size:
                for k in _metadata(data[at + off:at + off + size])["amdhsa.kernels"]:
                    out[k[".symbol"]] = [a[".value_kind"] for a in k[".args"]]
        at += len(magic)
    return out


def _metadata(elf):
    phoff, phsize, phnum = (struct.unpack_from("<Q", elf, 32)[0],
                            *struct.unpack_from("<HH", elf, 54))
    for i in range(phnum):
        kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phsize)
        if kind != 4:   # PT_NOTE
            continue
        p, end = off, off + size
        while p < end:
            nlen, dlen, ty = struct.unpack_from("<III", elf, p)
            d = p + 12 + (nlen + 3 & ~3)
            if elf[p + 12:p + 12 + 6] == b"AMDGPU" and ty == 32:
                return msgpack.unpackb(elf[d:d + dlen], strict_map_key=False)
            p = d + (dlen + 3 & ~3)
    raise AssertionError("no AMDGPU metadata note")


def test_gemv_kernels_take_no_hidden_arguments():
    gemv = {s: k for s, k in kernels(q4mi.LIB_PATH).items() if "mmvq_" in s}
    assert any("mmvq_u_k" in s for s in gemv) and any("mmvq_k" in s for s in gemv)
    assert not [s for s, k in gemv.items() if any(a.startswith("hidden_") for a in k)]
