"""The built gfx950 code: what the kernels rely on that no output shows."""
import os
import re
import struct
import subprocess

import pytest

import dance_amd as D

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects():
    """The gfx950 code objects in the library's offload bundles."""
    blob = open(D.LIB_PATH, "rb").read()
    magic, at, out = b"__CLANG_OFFLOAD_BUNDLE__", 0, []
    while (at := blob.find(magic, at)) >= 0:
        (count,), p = struct.unpack_from("<Q", blob, at + 24), at + 32
        for _ in range(count if count < 16 else 0):
            off, size, n = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + n]:
                out.append(blob[at + off:at + off + size])
            p += 24 + n
        at += len(magic)
    return out


@pytest.fixture(scope="module")
def notes(tmp_path_factory):
    if not os.path.exists(READELF) or not os.path.exists(D.LIB_PATH):
        pytest.skip("needs the built library and llvm-readelf")
    objs = code_objects()
    assert objs
    text = ""
    for i, o in enumerate(objs):
        path = tmp_path_factory.mktemp("co") / f"{i}.co"
        path.write_bytes(o)
        text += subprocess.run([READELF, "--notes", "--symbols", str(path)], check=True, capture_output=True,
                               text=True).stdout
    return text


def kernels(notes, field):
    """A metadata field of every kernel, by its mangled name."""
    out = {}
    for block in notes.split("  - .agpr_count")[1:]:
        block = block[:block.find(".wavefront_size")]
        out[re.search(r"\.name:\s+(_Z\S+)", block).group(1)] = int(re.search(rf"\.{field}:\s+(\d+)", block).group(1))
    return out


def test_search_state_is_not_in_scratch(notes):
    """A search kernel keeps its wave's state in registers. A variant whose body is
    not inlined keeps it in scratch (over 400 bytes a lane), and the values
    that the code takes for uniform are then spilled under lane masks."""
    sizes = kernels(notes, "private_segment_fixed_size")
    search = {k: v for k, v in sizes.items() if "k_search" in k}
    assert len(search) > 50
    assert {k: v for k, v in search.items() if v > 32} == {}


def test_every_device_function_is_inlined(notes):
    functions = {m.group(1) for m in re.finditer(r" FUNC\s+\S+\s+\S+\s+\S+\s+(\S+)", notes)}
    names = set(kernels(notes, "vgpr_count"))
    assert names and functions - names == set()


@pytest.mark.parametrize("kernel,waves", [("5k_rowILi1ELi1E", 8), ("5k_rowILi1ELi2E", 8), ("5k_rowILi1ELi3E", 7),
                                          ("5k_rowILi1ELi4E", 5), ("5k_csrILi1ELi2E", 7), ("5k_csrILi1ELi3E", 5),
                                          ("5k_csrILi1ELi4E", 4)])
def test_filtered_uint8_kernels_keep_their_waves(notes, kernel, waves):
    """The Gram tiles of the filtered prune do not take the searches' waves (per SIMD, by registers)."""
    counts = [v for k, v in kernels(notes, "vgpr_count").items() if kernel in k]
    assert len(counts) == 1
    assert 512 // (-(-counts[0] // 8) * 8) >= waves


def test_prune_kernels_hardly_spill(notes):
    """Registers spilled around lane masks are reloaded under the wrong one; what is
    left holds a few addresses (36 bytes)."""
    sizes = {k: v for k, v in kernels(notes, "private_segment_fixed_size").items() if "k_prune" in k}
    assert len(sizes) > 20
    assert {k: v for k, v in sizes.items() if v > 40} == {}
