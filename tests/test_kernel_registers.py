"""How many registers the built kernels take, which decides how many waves a SIMD holds (here without a GPU: the libraries carry
the numbers with the code that was compiled from the sources here)."""
import shutil
import struct

import pytest

from llm_inference_lab_amd.kernels import build

msgpack = pytest.importorskip("msgpack")
SIMD_REGISTERS = 512          # of a lane; gfx950 hands them out by 8


def kernels(path):
    """``{mangled name: (registers, spilled)}`` of the gfx950 code in a library."""
    data, found, at = open(path, "rb").read(), {}, 1
    while (at := data.find(b"\x7fELF", at)) > 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:          # an AMD GPU's
            offset, size, count = (struct.unpack_from("<Q", data, at + 32)[0], *struct.unpack_from("<HH", data, at + 54))
            for header in range(at + offset, at + offset + size * count, size):
                kind, _, start = struct.unpack_from("<IIQ", data, header)
                length = struct.unpack_from("<Q", data, header + 32)[0]
                if kind != 4:                                          # (notes)
                    continue
                note = at + start
                while note < at + start + length:
                    name, text, what = struct.unpack_from("<III", data, note)
                    body = note + 12 + (name + 3) // 4 * 4
                    if what == 32:
                        for k in msgpack.unpackb(data[body:body + text])["amdhsa.kernels"]:
                            found[k[".name"]] = (k[".vgpr_count"], k.get(".vgpr_spill_count", 0))
                    note = body + (text + 3) // 4 * 4
        at += 4
    return found


def library(make):
    if shutil.which("hipcc") is None and not build.hipcc_path():
        pytest.skip("no hipcc to build the library with")
    return make()


@pytest.mark.parametrize("make,kernel,waves,least", [
    (lambda: build.mixer_library("linear_attention"), "chunk_finish_kernel", 2, 24),
    (lambda: build.attention_library(64), "attention_rows_kernel", 2, 4),
    (lambda: build.attention_library(128), "attention_rows_kernel", 2, 3),
])
def test_waves_a_simd_holds(make, kernel, waves, least):
    """As many waves a SIMD as the kernels' notes count on, and nothing spilled."""
    taken = {name: v for name, v in kernels(library(make)).items() if kernel in name}
    assert len(taken) >= least
    for name, (registers, spilled) in taken.items():
        assert spilled == 0 and SIMD_REGISTERS // (-(-registers // 8) * 8) >= waves, (name, registers, spilled)
