"""A __shared__ array that is read or written as wider vectors has their alignment by its declaration (its element type or
__align__), not by where the compiler happens to put it: a misaligned 16-byte LDS access is wrong or faults.  Source only."""
import glob
import os
import re

import pytest

from frink_amd import build as fb

SIZES = {"uint8_t": 1, "int8_t": 1, "uint16_t": 2, "int16_t": 2, "_Float16": 2, "int": 4, "int32_t": 4, "uint32_t": 4, "float": 4, "int64_t": 8, "uint64_t": 8,
         "int2": 8, "uint2": 8, "float2": 8, "v2i": 8, "v2f": 8, "u2_t": 8, "int4": 16, "uint4": 16, "float4": 16, "v4i": 16, "v4f": 16, "u4_t": 16, "xv_t": 16}
DECLARED = re.compile(r"__shared__\s+(?:__align__\((\d+)\)\s*)?(?:const\s+)?(\w+)\s+([^;=]+);")
CAST = re.compile(r"reinterpret_cast<\s*(?:const\s+)?(\w+)\s*\*\s*(?:const\s*)?>\(\s*&?(\w+)")


def misaligned(text):
    """(array, its alignment, the type it is accessed as) of every cast to something wider than the declaration promises."""
    aligned = {}
    for align, kind, names in DECLARED.findall(text):
        if kind not in SIZES and not align:
            continue
        for name in re.findall(r"(\w+)\s*(?:\[[^\]]*\]\s*)*(?:,|$)", names.strip()):
            aligned[name] = max(int(align or 1), SIZES.get(kind, 1))
    return [(name, aligned[name], kind) for kind, name in CAST.findall(text) if name in aligned and SIZES.get(kind, 1) > aligned[name]]


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(fb.CSRC, "*.h*"))), ids=os.path.basename)
def test_vector_accesses_of_shared_arrays(path):
    assert misaligned(open(path).read()) == []


def test_vector_accesses_of_the_quantizers_record():
    """Q8KRecordLds, a shared structure: the members that its users read as wider vectors."""
    text = open(os.path.join(fb.CSRC, "frk_device.hpp")).read()
    members = re.findall(r"(?:alignas\((\d+)\) )?(\w+) (\w+)\[\d+\];", re.search(r"struct Q8KRecordLds \{(.*?)\};", text, re.S).group(1))
    aligned = {name: max(int(align or 1), SIZES[kind]) for align, kind, name in members}
    read = re.findall(r"reinterpret_cast<const (\w+) \*>\(L\.(\w+)\)", text)
    assert len(aligned) == 3 and read
    assert [(name, aligned[name], kind) for kind, name in read if SIZES[kind] > aligned[name]] == []


def test_the_check_sees_a_float_array_read_as_float4():
    kernel = "__shared__ %sfloat a[3], b[32], c[8];\n f = reinterpret_cast<const float4 *>(b)[t];"
    assert misaligned(kernel % "") == [("b", 4, "float4")]
    assert misaligned(kernel % "__align__(16) ") == []
