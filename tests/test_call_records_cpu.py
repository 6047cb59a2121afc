"""The packed records that the Python wrappers hand over as bytes, against the C header's structs: every field in its place."""
import ctypes
import os
import re
import struct
import subprocess

import pytest

from singe_amd import _native, error

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "singe_hip_attention.h")
RECORDS = {"SingePagedAttentionCall": _native.PAGED_ATTENTION_CALL, "SingeRotaryCacheCall": _native.ROTARY_CACHE_CALL}


def members(name):
    """The struct's members in the header, its problem's in the place of `problem`."""
    body = re.search(r"typedef struct %s \{(.*?)\} %s;" % (name, name), open(HEADER).read(), re.S).group(1)
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    found = []
    for kind, member in re.findall(r"([A-Za-z_][\w ]*?[\w*]\s*\**)\s*\b(\w+);", body):
        found += ["problem." + inner for inner in members(kind.strip())] if member == "problem" else [member]
    return found


def packed_offsets(format_):
    """Where a native format string has its items, and its size."""
    assert format_[0] == "@"
    codes = "".join(code * int(count or 1) for count, code in re.findall(r"(\d*)([A-Za-z])", format_[1:]))
    return [struct.calcsize("@" + codes[:i + 1]) - struct.calcsize("@" + codes[i]) for i in range(len(codes))], struct.calcsize(format_)


@pytest.mark.parametrize("name", RECORDS)
def test_every_field_lies_where_the_header_has_it(name, tmp_path):
    fields = members(name)
    lines = "".join(f'    printf("%zu %zu\\n", offsetof({name}, {field}), sizeof((({name}*)0)->{field}));\n' for field in fields)
    source, program = tmp_path / "record.c", tmp_path / "record"
    source.write_text(f'#include <stddef.h>\n#include <stdio.h>\n#include "singe_hip_attention.h"\nint main(void) {{\n{lines}'
                      f'    printf("%zu\\n", sizeof({name}));\n    return 0;\n}}\n')
    subprocess.run(["gcc", "-I", os.path.dirname(HEADER), str(source), "-o", str(program)], check=True)
    found = [[int(number) for number in line.split()] for line in subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.splitlines()]
    offsets, size = packed_offsets(RECORDS[name].format)
    assert len(offsets) == len(fields)
    assert [offset for offset, _ in found[:-1]] == offsets
    codes = "".join(code * int(count or 1) for count, code in re.findall(r"(\d*)([A-Za-z])", RECORDS[name].format[1:]))
    assert [width for _, width in found[:-1]] == [struct.calcsize(code) for code in codes]
    assert size <= found[-1][0] and found[-1][0] - size < 8  # (a struct may end in padding, which nobody reads)
    assert struct.calcsize("@" + RECORDS[name].format[1:] + "0q") == found[-1][0]


def test_a_record_that_asks_for_more_scratch_than_it_lends_is_told_how_much():
    lib = _native.lib()
    fields = (1, 32, 8, 128, 16, 1, 4096, 2000, 1, 1, 0, 0, 0, 0.0, 0.0, 0)
    wanted = lib.singe_hip_paged_attention_scratch_bytes(ctypes.byref(_native.PagedAttentionProblemC(*fields)))
    assert wanted > 0
    pack = lambda count, asks: _native.PAGED_ATTENTION_CALL.pack(_native.DATA_TYPE_BF16, 0, *[0x1000] * 10, 0x1000, count, asks, *fields)
    assert lib.singe_hip_paged_attention_every_row_call(pack(wanted - 1, 1)) == _native.LENGTH_TOO_SHORT
    with pytest.raises(error.LengthTooShort, match=str(wanted)):
        _native.check(_native.LENGTH_TOO_SHORT)


def test_no_record_is_refused():
    lib = _native.lib()
    assert lib.singe_hip_paged_attention_every_row_call(None) == lib.singe_hip_rotary_cache_write_call(None) != 0
