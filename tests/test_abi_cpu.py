"""No-GPU checks of the C-ABI library and the host layer: the library loads, exports every symbol the
header declares, and every validation that the reference performs before a launch returns the same
error without touching a device."""
import ctypes
import os
import re
import subprocess

import pytest

from singe_amd import _native, error
from singe_amd.kernel import attention as A

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "singe_hip_attention.h")).read()
    return sorted(set(re.findall(r"SINGE_HIP_API[^;(]*?\b(singe_hip_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _native.lib()
    names = declared_symbols()
    assert len(names) >= 20
    for name in names:
        assert hasattr(lib, name), name


def test_code_object_is_built_and_every_part_names_its_kernels():
    images = {}
    for part, path in zip(_native.CODE_OBJECT_PARTS, _native.CODE_OBJECT_PATHS):
        assert os.path.exists(path), path
        images[part] = open(path, "rb").read()
    lib, names = _native.lib(), []
    name, part = ctypes.c_char_p(), ctypes.c_char_p()
    index = 0
    while lib.singe_hip_kernel(index, ctypes.byref(name), ctypes.byref(part)) == 0:
        assert name.value in images[part.value.decode()], (name.value, part.value)
        names.append(name.value)
        index += 1
    assert len(names) == len(set(names)) >= 113
    for kernel in (b"singe_paged_decode_bf16_d128_g1_b16", b"singe_paged_decode_f8kv_wide_d128_b16",
                   b"singe_paged_decode_combine_bf16", b"singe_fmha_prefill_bf16_d128_causal",
                   b"singe_fmha_prefill_f32_d64", b"singe_paged_attention_bf16_d128_i64", b"singe_paged_attention_bf16_d128_i32_p16",
                   b"singe_paged_kv_prefill_bf16_d128_p16", b"singe_rotary_paged_attention_bf16_d128_i64_p16"):
        assert kernel in names, kernel


def test_status_strings():
    lib = _native.lib()
    assert lib.singe_hip_status_string(0) == b"ok"
    assert lib.singe_hip_status_string(1) == b"invalid length"
    assert lib.singe_hip_status_string(2) == b"length too short"


GOOD = dict(batch=2, heads=8, kv_heads=2, head_dim=128, block_size=16, physical_blocks=8,
            block_table_batch_stride=4, scale=0.1)


def decode_status(config, lens=None, pointers=None):
    lens = lens or dict(out=2 * 8 * 128, query=2 * 8 * 128, key=8 * 16 * 2 * 128, value=8 * 16 * 2 * 128, seq=2, table=8)
    fake = 0x1000
    p = pointers or {}
    return _native.lib().singe_hip_paged_kv_decode_attention_bf16(
        None, p.get("out", fake), lens["out"], p.get("query", fake), lens["query"], p.get("key", fake), lens["key"],
        p.get("value", fake), lens["value"], p.get("seq", fake), lens["seq"], p.get("table", fake), lens["table"],
        p.get("workspace", fake), 1 << 30, ctypes.byref(config))


def test_decode_validation_order_and_codes():
    # validate_paged_kv_decode_attention_config, then validate_lengths (mod.rs:711-743, 2963-2985)
    for bad in (dict(batch=0), dict(heads=7), dict(scale=float("inf")), dict(physical_blocks=0)):
        with pytest.raises(error.InvalidLength):
            A.PagedKvDecodeAttentionConfig.contiguous(**{**GOOD, **bad})
        c = A.PagedKvDecodeAttentionConfig(**{**GOOD, **bad})._c()
        assert decode_status(c) == 1
    with pytest.raises(error.LengthExceedsI32):
        A.PagedKvDecodeAttentionConfig.contiguous(**{**GOOD, "batch": 2**31})
    assert decode_status(A.PagedKvDecodeAttentionConfig(**{**GOOD, "batch": 2**31})._c()) == 3
    c = A.PagedKvDecodeAttentionConfig.contiguous(**GOOD)._c()
    full = dict(out=2 * 8 * 128, query=2 * 8 * 128, key=8 * 16 * 2 * 128, value=8 * 16 * 2 * 128, seq=2, table=8)
    for name in full:
        status = decode_status(c, {**full, name: full[name] - 1})
        assert status == 2, name
        detail = _native.ErrorDetail()
        _native.lib().singe_hip_last_error(ctypes.byref(detail))
        assert detail.minimum == full[name] and detail.actual == full[name] - 1
    assert decode_status(c, pointers=dict(query=None)) == 6
    big = 1 << 30  # buffers long enough for any width: head dimensions past 256 have no kernel at all
    wide = dict(out=big, query=big, key=big, value=big, seq=2, table=8)
    assert decode_status(A.PagedKvDecodeAttentionConfig(**{**GOOD, "head_dim": 320})._c(), wide) == 5
    with pytest.raises(error.UnsupportedWidth):
        _native.check(5, "paged_kv_decode_attention_bf16")


def test_decode_workspace_query_needs_no_device():
    c = A.PagedKvDecodeAttentionConfig.contiguous(**GOOD)
    assert c.workspace_bytes() > 0
    assert _native.lib().singe_hip_paged_kv_decode_attention_workspace_bytes(None) == 0


def test_fmha_config_validation():
    good = A.FmhaPrefillConfig.contiguous(1, 64, 64, 4, 2, 128, 0.1, True)
    lib = _native.lib()
    assert lib.singe_hip_fmha_prefill_config_validate(ctypes.byref(good._c())) == 0
    from dataclasses import replace
    for bad in (replace(good, key_len=0), replace(good, kv_heads=3), replace(good, scale=float("nan")),
                replace(good, query_head_stride=0)):
        assert lib.singe_hip_fmha_prefill_config_validate(ctypes.byref(bad._c())) == 1
    # validate_lengths: a buffer shorter than the strides can reach
    fake = 0x1000
    need = 64 * 4 * 128
    status = lib.singe_hip_fmha_prefill_bf16(None, fake, need, fake, need - 1, fake, 64 * 2 * 128, fake, 64 * 2 * 128,
                                             ctypes.byref(good._c()))
    assert status == 2
    assert lib.singe_hip_fmha_prefill_bf16(None, fake, need, fake, need, None, 64 * 2 * 128, fake, 64 * 2 * 128,
                                           ctypes.byref(good._c())) == 6


def test_paged_attention_problem_validation():
    lib = _native.lib()
    fake = 0x1000
    def call(**changes):
        fields = dict(tokens=2, heads=2, kv_heads=2, head_dim=128, page_size=4, sequences=1, cache_pages=2, page_table=1,
                      index_type=1, causal=1, has_scale=0, has_window=0, has_softcap=0, scale=0.0, softcap=0.0, window=0)
        fields.update(changes)
        problem = _native.PagedAttentionProblemC(*fields.values())
        return lib.singe_hip_paged_attention_bf16(None, *([fake] * 10), ctypes.byref(problem))
    assert call(kv_heads=0) == 9
    assert call(heads=3) == 9
    assert call(page_size=0) == 9
    assert call(index_type=7) == 9
    assert call(head_dim=300) == 5  # beyond the general kernel's 256
    detail = _native.ErrorDetail()
    lib.singe_hip_last_error(ctypes.byref(detail))
    assert detail.minimum == 300  # the refused width
    assert call(tokens=0) == 0  # nothing to attend, nothing launched


def test_rotary_paged_attention_validation():
    lib = _native.lib()
    fake = 0x1000
    def call(rotation, cos=fake, **changes):
        fields = dict(tokens=2, heads=2, kv_heads=2, head_dim=128, page_size=4, sequences=1, cache_pages=2, page_table=1,
                      index_type=1, causal=1, has_scale=0, has_window=0, has_softcap=0, scale=0.0, softcap=0.0, window=0)
        fields.update(changes)
        problem = _native.PagedAttentionProblemC(*fields.values())
        return lib.singe_hip_rotary_paged_attention_bf16(None, *([fake] * 7), cos, fake, None, fake, None, None, ctypes.byref(problem),
                                                         None if rotation is None else ctypes.byref(rotation))
    good = _native.QueryRotationC(0, 1, 1e-5)
    assert call(None) == 6                                       # no rotation attributes
    assert call(_native.QueryRotationC(7, 0, 0.0)) == 9          # unknown table type
    assert call(good, head_dim=72) == 5                          # the fused form takes the multiples of 16 up to 128
    assert call(good, head_dim=144) == 5 and call(good, head_dim=8) == 5
    assert call(good, has_softcap=1, softcap=float("nan")) == 9  # a cap is taken; a cap that is no number is not
    assert call(good, cos=None) == 6
    assert call(good, tokens=0) == 0
    assert call(good, tokens=0, head_dim=80, has_softcap=1, softcap=5.0) == 0


def test_paged_attention_scratch_query_needs_no_device():
    lib = _native.lib()
    def wanted(**changes):
        fields = dict(tokens=32, heads=32, kv_heads=8, head_dim=128, page_size=16, sequences=32, cache_pages=100, page_table=100,
                      index_type=0, causal=1, has_scale=0, has_window=0, has_softcap=0, scale=0.0, softcap=0.0, window=0)
        fields.update(changes)
        return lib.singe_hip_paged_attention_scratch_bytes(ctypes.byref(_native.PagedAttentionProblemC(*fields.values())))
    lib.singe_hip_set_paged_attention_splits(4)
    try:
        assert wanted() == 4 * 32 * 32 * 129 * 4     # shares x rows x (128 values + a log-sum-exp) of f32
        assert wanted(head_dim=64) == 4 * 32 * 32 * 65 * 4   # the head_dim 64 build splits the same way
        assert wanted(head_dim=96) == 4 * 32 * 32 * 97 * 4   # so do the builds for the other multiples of 16
        assert wanted(head_dim=80) == 4 * 32 * 32 * 81 * 4
        assert wanted(head_dim=72) == 0               # the general kernel does not split
    finally:
        lib.singe_hip_set_paged_attention_splits(0)
    assert lib.singe_hip_paged_attention_scratch_bytes(None) == 0


@pytest.mark.parametrize("heads,kv_heads,dim,sequences,chunk,decoding,keys,shares", [
    (16, 2, 128, 1, 64, 0, 16384, 16), (16, 2, 128, 1, 128, 0, 16384, 8), (16, 2, 128, 1, 256, 0, 16384, 4), (16, 2, 128, 4, 256, 0, 16384, 2),
    (64, 8, 128, 1, 64, 0, 16384, 16), (64, 8, 128, 1, 256, 0, 16384, 4), (32, 8, 128, 1, 128, 0, 16384, 16), (28, 4, 128, 1, 64, 0, 16384, 16), (28, 4, 128, 1, 256, 0, 16384, 4), (28, 4, 128, 2, 256, 0, 16384, 2),
    (28, 4, 128, 4, 256, 0, 16384, 2), (64, 8, 128, 1, 64, 0, 1024, 2),           # (two shares of eight key tiles are all there is)
    (16, 2, 128, 1, 1024, 20, 2112, 2), (16, 2, 128, 1, 64, 62, 2112, 4), (64, 8, 128, 1, 256, 32, 2112, 2)])
def test_key_shares_of_chunks_fill_the_chip_and_no_more(heads, kv_heads, dim, sequences, chunk, decoding, keys, shares):
    lib, both, tokens = _native.lib(), sequences + decoding, sequences * chunk + decoding
    problem = _native.PagedAttentionProblemC(tokens, heads, kv_heads, dim, 16, both, 100000, both * keys // 16, 0, 1, 0, 0, 0, 0.0, 0.0, 0)
    row = tokens * heads * (dim + 1) * 4
    assert lib.singe_hip_paged_attention_scratch_bytes(ctypes.byref(problem)) == shares * row
    own = _native.ThreadOptionsC(-1, 0, 0, 0, True, 1024)  # a caller's own number of workgroups is taken at its word
    lib.singe_hip_set_thread_options(ctypes.byref(own))
    try:
        tiles = kv_heads * (heads // kv_heads * tokens // 128 + both)
        wanted = min(-(-2 * 1024 // tiles), -(-keys // 512), 64)
        assert lib.singe_hip_paged_attention_scratch_bytes(ctypes.byref(problem)) == (wanted * row if wanted > 1 else 0)
    finally:
        lib.singe_hip_set_thread_options(None)


def test_paged_mla_attention_validation():
    lib = _native.lib()
    fake = 0x1000
    def call(**changes):
        fields = dict(tokens=2, heads=2, latent_dim=32, position_dim=8, page_size=4, sequences=1, cache_pages=2, page_table=1,
                      data_type=1, index_type=0, causal=1, has_scale=0, scale=0.0)
        fields.update(changes)
        problem = _native.PagedMlaAttentionProblemC(*fields.values())
        return lib.singe_hip_paged_mla_attention(None, *([fake] * 9), None, None, ctypes.byref(problem))
    assert call(page_size=0) == 9 and call(latent_dim=0) == 9      # paged_mla_attention_problem's own refusals
    assert call(data_type=4) == 9 and call(index_type=3) == 9
    assert call(has_scale=1, scale=float("nan")) == 9
    assert call(latent_dim=576) == 5 and call(position_dim=160) == 5
    assert call(tokens=0) == 0


def test_paged_kv_prefill_config_validation_mirrors_reference_cases():
    """singe-kernel/src/cuda/attention/tests.rs:349-375."""
    lib = _native.lib()
    good = _native.PagedKvPrefillAttentionConfigC(2, 7, 4, 2, 8, 3, 5, 4, 1, 0.5)
    assert lib.singe_hip_paged_kv_prefill_attention_config_validate(ctypes.byref(good)) == 0
    bad_heads = _native.PagedKvPrefillAttentionConfigC(2, 7, 3, 2, 8, 3, 5, 4, 1, 0.5)
    assert lib.singe_hip_paged_kv_prefill_attention_config_validate(ctypes.byref(bad_heads)) == 1
    fake = 0x1000
    status = lib.singe_hip_paged_kv_prefill_attention_bf16(None, fake, 224, fake, 27, fake, 224, fake, 240, fake, 240, fake, 2,
                                                           fake, 2, fake, 2, fake, 8, ctypes.byref(good))
    assert status == 2
    detail = _native.ErrorDetail()
    lib.singe_hip_last_error(ctypes.byref(detail))
    assert detail.name == b"lse" and detail.minimum == 28 and detail.actual == 27


def test_dense_problem_and_splitk_validation():
    lib = _native.lib()
    fake = 0x1000
    def dense(**changes):
        fields = dict(batch=1, heads=4, kv_heads=2, query_len=3, key_len=5, head_dim=64, value_dim=64,
                      mask_strides=(ctypes.c_int64 * 4)(0, 0, 0, 0), data_type=0, causal=0, has_scale=0, has_window=0,
                      has_softcap=0, scale=0.0, softcap=0.0, window=0)
        fields.update(changes)
        problem = _native.AttentionProblemC(*fields.values())
        return lib.singe_hip_scaled_dot_product_attention(None, fake, fake, fake, None, None, None, fake, ctypes.byref(problem))
    assert dense(kv_heads=3) == 9
    assert dense(key_len=0) == 9
    assert dense(head_dim=0) == 9
    assert dense(data_type=5) == 9
    assert dense(head_dim=257) == 5
    assert dense(query_len=0) == 0  # an empty output, nothing launched
    assert dense(has_softcap=1, softcap=0.0) == 9
    config = _native.SplitKReduceConfigC(1, 2, 5, 8, 80, 40, 8, 10, 5, 16, 8)
    assert lib.singe_hip_splitk_reduce_f32(None, fake, 16, fake, 80, fake, 10, ctypes.byref(config)) != 2
    assert lib.singe_hip_splitk_reduce_f32(None, fake, 16, fake, 79, fake, 10, ctypes.byref(config)) == 2
    zero = _native.SplitKReduceConfigC(1, 2, 0, 8, 80, 40, 8, 10, 5, 16, 8)
    assert lib.singe_hip_splitk_reduce_f32(None, fake, 16, fake, 80, fake, 10, ctypes.byref(zero)) == 1


def test_f32_block_table_ops_validate_like_the_bf16_ones():
    lib = _native.lib()
    fake = 0x1000
    config = _native.PagedKvDecodeAttentionConfigC(**GOOD)
    lens = dict(out=2 * 8 * 128, query=2 * 8 * 128, key=8 * 16 * 2 * 128, value=8 * 16 * 2 * 128, seq=2, table=8)
    def decode(config=config, workspace=fake, workspace_bytes=1 << 30, **short):
        n = dict(lens, **short)
        return lib.singe_hip_paged_kv_decode_attention_f32(None, fake, n["out"], fake, n["query"], fake, n["key"], fake, n["value"],
                                                           fake, n["seq"], fake, n["table"], workspace, workspace_bytes, ctypes.byref(config))
    need = lib.singe_hip_paged_kv_decode_attention_f32_workspace_bytes(ctypes.byref(config))
    assert need == 2 * 8 * 64 * 129 * 4
    for name in ("out", "query", "key", "value", "seq", "table"):
        assert decode(**{name: lens[name] - 1}) == 2, name
    assert decode(workspace=None) == 6
    assert decode(workspace_bytes=need - 1) == 2
    assert decode(config=_native.PagedKvDecodeAttentionConfigC(**dict(GOOD, kv_heads=3))) == 1
    assert decode(config=_native.PagedKvDecodeAttentionConfigC(**dict(GOOD, head_dim=48)), out=1 << 20, query=1 << 20) == 5
    assert lib.singe_hip_paged_kv_decode_attention_f32_workspace_bytes(
        ctypes.byref(_native.PagedKvDecodeAttentionConfigC(**dict(GOOD, batch=0)))) == 0
    prefill = A.PagedKvPrefillAttentionConfig(2, 10, 4, 2, 64, 16, 8, 4, True, 0.1)._c()
    sizes = [10 * 4 * 64, 10 * 4, 10 * 4 * 64, 8 * 16 * 2 * 64, 8 * 16 * 2 * 64, 2, 2, 2, 8]
    def run(sizes, pointer=fake):
        flat = []
        for n in sizes:
            flat += [pointer, n]
        return lib.singe_hip_paged_kv_prefill_attention_f32(None, *flat, ctypes.byref(prefill))
    for index in range(9):
        short = list(sizes)
        short[index] -= 1
        assert run(short) == 2, index
    assert run(sizes, pointer=None) == 6


def test_parts_archive_is_checked_before_anything_changes():
    """singe_hip_load on an archive of parts: the build's own archive is taken; a wrong version, an entry count of
    zero, a part name the library does not know, a part listed twice and an entry that runs past the image are each
    refused with the status the header names, without a device."""
    import struct

    from singe_amd import build

    lib = _native.lib()
    magic = build.ARCHIVE_MAGIC
    entry = lambda name, offset, size: struct.pack("<48sQQ", name, offset, size)
    body = b"\x7fELF" + b"\0" * 60
    good = magic + struct.pack("<II", 1, 1) + entry(b"hbm_stream", 88, 64) + body
    try:
        assert lib.singe_hip_load(good, len(good)) == 0
        cases = {
            "version": (magic + struct.pack("<II", 2, 1) + entry(b"hbm_stream", 88, 64) + body, 9),
            "no entries": (magic + struct.pack("<II", 1, 0), 1),
            "entries past the image": (magic + struct.pack("<II", 1, 3) + entry(b"hbm_stream", 88, 64) + body, 1),
            "unknown part": (magic + struct.pack("<II", 1, 1) + entry(b"not_a_part", 88, 64) + body, 9),
            "part twice": (magic + struct.pack("<II", 1, 2) + entry(b"hbm_stream", 152, 64) + entry(b"hbm_stream", 152, 64) + body, 9),
            "runs past the end": (magic + struct.pack("<II", 1, 1) + entry(b"hbm_stream", 88, 65) + body, 2),
            "empty part": (magic + struct.pack("<II", 1, 1) + entry(b"hbm_stream", 88, 0) + body, 2),
            "header only": (magic + b"\x01", 1),
        }
        for name, (image, status) in cases.items():
            assert lib.singe_hip_load(image, len(image)) == status, name
        assert lib.singe_hip_load(None, 4) == 6 and lib.singe_hip_load(good, 0) == 1
        assert lib.singe_hip_load_part(b"hbm_stream", body, len(body)) == 0
        assert lib.singe_hip_load_part(b"hbm_strea", body, len(body)) == 9
        assert lib.singe_hip_load_part(b"hbm_stream_", body, len(body)) == 9
        assert lib.singe_hip_load_part(None, body, len(body)) == 6
    finally:
        lib.singe_hip_unload()


def test_build_archive_lists_every_part_at_aligned_offsets():
    import struct

    from singe_amd import build

    image = build.pack_archive()
    assert image[:16] == build.ARCHIVE_MAGIC
    version, entries = struct.unpack_from("<II", image, 16)
    assert version == 1 and entries == len(_native.CODE_OBJECT_PARTS)
    for index, (part, path) in enumerate(zip(_native.CODE_OBJECT_PARTS, _native.CODE_OBJECT_PATHS)):
        name, offset, size = struct.unpack_from("<48sQQ", image, 24 + 64 * index)
        assert name.rstrip(b"\0").decode() == part and offset % 16 == 0
        assert image[offset:offset + size] == open(path, "rb").read()


def test_fixed_scratch_limit_is_where_the_documents_say():
    """The entry point that allocates nothing refuses a config whose scratch exceeds the fixed array: at 32 query / 8 KV
    heads (and the 256 compute units the library assumes without a device) that is 759 sequences, not one more."""
    sized = lambda batch: A.PagedKvDecodeAttentionConfig.contiguous(batch, 32, 8, 128, 16, 16384, 256, 0.1).workspace_bytes()
    if not (0 < sized(1) < A.STATIC_SCRATCH_BYTES):
        pytest.skip("the library sees a device with another compute-unit count")
    text = open(os.path.join(ROOT, "include", "singe_hip_attention.h")).read()
    assert re.search(r"#define SINGE_HIP_STATIC_SCRATCH_BYTES \(16u << 20\)", text) and A.STATIC_SCRATCH_BYTES == 16 << 20
    assert sized(759) <= A.STATIC_SCRATCH_BYTES < sized(760)
    assert sized(32) < 5 << 20  # the headline decode shape uses under a third of it


def test_two_threads_hold_different_settings():
    """Per-thread options: each thread reads its own relaxed-numerics flag, decode workers and split threshold in the
    size queries it makes, whatever the other thread and the process-wide setters say meanwhile."""
    import threading

    lib = _native.lib()
    config = A.PagedKvDecodeAttentionConfig.contiguous(8, 32, 8, 128, 16, 1024, 64, 0.1)
    c = config._c()
    default_workers = int(lib.singe_hip_decode_workers(ctypes.byref(c)))
    default_bytes = config.workspace_bytes()
    barrier = threading.Barrier(2)
    seen, failures = {}, []

    def body(name, workers, relaxed, below):
        try:
            options = _native.ThreadOptionsC(relaxed, workers, 0, 0, 1, below)
            assert lib.singe_hip_set_thread_options(ctypes.byref(options)) == 0
            barrier.wait(timeout=10)
            if name == "a":  # a process-wide change made while both threads hold their own
                lib.singe_hip_set_decode_workers(48)
                lib.singe_hip_set_relaxed_numerics(1 - relaxed)
            barrier.wait(timeout=10)
            parameters = _native.AttentionParametersC()
            for _ in range(200):
                lib.singe_hip_attention_parameters(ctypes.byref(parameters))
                seen[name] = (int(lib.singe_hip_decode_workers(ctypes.byref(c))), config.workspace_bytes(),
                              int(lib.singe_hip_relaxed_numerics()), int(parameters.split_below_blocks))
                assert seen[name][0] == workers and seen[name][2] == relaxed and seen[name][3] == below
            barrier.wait(timeout=10)
            assert lib.singe_hip_set_thread_options(None) == 0
            cleared = _native.ThreadOptionsC()
            lib.singe_hip_thread_options(ctypes.byref(cleared))
            assert (cleared.relaxed_numerics, cleared.decode_workers, cleared.has_split_below_blocks) == (-1, 0, 0)
            assert int(lib.singe_hip_decode_workers(ctypes.byref(c))) == 48  # back on the process-wide value
        except Exception as problem:  # noqa: BLE001 - reported by the test's own thread
            failures.append((name, repr(problem)))
            barrier.abort()

    try:
        threads = [threading.Thread(target=body, args=("a", 64, 1, 7)), threading.Thread(target=body, args=("b", 512, 0, 300))]
        for thread in threads:
            thread.start()
        for thread in threads:
            thread.join(timeout=30)
        assert not failures, failures
        assert seen["a"][1] < seen["b"][1]  # more key ranges, more partial rows
        bad = _native.ThreadOptionsC(2, 0, 0, 0, 0, 0)
        assert lib.singe_hip_set_thread_options(ctypes.byref(bad)) == 9
        bad = _native.ThreadOptionsC(-1, 0, 65, 0, 0, 0)
        assert lib.singe_hip_set_thread_options(ctypes.byref(bad)) == 9
    finally:
        lib.singe_hip_set_decode_workers(0)
        lib.singe_hip_set_relaxed_numerics(0)
        lib.singe_hip_set_thread_options(None)
    assert int(lib.singe_hip_decode_workers(ctypes.byref(c))) == default_workers and config.workspace_bytes() == default_bytes


def test_dense_family_validation_order_needs_no_device():
    """The rest of the dense family checks config and lengths in the order of the reference's validate_lengths, before
    any pointer is read: statuses and the names they carry, on fake pointers."""
    lib = _native.lib()
    fake = 0x1000
    detail = _native.ErrorDetail()

    def named(status):
        lib.singe_hip_last_error(ctypes.byref(detail))
        return status, (detail.name or b"").decode()

    prefill = A.FmhaPrefillConfig.contiguous(2, 8, 8, 4, 2, 64, 0.1, True)
    full = 2 * 8 * 4 * 64
    sink = _native.AttentionSinkPrefillConfigC(prefill._c(), 3, 2)
    call = lambda lengths, config=sink: named(lib.singe_hip_attention_sink_prefill_f32(
        None, fake, lengths[0], fake, lengths[1], fake, lengths[2], fake, lengths[3], fake, lengths[4], ctypes.byref(config)))
    kv = 2 * 8 * 2 * 64
    assert call([full, full - 1, kv, kv, 4]) == (2, "query")          # query, key, value, out, then sinks (mod.rs:1843-1858)
    assert call([full - 1, full, kv - 1, kv, 4]) == (2, "key")
    assert call([full - 1, full, kv, kv, 4]) == (2, "out")
    assert call([full, full, kv, kv, 3]) == (2, "sinks")
    assert call([full, full, kv, kv, 4], _native.AttentionSinkPrefillConfigC(prefill._c(), 1 << 31, 2)) == (3, "start_q")
    assert named(lib.singe_hip_attention_sink_prefill_f32(None, fake, full, fake, full, fake, kv, fake, kv, None, 4, ctypes.byref(sink))) == (6, "sinks")

    decode = A.FmhaDecodeConfig.contiguous(2, 9, 4, 2, 64, 0.1)
    capped = _native.SoftcappedWindowDecodeConfigC(decode._c(), 4, 1, 0.0)   # a cap of zero is invalid
    rows, keys = 2 * 4 * 64, 2 * 9 * 2 * 64
    windowed = lambda config, lse_len=8: named(lib.singe_hip_softcapped_window_decode_lse_bf16(
        None, fake, rows, fake, lse_len, fake, rows, fake, keys, fake, keys, ctypes.byref(config)))
    assert windowed(capped) == (1, "soft_cap")
    assert windowed(_native.SoftcappedWindowDecodeConfigC(decode._c(), 1 << 31, 0, 0.0)) == (3, "window_size")
    assert windowed(_native.SoftcappedWindowDecodeConfigC(decode._c(), 4, 1, 2.0), lse_len=7) == (2, "lse")
    assert named(lib.singe_hip_fmha_decode_lse_f16(None, fake, rows, fake, 8, fake, rows, fake, keys - 1, fake, keys,
                                                   ctypes.byref(decode._c()))) == (2, "key")

    ragged = A.RaggedKvPrefillAttentionConfig.contiguous(3, 10, 12, 4, 2, 32, True, 0.2)._c()
    lengths = [10 * 4 * 32, 40, 10 * 4 * 32, 12 * 2 * 32, 12 * 2 * 32, 3, 3, 3]
    names = ["out", "lse", "query", "key", "value", "actual_seq_lens_q", "actual_seq_lens_kv", "actual_seq_offsets"]
    for position in reversed(range(8)):   # with every later length good, the first short one is the one reported
        short = list(lengths)
        for earlier in range(position, 8):
            short[earlier] = lengths[earlier] - (1 if earlier == position else 0)
        arguments = []
        for length in short:
            arguments += [fake, length]
        assert named(lib.singe_hip_ragged_kv_prefill_attention_f32(None, *arguments, ctypes.byref(ragged))) == (2, names[position])
    with pytest.raises(error.InvalidLength):
        A.RaggedKvPrefillAttentionConfig.contiguous(3, 10, 12, 4, 3, 32, True, 0.2)   # kv heads must divide heads

    sliding = A.SlidingWindowAttentionConfig.contiguous(2, 5, 13, 4, 2, 16, 8, 0, 4, 0.3)
    paged = _native.PagedKvAttentionConfigC(sliding._c(), 4, 11, 4, 4 * 2 * 16, 4 * 2 * 16)
    cache = 11 * 4 * 2 * 16
    through = lambda table_len, cache_len=cache, config=paged: named(lib.singe_hip_sliding_window_attention_paged_kv_f32(
        None, fake, 2 * 5 * 4 * 16, fake, 2 * 5 * 4 * 16, fake, cache_len, fake, cache, fake, table_len, ctypes.byref(config)))
    assert through(7) == (2, "block_table")       # (batch - 1) * stride + ceil(13 / 4) = 8 entries (mod.rs:2893-2900)
    assert through(8, cache - 1) == (2, "key_cache")
    assert through(8, cache, _native.PagedKvAttentionConfigC(sliding._c(), 0, 11, 4, 128, 128))[0] == 1
    packed = _native.PackedQkvAttentionConfigC(sliding._c(), 0, 10, 1 << 40)
    assert named(lib.singe_hip_sliding_window_attention_packed_qkv_f32(None, fake, 640, fake, 5000, ctypes.byref(packed))) == (2, "qkv")


@pytest.mark.parametrize("batch,heads,query_len,key_len,head_dim,causal,shares", [
    (1, 8, 2500, 2500, 128, 1, 2),      # 160 tiles, long rows: two shares
    (1, 8, 2500, 2500, 96, 1, 2),
    (1, 16, 2000, 2000, 128, 1, 2),     # 256 tiles, one a compute unit
    (1, 32, 773, 773, 128, 1, 1),       # 224 tiles, short rows: none
    (1, 11, 1535, 1535, 64, 1, 1),      # either side of 1536 keys
    (1, 11, 1536, 1536, 64, 1, 2),
    (1, 80, 200, 100000, 128, 1, 1),    # causal rows see no more keys than there are queries
    (1, 48, 512, 4095, 64, 0, 1),       # either side of 4096 without a mask
    (1, 48, 512, 4096, 64, 0, 2),
    (1, 24, 2000, 2000, 128, 1, 1),     # 384 tiles: more than compute units
    (1, 8, 2000, 2000, 128, 1, 4),      # 128 tiles, half the compute units: as many as the keys allow
    (1, 8, 1, 4096, 128, 0, 8),         # a decode step
])
def test_dense_key_shares(batch, heads, query_len, key_len, head_dim, causal, shares):
    # (without a device the library counts on 256 compute units)
    problem = _native.AttentionProblemC(batch, heads, heads, query_len, key_len, head_dim, head_dim, (ctypes.c_int64 * 4)(0, 0, 0, 0), 1, causal,
                                        0, 0, 0, 0.0, 0.0, 0)
    wanted = shares * batch * heads * query_len * (head_dim + 1) * 4 if shares > 1 else 0   # shares x rows x (values + log-sum-exp) of f32
    assert _native.lib().singe_hip_scaled_dot_product_attention_scratch_bytes(ctypes.byref(problem)) == wanted


@pytest.mark.parametrize("heads,kv_heads,head_dim,chunks,chunk,decoding,rows", [
    (64, 8, 128, 2, 512, 62, 32),     # few chunks beside many decoding sequences
    (64, 8, 128, 2, 512, 56, 64),     # 33 whole 256-row tiles: either side of 9/16 of one a sequence
    (64, 8, 128, 2, 512, 57, 32),
    (64, 8, 64, 1, 1025, 62, 32),     # either side of 1024 tokens more than sequences
    (64, 8, 64, 1, 1026, 62, 64),
    (64, 8, 32, 2, 512, 62, 64),      # narrow heads: 256-row tiles
    (28, 4, 64, 1, 4096, 126, 64),    # a long chunk: 256-row tiles, however many sequences decode beside it
    (32, 8, 64, 1, 2048, 65, 64),
    (64, 8, 128, 64, 32, 0, 64),      # many short chunks
    (8, 8, 128, 1, 512, 62, 32),      # too few tiles for the chip
])
def test_paged_attention_row_tiles(heads, kv_heads, head_dim, chunks, chunk, decoding, rows):
    # (without a device the library counts on 256 compute units)
    tokens, sequences = chunks * chunk + decoding, chunks + decoding
    fields = dict(tokens=tokens, heads=heads, kv_heads=kv_heads, head_dim=head_dim, page_size=16, sequences=sequences, cache_pages=20000,
                  page_table=20000, index_type=0, causal=1, has_scale=0, has_window=0, has_softcap=0, scale=0.0, softcap=0.0, window=0)
    problem = _native.PagedAttentionProblemC(*fields.values())
    assert _native.lib().singe_hip_paged_attention_rows_per_wave(ctypes.byref(problem)) == rows


@pytest.mark.parametrize("tokens,heads,kv_heads,batch", [
    (2**31 - 1, 64, 1, 1),         # 2^37 rows to the one kv head: more than the packed kernel's 32-bit row counts hold
    (2**29, 64, 4, 3),             # 2^33
])
def test_packed_prefill_leaves_row_counts_beyond_32_bits_to_the_row_kernel(tokens, heads, kv_heads, batch):
    # which refuses these for their number of workgroups, before anything is launched or read
    config = A.RaggedKvPrefillAttentionConfig.contiguous(batch, tokens, 16, heads, kv_heads, 16, True, 0.25)._c()
    address, many = 1 << 20, 2**60
    arguments = [address if i % 2 == 0 else many for i in range(16)]
    assert _native.lib().singe_hip_ragged_kv_prefill_attention_bf16(None, *arguments, ctypes.byref(config)) == 8


@pytest.mark.parametrize("chunks,chunk,decoding,keys,rows", [
    (2, 512, 32, 2112, 32),           # less than a whole 256-row tile a sequence, sequences of 1024 to 4096 keys
    (2, 512, 30, 2112, 64),           # 32 whole tiles, 32 sequences
    (2, 512, 32, 1023, 64),           # either side of 1024 and 4096 keys
    (2, 512, 32, 4097, 64),
    (1, 2049, 80, 2112, 32),          # either side of 2048 tokens more than sequences
    (1, 2050, 80, 2112, 64),
])
def test_paged_attention_row_tiles_by_the_keys_a_sequence_has(chunks, chunk, decoding, keys, rows):
    tokens, sequences = chunks * chunk + decoding, chunks + decoding
    fields = dict(tokens=tokens, heads=64, kv_heads=8, head_dim=128, page_size=16, sequences=sequences, cache_pages=20000,
                  page_table=-(-keys * sequences // 16), index_type=0, causal=1, has_scale=0, has_window=0, has_softcap=0, scale=0.0, softcap=0.0,
                  window=0)
    problem = _native.PagedAttentionProblemC(*fields.values())
    assert _native.lib().singe_hip_paged_attention_rows_per_wave(ctypes.byref(problem)) == rows


@pytest.mark.parametrize("heads,kv_heads,head_dim,chunks,chunk,decoding,rows", [
    (64, 8, 96, 2, 512, 40, 32),      # past 9/16 of a whole 256-row tile a sequence, where the 128-row kernel has a loop for few rows
    (64, 8, 80, 2, 512, 40, 64),      # ... and where it has none
    (64, 8, 112, 2, 512, 40, 64),
    (68, 4, 128, 2, 512, 100, 64),    # ... or the rows of a token are more than the loop takes
    (64, 4, 128, 2, 512, 100, 32),
    (64, 8, 80, 2, 512, 62, 32),
])
def test_paged_attention_row_tiles_by_the_loop_for_few_rows(heads, kv_heads, head_dim, chunks, chunk, decoding, rows):
    tokens, sequences = chunks * chunk + decoding, chunks + decoding
    problem = _native.PagedAttentionProblemC(tokens, heads, kv_heads, head_dim, 16, sequences, 20000, 132 * sequences, 0, 1, 0, 0, 0, 0.0, 0.0, 0)
    assert _native.lib().singe_hip_paged_attention_rows_per_wave(ctypes.byref(problem)) == rows


@pytest.mark.parametrize("batch,heads,head_dim,query_len,key_len,causal,rows", [
    (4, 32, 128, 4096, 4096, 1, 64),    # whole rounds of long rows
    (4, 32, 128, 1024, 1024, 1, 32),    # short causal rows
    (2, 32, 128, 1535, 1535, 1, 32),    # either side of 1536 keys, less than a round
    (2, 32, 128, 1536, 1536, 1, 64),
    (4, 32, 128, 1536, 1536, 1, 32),    # one and a half rounds
    (4, 32, 128, 2048, 2048, 1, 64),
    (2, 32, 128, 2560, 2560, 1, 32),    # one and a quarter
    (1, 32, 128, 3072, 3072, 1, 64),    # three quarters of a round
    (1, 31, 128, 2048, 2048, 1, 32),    # half of one
    (4, 32, 128, 899, 899, 0, 32),      # either side of 900 keys without a mask
    (4, 32, 128, 900, 900, 0, 64),
    (4, 32, 128, 1024, 899, 0, 32),
    (3, 32, 96, 1280, 1280, 0, 32),     # a little more than a round
    (3, 32, 96, 1536, 1536, 0, 64),
    (1, 32, 128, 2560, 2560, 0, 64),
    (4, 32, 64, 4096, 4096, 1, 32),     # narrow heads
    (4, 32, 64, 4096, 4096, 0, 64),
    (4, 32, 64, 2048, 2048, 0, 32),
    (4, 32, 32, 4096, 4096, 0, 32),
])
def test_dense_prefill_rows_per_wave(batch, heads, head_dim, query_len, key_len, causal, rows):
    # (without a device the library counts on 256 compute units)
    config = A.FmhaPrefillConfig.contiguous(batch, query_len, key_len, heads, heads, head_dim, 0.125, bool(causal))
    assert _native.lib().singe_hip_dense_prefill_rows_per_wave(ctypes.byref(config._c())) == rows


@pytest.mark.parametrize("batch,heads,head_dim,query_len,key_len,causal,rows", [
    (2, 32, 128, 4096, 1600, 1, 64),    # most causal rows see all keys
    (2, 32, 128, 4096, 1650, 1, 64),    # (either side of two and a half times as many queries as keys, 1536 keys and up)
    (2, 32, 128, 4096, 1535, 1, 64),
    (1, 64, 128, 2559, 1024, 1, 32),
    (4, 32, 128, 4096, 1023, 1, 32),    # either side of 1024 keys
    (4, 32, 128, 4096, 1024, 1, 64),
    (2, 32, 96, 2048, 512, 0, 64),      # one round of full tiles over few keys
    (2, 32, 96, 2048, 511, 0, 32),
    (4, 32, 96, 2048, 512, 0, 32),      # ... two
    (16, 32, 48, 256, 512, 0, 64),      # one 256-row tile to a head
    (16, 32, 48, 128, 512, 0, 32),      # ... one 128-row tile
    (16, 32, 48, 257, 512, 0, 32),
    (16, 32, 48, 256, 511, 0, 32),
    (15, 32, 80, 256, 512, 0, 32),      # ... less than two to a compute unit
    (16, 32, 80, 256, 512, 1, 32),
    (16, 32, 64, 256, 2047, 0, 32),
    (16, 32, 64, 256, 2048, 0, 64),
    (2, 32, 64, 4096, 4096, 1, 64),     # narrow heads in two whole rounds
    (2, 32, 64, 4096, 999, 1, 32),
    (2, 32, 48, 4096, 4096, 1, 32),
    (2, 32, 48, 3500, 3500, 0, 64),
    (2, 32, 64, 3072, 3072, 0, 32),     # one and a half
    (2, 32, 64, 3500, 2999, 0, 32),
    (8, 32, 64, 700, 3000, 0, 32),      # short rows, the last tile of each not whole
])
def test_dense_prefill_rows_per_wave_of_unequal_lengths_and_narrow_heads(batch, heads, head_dim, query_len, key_len, causal, rows):
    config = A.FmhaPrefillConfig.contiguous(batch, query_len, key_len, heads, heads, head_dim, 0.125, bool(causal))
    assert _native.lib().singe_hip_dense_prefill_rows_per_wave(ctypes.byref(config._c())) == rows


@pytest.mark.parametrize("fields,status", [
    (dict(head_dim=0), 9),         # a problem that makes no sense is refused as the other entry points refuse it
    (dict(page_size=0), 9),
    (dict(head_dim=24), 5),        # one that does, at a width without a matrix-core build
    (dict(sequences=0), 5),
    (dict(tokens=0), 0),
])
def test_every_row_refuses_what_makes_no_sense_before_what_it_has_no_build_for(fields, status):
    lib = _native.lib()
    known = dict(tokens=4, heads=8, kv_heads=2, head_dim=64, page_size=16, sequences=2, cache_pages=4, page_table=4, index_type=0, causal=1,
                 has_scale=0, has_window=0, has_softcap=0, scale=0.0, softcap=0.0, window=0)
    problem = _native.PagedAttentionProblemC(*{**known, **fields}.values())
    assert lib.singe_hip_paged_attention_every_row(1, None, *[0x1000] * 10, None, 0, ctypes.byref(problem)) == status
    if status != 5 or "sequences" in fields:
        latent = _native.PagedMlaAttentionProblemC(fields.get("tokens", 4), 8, fields.get("head_dim", 512), 64, fields.get("page_size", 16),
                                                   fields.get("sequences", 2), 4, 4, 1, 0, 1, 0, 0.0)
        assert lib.singe_hip_paged_mla_attention_every_row(None, *[0x1000] * 11, None, 0, ctypes.byref(latent)) == status


ROW_TILES, DECODE_KERNELS, ONE_LAUNCH = 0, 1, 2


def paged_route(heads, kv_heads, head_dim, sequences, keys, scratch="asked for", page_size=16, **fields):
    """The route of a step of a token a sequence, `keys` each on average, with no scratch, as much as it asks for, or (address, bytes)."""
    lib = _native.lib()
    known = dict(tokens=sequences, heads=heads, kv_heads=kv_heads, head_dim=head_dim, page_size=page_size, sequences=sequences,
                 cache_pages=1 << 20, page_table=sequences * keys // page_size, index_type=1, causal=1, has_scale=0, has_window=0, has_softcap=0,
                 scale=0.0, softcap=0.0, window=0)
    problem = _native.PagedAttentionProblemC(*{**known, **fields}.values())
    wanted = lib.singe_hip_paged_attention_scratch_bytes(ctypes.byref(problem))
    address, count = (0x1000, wanted) if scratch == "asked for" else (None, 0) if scratch is None else scratch(wanted)
    return lib.singe_hip_paged_attention_route(ctypes.byref(problem), address, count)


@pytest.mark.parametrize("heads,kv_heads,head_dim,sequences,keys,route", [
    (32, 8, 128, 1, 32000, ONE_LAUNCH),        # few units: 2^18 keys between them
    (32, 8, 128, 1, 32784, DECODE_KERNELS),
    (32, 8, 64, 1, 7168, ONE_LAUNCH),          # ... of up to four narrow rows, and of fewer than four: 7 * 2^13
    (32, 8, 64, 1, 7184, DECODE_KERNELS),
    (32, 32, 128, 1, 1792, ONE_LAUNCH),
    (32, 32, 128, 1, 2000, DECODE_KERNELS),
    (32, 8, 128, 16, 896, ONE_LAUNCH),         # up to 128 units of 896 keys
    (32, 8, 128, 16, 912, DECODE_KERNELS),
    (32, 8, 128, 24, 704, ONE_LAUNCH),         # ... 192 of 704
    (32, 8, 128, 24, 720, DECODE_KERNELS),
    (32, 8, 128, 24, 864, DECODE_KERNELS),
    (32, 8, 128, 64, 384, ONE_LAUNCH),         # more: 576 of more than four rows, else 384
    (32, 8, 128, 64, 400, DECODE_KERNELS),
    (64, 8, 128, 64, 576, ONE_LAUNCH),
    (64, 8, 128, 64, 592, DECODE_KERNELS),
    (32, 8, 128, 128, 96, ONE_LAUNCH),         # up to 1024 units, 512 of four narrower rows and of fewer
    (32, 8, 96, 64, 96, ONE_LAUNCH),
    (32, 8, 96, 80, 96, DECODE_KERNELS),
    (64, 8, 64, 128, 96, ONE_LAUNCH),
    (32, 32, 128, 16, 96, ONE_LAUNCH),
    (32, 32, 128, 24, 96, DECODE_KERNELS),
    (64, 8, 128, 129, 96, DECODE_KERNELS),
])
def test_decode_steps_in_one_launch_are_those_that_gain_by_it_whatever_their_lengths(heads, kv_heads, head_dim, sequences, keys, route):
    # (200 to 1500 keys on 24 sequences of 32 / 8 heads x 128 took 30 us in one launch and 26 in three)
    assert paged_route(heads, kv_heads, head_dim, sequences, keys) == route


@pytest.mark.parametrize("sequences,keys,scratch,route", [
    (1, 32000, lambda wanted: (0x1000, wanted), ONE_LAUNCH),
    (1, 32000, lambda wanted: (0x1010, wanted), ROW_TILES),                       # not on a 256-byte boundary: key shares of the row tiles
    (1, 32000, lambda wanted: (0x1010, 63 * 32 * 129 * 4), ROW_TILES),            # ... which 63 shares of 32 rows need
    (1, 32000, lambda wanted: (0x1010, 63 * 32 * 129 * 4 - 1), ONE_LAUNCH),
    (1, 32000, lambda wanted: (None, 0), ONE_LAUNCH),
    (1, 32000, lambda wanted: (0x1000, 16), ONE_LAUNCH),
    (1, 400, lambda wanted: (0x1010, wanted), ONE_LAUNCH),                        # too few keys for shares
])
def test_scratch_that_the_one_launch_has_no_use_for_goes_to_key_shares(sequences, keys, scratch, route):
    assert paged_route(32, 8, 128, sequences, keys, scratch) == route


def test_no_entry_point_draws_random_numbers_that_may_throw():
    # (std::random_device throws where the system has no source of them, through a C entry: the process ends)
    symbols = subprocess.run(["nm", "-D", "--undefined-only", "-C", _native.LIBRARY_PATH], check=True, capture_output=True, text=True).stdout
    assert "std::random_device" not in symbols
