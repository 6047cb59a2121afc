"""Kernels whose loops cannot afford memory behind a register: a spilled register's reload waits on the counter that
the direct-to-LDS tile loads run on and drains them, and an accumulator array indexed by a variable anywhere in the
kernel lives in scratch memory for all of it (a loop that may end early is not unrolled).  This test compiles those
sources for gfx950 with the compiler's resource remarks and checks that the kernels named here use no scratch memory."""
import os
import re
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

import pytest

from singe_amd import build

CSRC = os.path.join(os.path.dirname(build.__file__), "csrc")
# source, flags, kernels (regular expressions) that must not touch scratch memory
BUILDS = [
    ("latent_attention_mfma.hip", [], [r"singe_paged_mla_attention_(bf16|f16)_(l512_p64|any)"]),
    ("fmha_prefill_pair.hip", [], [r"singe_fmha_prefill_pair_.*"]),
    ("paged_attention_pair.hip", [], [r"singe_(rotary_)?paged_attention_pair_.*"]),
    ("fmha_prefill.hip", [], [r"singe_fmha_prefill_(bf16|f16)_d128_(causal|full)(_options)?", r"singe_fmha_prefill_(bf16|f16)_d128_causal_window"]),
    ("fmha_prefill.hip", ["-DSINGE_HEAD_DIM=64"], [r"singe_fmha_prefill_(bf16|f16)_d64_causal_window"]),
    ("paged_attention.hip", [], [r"singe_ragged_prefill_(bf16|f16)_d128", r"singe_paged_decode_step_(bf16|f16)_d128_i(32|64)", r"singe_paged_decode_step_(bf16|f16)_d128_i(32|64)_w8"]),
    ("paged_attention.hip", ["-DSINGE_HEAD_DIM=96"], [r"singe_paged_decode_step_(bf16|f16)_d96_i(32|64)(_w8)?"]),
    ("attention_mfma_f32.hip", [], [r"singe_attention_mfma_f32_d\d+_r\d+"]),
    ("paged_decode.hip", [], [r"singe_paged_decode_(bf16|f16)_d128_g1_b16", r"singe_paged_decode_f8kv_wide(_relaxed)?_d128_b16",
                              r"singe_paged_decode_(bf16|f16)_wide_d128_b16"]),
]


def remarks_of(name, flags):
    source = os.path.join(CSRC, name)
    with tempfile.TemporaryDirectory() as scratch:
        command = [build.hipcc()] + build.HIPCC_FLAGS + flags + ["-Rpass-analysis=kernel-resource-usage", "-I", os.path.dirname(source),
                                                                  source, "-o", os.path.join(scratch, "out.hsaco")]
        return subprocess.run(command, check=True, capture_output=True, text=True).stderr


@pytest.fixture(scope="module")
def remarks():
    with ThreadPoolExecutor(max_workers=min(4, os.cpu_count() or 1)) as pool:
        texts = list(pool.map(lambda item: remarks_of(item[0], item[1]), BUILDS))
    return {(name, *flags): text for (name, flags, _), text in zip(BUILDS, texts)}


@pytest.mark.parametrize("name,flags,patterns", BUILDS, ids=[" ".join([item[0], *item[1]]) for item in BUILDS])
def test_no_scratch_memory_in_the_kernels_that_cannot_afford_it(remarks, name, flags, patterns):
    scratch = {}
    kernel = None
    for line in remarks[(name, *flags)].splitlines():
        found = re.search(r"Function Name: (\S+)", line)
        if found:
            kernel = found.group(1)
        found = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)
        if found and kernel is not None:
            scratch[kernel] = int(found.group(1))
    for pattern in patterns:
        named = {kernel: size for kernel, size in scratch.items() if re.fullmatch(pattern, kernel)}
        assert named, f"no kernel of {name} matches {pattern}"
        assert all(size == 0 for size in named.values()), {kernel: size for kernel, size in named.items() if size}


@pytest.mark.parametrize("head_dim,past_the_caches", [(32, True), (48, False)])
def test_rows_that_end_inside_64_byte_pieces_leave_through_the_caches(head_dim, past_the_caches):
    # (past them such rows of a causal window's call go out in parts: 4 x 28 / 4 heads x 9401 x 112, window 16, 219 us and 120)
    source, flags = os.path.join(CSRC, "fmha_prefill.hip"), [flag for flag in build.HIPCC_FLAGS if flag != "--genco"]
    with tempfile.TemporaryDirectory() as scratch:
        listing = os.path.join(scratch, "out.s")
        subprocess.run([build.hipcc(), *flags, f"-DSINGE_HEAD_DIM={head_dim}", "--cuda-device-only", "-S", "-I", CSRC, source, "-o", listing],
                       check=True, capture_output=True)
        text = open(listing).read()
    for name in ("bf16", "f16"):
        kernel = f"singe_fmha_prefill_{name}_d{head_dim}_causal_window"
        stores = re.findall(r"global_store_dwordx4 .*", re.search(rf"^{kernel}:(.*?)s_endpgm", text, re.S | re.M).group(1))
        assert stores and any(store.endswith(" nt") for store in stores) == past_the_caches
