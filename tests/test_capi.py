"""CPU checks of the C ABI: the library loads next to torch's HIP runtime, exports every entry
point include/miniserve_amd.h declares with the signatures the ctypes binding uses, and rejects
bad arguments before launching anything (no GPU needed: these calls fail in host code)."""

from __future__ import annotations

import ctypes
import re
from pathlib import Path

import pytest

from miniserve_amd import _native

HEADER = Path(__file__).resolve().parent.parent / "include" / "miniserve_amd.h"


def _declared() -> list[str]:
    text = HEADER.read_text()
    return sorted(set(re.findall(r"^\s*(?:const\s+)?\w+\*?\s+\*?(msa_\w+)\(", text, flags=re.M)))


def test_header_declares_the_binding():
    assert _declared() == sorted(_native.SIGNATURES)


def test_library_exports_every_symbol():
    lib = _native.load()
    for name in _declared():
        assert getattr(lib, name) is not None
    assert lib.msa_abi_version() == _native.ABI_VERSION


def test_single_hip_runtime_mapped():
    _native.load()
    assert len(_native._hip_runtimes_mapped()) <= 1


def _err(name, *args):
    with pytest.raises(RuntimeError) as e:
        _native.call(name, *args)
    return str(e.value)


NULL = ctypes.c_void_p(0)
FAKE = ctypes.c_void_p(0x1000)  # never dereferenced: every call below fails validation first


def test_argument_errors_are_reported():
    assert "null pointer" in _err("msa_int8_quantize", NULL, 0, 4, 4, NULL, NULL, NULL)
    assert "weight_dtype" in _err("msa_int8_quantize", FAKE, 7, 4, 4, FAKE, FAKE, NULL)
    assert "multiple of 16" in _err(
        "msa_int8_linear", FAKE, 4, 40, 40, FAKE, FAKE, 32, FAKE, 32, 0, NULL, 0, NULL, 0, NULL
    )
    assert "epilogue" in _err("msa_int8_linear", FAKE, 4, 64, 64, FAKE, FAKE, 32, FAKE, 32, 9, NULL, 0, NULL, 0, NULL)
    assert "head_dim must be 128" in _err(
        "msa_paged_attention_decode", FAKE, 64, FAKE, FAKE, 16, 2, 1, 64, 16, FAKE, 1, FAKE, FAKE, 1, 16, 1, 1.0,
        FAKE, 64, NULL, 0, NULL,
    )
    assert "null pointer" in _err(
        "msa_int8_linear_add_rmsnorm", FAKE, 4, 64, 64, FAKE, FAKE, 64, NULL, FAKE, 1e-6, FAKE, NULL, 0, NULL
    )
    assert "at most 4096" in _err(  # a split's keys: one block-table entry per lane of each wavefront
        "msa_paged_attention_decode", FAKE, 128 * 2, FAKE, FAKE, 16, 2, 1, 128, 16, FAKE, 1, FAKE, FAKE, 1, 4112, 1,
        1.0, FAKE, 128 * 2, NULL, 0, NULL,
    )
    assert "block_size must be 16" in _err(
        "msa_paged_attention_prefill", FAKE, 128, FAKE, FAKE, 16, 2, 1, 128, 8, FAKE, 1, FAKE, FAKE, 1, 1.0, FAKE,
        128, NULL,
    )
    assert "heads / kv_heads" in _err(
        "msa_paged_attention_prefill", FAKE, 128 * 8, FAKE, FAKE, 16, 8, 1, 128, 16, FAKE, 1, FAKE, FAKE, 1, 1.0,
        FAKE, 128 * 8, NULL,
    )
    # the allocation-free decode entry point refuses partials larger than its 16 MiB scratch
    assert "16 MiB scratch" in _err(
        "msa_paged_attention_decode_noalloc", FAKE, 128 * 32, FAKE, FAKE, 16, 32, 8, 128, 16, FAKE, 256, FAKE, FAKE,
        2048, 64, 64, 1.0, FAKE, 128 * 32, NULL,
    )
    assert "head_dim must be even" in _err(
        "msa_qk_norm_rope_cache", FAKE, 64, 1, 2, 1, 7, FAKE, FAKE, 1e-6, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, 4, NULL
    )


def test_zero_sized_calls_are_no_ops():
    _native.call("msa_int8_linear", NULL, 0, 64, 64, NULL, NULL, 32, NULL, 32, 0, NULL, 0, NULL, 0, NULL)
    _native.call("msa_rmsnorm", NULL, 64, NULL, NULL, 64, 0, 64, 1e-6, NULL)


def test_workspace_sizes():
    assert _native.query("msa_int8_linear_workspace_size", 1, 1024, 64) == 0  # one K chunk per wave: no split
    assert _native.query("msa_int8_linear_workspace_size", 64, 1024, 2048) == 0  # token-split kernel
    assert _native.query("msa_int8_linear_workspace_size", 2048, 4096, 1024) == 0  # GEMM, 512 tiles: no split
    # GEMM with few output tiles: split-K float32 partials (8B o_proj at 256 tokens: 64 tiles of
    # 128 x 128 x 4 splits; the down_proj: 32 tiles of 256 x 128 x 6 splits)
    assert _native.query("msa_int8_linear_workspace_size", 256, 4096, 4096) == 4 * 256 * 4096 * 4
    assert _native.query("msa_int8_linear_workspace_size", 256, 4096, 12288) == 6 * 256 * 4096 * 4
    assert _native.query("msa_int8_linear_workspace_size", 64, 1024, 2000) > 0  # K % 64 != 0: split-K
    # LM head: up to 64 rows stream the weight (candidates of 256 workgroups); more rows take the
    # GEMM route (normalized rows + candidates of 128-entry vocabulary blocks)
    assert _native.query("msa_lm_head_argmax_workspace_size", 64, 1024, 151936) == 64 * 256 * 8
    assert _native.query("msa_lm_head_argmax_workspace_size", 65, 1024, 151936) == 65 * 1024 * 2 + 65 * 1187 * 8
    assert _native.query("msa_lm_head_argmax_workspace_size", 17, 4096, 151936) == 17 * 4096 * 2 + 17 * 1187 * 8
    assert _native.query("msa_lm_head_argmax_workspace_size", 16, 4096, 151936) == 16 * 256 * 8
    assert _native.query("msa_lm_head_logits_workspace_size", 64, 1024, 151936) == 0  # streaming route
    assert _native.query("msa_lm_head_logits_workspace_size", 65, 1024, 151936) == 65 * 1024 * 2  # normalized rows
    # chunked sampling: 15 chunks of 10240 per 151936-entry row, 512 (key, index) pairs + 3 words each
    assert _native.query("msa_sample_workspace_size", 64, 151936) == 64 * 15 * (512 * 8 + 12)
    assert _native.query("msa_sample_workspace_size", 65536, 151936) == 0  # rows above the chunked path's limit
    assert _native.query("msa_paged_attention_decode_workspace_size", 64, 16, 128, 1) == 0
    ws = _native.query("msa_paged_attention_decode_workspace_size", 64, 16, 128, 8)
    assert ws >= 64 * 16 * 8 * (128 + 2) * 4


def test_linear_workspaces_follow_each_route():
    """Each linear asks for the partials of its own route: the plain one for none where only the fused ones
    split, and a capture has to hold no more than the splits without which the chip stays idle."""

    def sizes(m, n, k):
        return tuple(_native.query(f"msa_{c}_workspace_size", m, n, k)
                     for c in ("int8_linear", "int8_linear_add_rmsnorm", "int8_linear_min"))

    for m, n, k in [(27, 4096, 4096), (27, 6144, 4096), (64, 24576, 4096), (16, 4096, 12288), (768, 4096, 2048)]:
        assert sizes(m, n, k)[0] == 0 == sizes(m, n, k)[2], (m, n, k)
    assert sizes(27, 4096, 4096)[1] == 4 * 27 * 4096 * 4 and sizes(768, 4096, 2048)[1] == 2 * 768 * 4096 * 4
    plain, normed, least = sizes(96, 4096, 4096)  # the GEMM's splits, which no call had to hold before 128 rows
    assert plain == normed == 8 * 96 * 4096 * 4 and least == 0
    assert sizes(256, 4096, 4096) == (4 * 256 * 4096 * 4,) * 3
    assert sizes(27, 4096, 12288)[0] == 4 * 27 * 4096 * 4  # a long K
    assert sizes(17, 512, 24576)[2] > 0  # (and few outputs: split before, too)
    qk = _native.query("msa_int8_gemm_qk_norm_rope_cache_workspace_size", 448, 6144, 4096)
    assert qk == 2 * 448 * 6144 * 4 and _native.query("msa_int8_linear_min_workspace_size", 448, 6144, 4096) == 0
