"""CPU checks of the C ABI: the built library loads, exports every entry point
declared in include/gdn_mi355x.h, and the ctypes table matches the header's
parameter types one by one (no compute call is made)."""

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gdn_mi355x.h")


def _declarations():
    src = open(HEADER).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    out = {}
    for m in re.finditer(r"(?:int64_t|int|const char\*)\s+(gdn_\w+)\s*\(([^;]*?)\);", src, re.S):
        params = [p.strip() for p in m.group(2).split(",") if p.strip() and p.strip() != "void"]
        out[m.group(1)] = params
    return out


def _ctype_of(param):
    decl = re.sub(r"\s+", " ", param)
    if "int64_t*" in decl.replace(" ", ""):
        return ctypes.POINTER(ctypes.c_int64)
    if "*" in decl:
        return ctypes.c_void_p
    if decl.startswith("int64_t"):
        return ctypes.c_int64
    if decl.startswith("int "):
        return ctypes.c_int
    if decl.startswith("float"):
        return ctypes.c_float
    raise AssertionError(f"unmapped parameter type: {param}")


def test_header_declares_expected_entry_points():
    names = set(_declarations())
    assert {"gdn_last_error", "gdn_abi_version", "gdn_chunk_gated_delta_rule", "gdn_fused_recurrent",
            "gdn_fused_conv_recurrent", "gdn_packed_causal_conv1d", "gdn_prepare", "gdn_prefill_frontend",
            "gdn_conv_decode", "gdn_store_state", "gdn_copy_rows", "gdn_zero_rows",
            "gdn_commit_accepted", "gdn_prefill_qk", "gdn_prefill_fused", "gdn_conv_snapshots",
            "gdn_rms_norm_gated", "gdn_metadata_copy", "gdn_metadata_pad", "gdn_prefill_fused_noalloc",
            "gdn_prefill_noalloc_scratch_bytes", "gdn_gather_linear_slots"} <= names
    assert "gdn_probe_rmw" not in names  # the bench-only probe lives in libgdn_probe.so


def test_ctypes_table_matches_header():
    from logssms_amd import _lib
    decls = _declarations()
    for name, params in decls.items():
        if name in ("gdn_last_error", "gdn_abi_version", "gdn_prefill_noalloc_scratch_bytes"):
            assert params == []
            continue
        assert name in _lib.SIGNATURES, name
        want = [_ctype_of(p) for p in params]
        assert _lib.SIGNATURES[name] == want, name


def test_library_loads_and_exports_every_symbol():
    from logssms_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.lib()
    for name in _declarations():
        assert hasattr(lib, name), name
    assert lib.gdn_abi_version() == 6
    assert lib.gdn_prefill_noalloc_scratch_bytes() == 256 << 20
    assert lib.gdn_last_error() in (b"",) or isinstance(lib.gdn_last_error(), bytes)


def test_invalid_arguments_report_errors_without_a_gpu():
    """Argument validation happens before any HIP call, so it runs on a CPU box."""
    from logssms_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.lib()
    rc = lib.gdn_store_state(None, 0, None, 5, None, 0, 3, 128, None)
    assert rc == 1
    assert b"indices" in lib.gdn_last_error()
    rc = lib.gdn_fused_conv_recurrent(*([None, 0, 0, 1, None, 0, None, None, 4, None, 0, 0, 1, None, 0, 0, 1, None,
                                         0, None, 0, 1, 17, 2, 4, 64, 64, None, 0, 0, None, 0, 0, 0, 0, 0, None, 0,
                                         1, None, 0, 1, 1, None, 1.0, None]))
    assert rc == 1
    assert b"steps" in lib.gdn_last_error()
    # empty work is a no-op success
    assert lib.gdn_copy_rows(None, 0, None, 1, None, 0, None, 1, 0, 1, 16, 0, None) == 0
    assert lib.gdn_rms_norm_gated(None, 1, 0, 128, None, 1, 32, 4096, 128, 1, None, 0, 1e-6, None, None) == 0
    assert lib.gdn_rms_norm_gated(None, 1, 4, 0, None, 1, 32, 4096, 128, 1, None, 0, 1e-6, None, None) == 1
    assert b"bad shape" in lib.gdn_last_error()
    assert lib.gdn_rms_norm_gated(None, 7, 4, 128, None, 1, 32, 4096, 128, 1, None, 0, 1e-6, None, None) == 1
    assert lib.gdn_rms_norm_gated(None, 1, 4, 128, None, 1, 32, 4096, 128, 1, None, 0, 1e-6, None, None) == 1
    assert b"null" in lib.gdn_last_error()
    assert lib.gdn_metadata_copy(None, None, None, None, None, None, 0, None) == 0  # nothing to move
    assert lib.gdn_metadata_pad(None, None, None, None, None, None, None, 0, None) == 0
    assert lib.gdn_metadata_pad(None, None, None, None, None, None, None, 2, None) == 1
    assert b"null table" in lib.gdn_last_error()


def test_fused_prefill_reports_uncovered_shapes_without_launching():
    """gdn_prefill_qk / gdn_prefill_fused check their coverage on the host and
    return GDN_ERR_UNSUPPORTED (the caller then takes the two-step path)
    before any HIP call; the dummy device pointers are never dereferenced."""
    from logssms_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.lib()
    d = 0x10000  # 16-byte aligned dummy address

    def qk(width, dk, row_stride=8192):
        return lib.gdn_prefill_qk(d, row_stride, 1, d, width, d, 1, 1, 64, 16, dk, d, 0, 0, 0, d, 1, d, d, 2, 32,
                                  d, 32, 1, 1, d, 32, 1, 1, d, 0, d, 0, d, d, None)

    def fused(width, dk, dv, row_stride=8192):
        return lib.gdn_prefill_fused(d, d, d, row_stride, 1, d, width, d, 1, 1, 64, 16, 32, dk, dv, d, 0, 0, d, d, d,
                                     0, 0, 0, 0, 0, d, 1, d, 1, None, 1, None, 0, None, 0, 0, d, 0.1, None)
    assert qk(3, 128) == 2
    assert b"not covered" in lib.gdn_last_error()
    assert qk(4, 256) == 2
    assert qk(4, 128, row_stride=8190) == 2
    assert fused(3, 128, 128) == 2
    assert b"not covered" in lib.gdn_last_error()
    assert fused(4, 128, 96) == 2
    assert lib.gdn_conv_snapshots(d, 8192, 0, d, 1, 1, 64, 8192, 4, d, 0, 0, 0, d, 1, d, 1, d, 1, 4, None) == 1


def test_split_prefill_refuses_before_its_first_launch():
    """gdn_prefill_split checks what all of its launches need before the first
    one (without a GPU a launch would come back as GDN_ERR_HIP, 3); a 32-bit
    io type would not fit the 16-bit staging."""
    from logssms_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.lib()
    d = 0x10000  # 16-byte aligned dummy address, never dereferenced

    def split(io=1, width=4, dk=128, dv=128, state=d, state_dtype=0, layer=0, writes=d, rows=d, slots=d, count=1,
              out=d, base=d, workspace=d):
        return lib.gdn_prefill_split(d, 8192, io, d, width, d, 1, 1, 1000, 16, 32, dk, dv, d, 24576, 24576, d, 32, 1,
                                     1, d, 32, 1, 1, d, 0, d, 0, state, state_dtype, 1 << 19, 1 << 19, 1 << 14, layer,
                                     base, 1, writes, 1, rows, 1, slots, 1, count, out, 0.1, workspace, 1 << 40, None)

    for kw in (dict(io=0), dict(io=0, state_dtype=0), dict(io=7), dict(dk=256), dict(dk=48), dict(dv=96), dict(dv=16),
               dict(state_dtype=2), dict(io=2, state_dtype=1)):
        assert split(**kw) == 2, kw
        assert b"gdn_prefill_split" in lib.gdn_last_error()
    for kw in (dict(width=1), dict(width=9), dict(state=None), dict(writes=None), dict(out=None), dict(base=None),
               dict(rows=None), dict(slots=None), dict(count=-1), dict(layer=-1), dict(workspace=None),
               dict(workspace=d + 8)):
        assert split(**kw) == 1, kw
        assert b"gdn_prefill_split" in lib.gdn_last_error()


def test_workspace_queries_where_two_launches_pay():
    """The chunked rule alone asks for a workspace from 6 chunks a sequence on
    (7 of heads narrower than 128; below, the second launch costs the host more
    than the GPU gains); the split prefill, one call either way, from 2 on."""
    from logssms_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.lib()
    for n, h, hv, d in ((1, 1, 1, 64), (1, 2, 4, 64), (3, 2, 4, 32), (2, 2, 4, 128), (1, 8, 8, 128)):
        least = 384 if d == 128 else 448
        rule = [lib.gdn_chunk_workspace_bytes(n, n * t, h, hv, d, d, 0) for t in (128, least - 1, least, 4096)]
        assert rule[:2] == [0, 0] and rule[2] > 0 and rule[3] > rule[2], (n, h, hv, d)
        assert lib.gdn_prefill_workspace_bytes(n, n * 127, h, hv, d, d) == 0
    assert lib.gdn_prefill_workspace_bytes(1, 128, 2, 4, 64, 64) > 0
    assert lib.gdn_chunk_workspace_bytes(1, 767, 16, 32, 128, 128, 0) == 0  # 12 tokens a one-launch workgroup
    assert lib.gdn_chunk_workspace_bytes(1, 768, 16, 32, 128, 128, 0) > 0
    assert lib.gdn_chunk_workspace_bytes(1, 8192, 32, 64, 128, 128, 0) == 0  # one launch fills the chip


def test_chunked_rule_refuses_a_misaligned_workspace():
    """The records are stored and read 16 bytes at a time (no launch is made:
    without a GPU one would come back as GDN_ERR_HIP, 3)."""
    from logssms_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.lib()
    d = 0x10000  # 16-byte aligned dummy address, never dereferenced
    shape = (d, d, d, 1, d, d, d, 1, 1, 4096, 2, 4, 128, 128)
    for offset in (2, 4, 8):
        assert lib.gdn_chunk_gated_delta_rule_ws(*shape, d, 0, 1 << 16, 1 << 16, 1 << 14, 0, d, 1, d, 1, None, 0, 64,
                                                 None, 0, 0, 0, 0, 0, 0, d, None, 0.1, d + offset, 1 << 40, None) == 1
        assert b"workspace" in lib.gdn_last_error()
        assert lib.gdn_chunk_gated_delta_rule_logged_ws(*shape, d, 1, 0, d, 1, d, 1, None, 0, 64, d, 0, 8, 64, 1 << 16,
                                                        1 << 15, 512, d, 0, d, 0, 2, 1, 256, d, 0.1, d + offset,
                                                        1 << 40, None) == 1
        assert b"workspace" in lib.gdn_last_error()
