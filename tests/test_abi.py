"""The C ABI: the library builds, loads, and exports every entry point the header declares
with the argument list the Python binding uses (no GPU needed)."""
import ctypes
import os
import re

import pytest

from gstar_evict import _native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gstar_evict.h")

CTYPES = {"void*": ctypes.c_void_p, "int": ctypes.c_int, "int64_t": ctypes.c_int64, "float": ctypes.c_float,
          "double": ctypes.c_double, "gse_stream_t": ctypes.c_void_p, "char*": ctypes.c_char_p}


def header_prototypes():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    protos = {}
    for m in re.finditer(r"^\s*(int64_t|int|const char\*)\s+(gse_\w+)\s*\(([^)]*)\)\s*;", text, flags=re.M):
        ret, name, args = m.group(1), m.group(2), m.group(3).strip()
        kinds = []
        if args and args != "void":
            for arg in args.split(","):
                arg = " ".join(arg.replace("const", " ").split())
                if "*" in arg:
                    kinds.append("void*")
                else:
                    kinds.append(arg.rsplit(" ", 1)[0])
        protos[name] = (ret.replace("const ", ""), kinds)
    return protos


def test_header_and_binding_agree():
    protos = header_prototypes()
    assert len(protos) >= 15
    assert set(protos) == set(_native.SIGNATURES), set(protos) ^ set(_native.SIGNATURES)
    for name, (ret, kinds) in protos.items():
        res, args = _native.SIGNATURES[name]
        want_ret = {"int": ctypes.c_int, "int64_t": ctypes.c_int64, "char*": ctypes.c_char_p}[ret]
        assert res is want_ret, name
        assert [CTYPES[k] for k in kinds] == list(args), name


def test_library_exports_every_declared_symbol():
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built")
    handle = ctypes.CDLL(_native.LIB_PATH)
    missing = [n for n in header_prototypes() if not hasattr(handle, n)]
    assert not missing, missing
    assert _native.lib().gse_version() >= 100


def test_a_missing_library_raises_instead_of_falling_back(monkeypatch, tmp_path):
    """With no built library every entry point raises NativeError: there is no host path to
    fall back on."""
    monkeypatch.setattr(_native, "LIB_PATH", str(tmp_path / "libgstar_evict.so"))
    monkeypatch.setattr(_native, "_lib", None)
    with pytest.raises(_native.NativeError, match="missing"):
        _native.lib()
    with pytest.raises(_native.NativeError, match="missing"):
        _native.call("gse_decode")


def test_entry_points_reject_bad_arguments_without_a_gpu():
    """Argument validation runs on the host before any launch."""
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built")
    lib = _native.lib()
    rc = lib.gse_decode(None, 0, 0, None, None, 0, 0, None, None, 0, None, 0, None, None, 0, None, 0, 1, None, 0, 0,
                        None, None, None, None, None, 0, 4, 64, 8, 128, 0.125, 512, 0, None, None, 0, 0, None, 0, 0, None, 0,
                        None)
    assert rc != 0 and b"head_dim" in lib.gse_last_error()
    rc = lib.gse_fill(None, 0, None, 0, None, 0, None, 0, None, None, -1, 0, None, None, 0, None)
    assert rc != 0
    assert lib.gse_fill(None, 0, None, 0, None, 0, None, 0, None, None, 0, 0, None, None, 0, None) == 0
    rc = lib.gse_score_flush(None, 12, 512, 64, None, 0, 0, 0, None, 0, None, 0, None, None, None, None, 0, 1, 100,
                             None, None, None, None, 4, 65, 64, 8, 64, 0.125, None, None)
    assert rc != 0 and b"queue_cap" in lib.gse_last_error()
    # Slot rows of 16 KiB or more cannot be one record of the flush's buffer resource.
    rc = lib.gse_score_flush(None, 12, 8192, 64, None, 0, 0, 0, None, 0, None, 0, None, None, None, None, 0, 1, 100,
                             None, None, None, None, 4, 64, 64, 8, 64, 0.125, None, None)
    assert rc == 2 and b"16 KiB" in lib.gse_last_error()  # GSE_ESHAPE
    rc = lib.gse_diagnose_chunk(None, 0, 0, 10, None, 0, 0, None, 0, 10, 0, None, 0, None, None, 0, 0, None, 9, 0,
                                0, None, 0, 1.0, 64, 8, 64, 0.125, None, 0, None)
    assert rc != 0 and b"specs" in lib.gse_last_error()
    rc = lib.gse_diagnose_chunk(None, 0, 0, 10, None, 0, 0, None, 0, 10, 0, None, 0, None, None, 0, 0, None, 2, 0,
                                0, None, 0, 1.0, 64, 8, 64, 0.125, None, 0, None)
    assert rc != 0 and b"null pointer" in lib.gse_last_error()


def test_score_word_layout_matches_the_header():
    """The host packs a row's score delay above GSE_SCORE_DELAY_SHIFT and a block counter's
    kind and block size as the header defines them, as the kernels unpack them."""
    from gstar_evict import requests
    text = open(HEADER).read()
    for name, value in (("GSE_SCORE_DELAY_SHIFT", requests.SCORE_DELAY_SHIFT),
                        ("GSE_SCORE_KIND_BLOCK_STEP", requests.BLOCK_STEP),
                        ("GSE_SCORE_BLOCK_SHIFT", requests.BLOCK_SHIFT)):
        m = re.search(rf"#define\s+{name}\s+(\d+)", text)
        assert m and int(m.group(1)) == value, name
    cfg = dict(name="block_max_2048", budget=4096, prefix=64, recent=256, block=4, score_delay=128,
               block_score="step_max")
    entry = dict(mode=requests.policy_mode(cfg), cfg=cfg)
    assert requests.score_word(entry) == 4 | 2 << 4 | 128 << 8


def test_block_flush_rejects_bad_arguments_without_a_gpu():
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built")
    lib = _native.lib()
    rc = lib.gse_score_flush_blocks(None, 12, 512, 64, None, 0, 0, 0, None, 0, None, 0, None, None, None, None, 0, 1,
                                    100, None, None, None, None, 4, 65, 64, 8, 64, 0.125, None, None)
    assert rc != 0 and b"queue_cap" in lib.gse_last_error()
    rc = lib.gse_prefill_scores(None, 0, 0, 10, None, 0, 0, None, 0, 10, 0, None, 0, 4 | 7 << 4, None, 0, 0, 64, 8,
                                64, 0.125, None, 0, None)
    assert rc != 0 and b"block size" in lib.gse_last_error()
    rc = lib.gse_prefill_scores(None, 0, 0, 10, None, 0, 0, None, 0, 10, 0, None, 0, 1 | 2 << 4, None, 0, 0, 64, 8,
                                64, 0.125, None, 0, None)
    assert rc != 0 and b"block size" in lib.gse_last_error()


def test_logit_flush_rejects_bad_arguments_without_a_gpu():
    """Host-side checks of gse_score_flush_logits and of gse_decode's kept-logit arguments (the
    pointers are host buffers: validation fails before any launch)."""
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built")
    import ctypes
    lib = _native.lib()
    buf = ctypes.create_string_buffer(256)
    p = ctypes.addressof(buf)
    args = [p, 12, 512, 64, p, 0, 0, 0, p, 0, p, 0, p, p, p, p, 0, 1, 100, p, p, p, p, 4, 64, 64, 8, 64, 0.125]
    rc = lib.gse_score_flush_logits(*args, None, 0, p, 1, 100, None, None)
    assert rc != 0 and b"logits" in lib.gse_last_error()
    rc = lib.gse_score_flush_logits(*args, p, 10, p, 1, 100, None, None)
    assert rc != 0 and b"overlap" in lib.gse_last_error()
    rc = lib.gse_decode(p, 0, 0, p, p, 0, 0, p, p, 0, p, 0, p, p, 0, None, 0, 1, p, 0, 0, None, p, p, p, p, 4, 4, 64,
                        8, 64, 0.125, 512, 2, p, None, 1, 10, None, 0, 0, p, 1 << 30, None)
    assert rc != 0 and b"kept logits" in lib.gse_last_error()


def test_noalloc_decode_refuses_a_batch_beyond_its_scratch_without_a_gpu():
    """bs = 1024 at 64 query heads needs more partials than the static scratch holds: refused
    before any device call."""
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built")
    lib = _native.lib()
    assert lib.gse_decode_workspace_bytes(1024, 64, 64) > (9 << 20)
    buf = ctypes.create_string_buffer(256)
    p = ctypes.addressof(buf)
    rc = lib.gse_decode_noalloc(p, 0, 0, p, p, 0, 0, p, p, 0, p, 0, p, p, 0, None, 0, 1, p, 0, 0, None, p, p, p, p,
                                4, 1024, 64, 8, 64, 0.125, 512, 2, None, None, 0, 0, None, 0, 0, None)
    assert rc != 0
    msg = lib.gse_last_error()
    assert b"GSE_DECODE_NOALLOC_SCRATCH_BYTES" in msg and b"bs=1024" in msg


def test_row_descriptors_match_the_header_layout(tmp_path):
    """The ctypes mirrors of gse_boundary_row and gse_live_row have the C structs' size and
    field offsets (a C program built against the header reports them)."""
    import shutil
    import subprocess
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    structs = {"gse_boundary_row": _native.BoundaryRow, "gse_live_row": _native.LiveRow}
    lines = ["#include <stddef.h>", "#include <stdio.h>", '#include "gstar_evict.h"', "int main(void) {"]
    for cname, mirror in structs.items():
        lines.append(f'  printf("{cname} size %zu\\n", sizeof({cname}));')
        for field, _ in mirror._fields_:
            lines.append(f'  printf("{cname} {field} %zu\\n", offsetof({cname}, {field}));')
    lines += ["  return 0;", "}"]
    src = tmp_path / "layout.c"
    src.write_text("\n".join(lines))
    exe = tmp_path / "layout"
    subprocess.run([cc, "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    got = {}
    for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines():
        name, field, value = line.split()
        got[(name, field)] = int(value)
    for cname, mirror in structs.items():
        assert got[(cname, "size")] == ctypes.sizeof(mirror), cname
        for field, _ in mirror._fields_:
            assert got[(cname, field)] == getattr(mirror, field).offset, (cname, field)


def test_prefill_entries_refuse_key_counts_of_2_to_the_31_without_a_gpu():
    """Their kernels index keys in 32 bits: both entries refuse a longer list before any launch (the
    pointers are host buffers)."""
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built")
    lib = _native.lib()
    buf = ctypes.create_string_buffer(256)
    p = ctypes.addressof(buf)
    total, count = 1 << 31, 10
    rc = lib.gse_prefill_scores(p, 0, 0, count, p, 0, 0, p, 0, total, total - count, p, 0, 1, p, 0, 0, 64, 8, 64,
                                0.125, p, 1 << 30, None)
    assert rc == 1 and b"too many keys" in lib.gse_last_error()  # GSE_EINVAL
    rc = lib.gse_diagnose_chunk(p, 0, 0, count, p, 0, 0, p, 0, total, total - count, p, 0, p, p, 0, 0, p, 2, 0,
                                total // 32, p, 0, 1.0, 64, 8, 64, 0.125, p, 1 << 30, None)
    assert rc == 1 and b"too many keys" in lib.gse_last_error()
