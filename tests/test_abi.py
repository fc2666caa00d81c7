"""The C-ABI library loads and exports exactly what include/emm_kv.h declares (no GPU needed)."""
import ctypes
import os
import re

import pytest

from elasticmm_amd import _lib, library_path

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "emm_kv.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(emm_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    syms = declared_symbols()
    for name in ("emm_kv_pack", "emm_kv_unpack", "emm_copy_blocks", "emm_reshape_and_cache",
                 "emm_reshape_and_cache_fp8", "emm_kv_unpack_dequant_fp8", "emm_concat_rows", "emm_last_error"):
        assert name in syms


def test_library_exports_every_declared_symbol():
    assert os.path.exists(library_path()), "libemm_kv.so has not been built"
    lib = ctypes.CDLL(library_path())
    for name in declared_symbols():
        assert hasattr(lib, name), f"{name} declared in emm_kv.h but not exported"


def test_hooks_exist_only_in_the_hooks_build():
    """The product library carries no benchmark switch or probe: those live in libemm_kv_hooks.so, which
    exports the whole product ABI next to them (so a benchmark can route its calls through it)."""
    from elasticmm_amd.build import hooks_library_path

    hooks_header = open(os.path.join(ROOT, "elasticmm_amd", "csrc", "emm_kv_hooks.h")).read()
    hooks_header = re.sub(r"/\*.*?\*/", "", hooks_header, flags=re.S)
    hook_syms = sorted(set(re.findall(r"\b(emm_hook_[a-z0-9_]+)\s*\(", hooks_header)))
    assert hook_syms == sorted(_lib.HOOK_SIGNATURES) and len(hook_syms) >= 3
    product = ctypes.CDLL(library_path())
    for name in hook_syms + ["emm_set_move_variant"]:
        assert not hasattr(product, name), f"{name} must not be exported by the product library"
    assert os.path.exists(hooks_library_path()), "libemm_kv_hooks.so has not been built"
    hooks = ctypes.CDLL(hooks_library_path())
    for name in hook_syms + declared_symbols():
        assert hasattr(hooks, name), f"{name} missing from the hooks build"
    # nothing in the package reaches for the hooks build on its own
    pkg = os.path.join(ROOT, "elasticmm_amd")
    for fn in os.listdir(pkg):
        if fn.endswith(".py") and fn not in ("_lib.py", "build.py"):
            text = open(os.path.join(pkg, fn)).read()
            assert "hooks" not in text, f"{fn} refers to the hooks build"


def test_binding_table_matches_header():
    assert sorted(_lib.SIGNATURES) == declared_symbols()
    text = open(HEADER).read()
    assert int(re.search(r"#define EMM_MAX_LAYERS (\d+)", text).group(1)) == _lib.EMM_MAX_LAYERS
    assert int(re.search(r"#define EMM_MAX_SEGMENTS (\d+)", text).group(1)) == _lib.EMM_MAX_SEGMENTS
    assert int(re.search(r"#define EMM_KV_ABI_VERSION (\d+)", text).group(1)) == _lib.EMM_KV_ABI_VERSION
    for name in ("EMM_MAX_INLINE_IDS", "EMM_MAX_INLINE_PAIRS", "EMM_MAX_INLINE_PAIRS_TABLES", "EMM_MAX_SLOT_WORDS"):
        assert int(re.search(rf"#define {name} (\d+)", text).group(1)) == getattr(_lib, name)


def test_load_and_argument_errors_without_gpu():
    """Argument validation happens before any HIP call, so it can be exercised on a CPU-only host."""
    lib = _lib.load()
    assert lib.emm_abi_version() == _lib.EMM_KV_ABI_VERSION
    table = _lib.ptr_table([0x1000])
    rc = lib.emm_kv_pack(table, 200, 2, 4, 64, 0x1000, 1, 0x1000, None)
    assert rc == -1 and b"num_layers" in lib.emm_last_error()
    rc = lib.emm_kv_pack(table, 1, 2, 4, -64, 0x1000, 1, 0x1000, None)
    assert rc == -1 and b"negative" in lib.emm_last_error()
    rc = lib.emm_kv_pack(table, 1, 2, 4, 64, None, 1, 0x1000, None)
    assert rc == -1 and b"null" in lib.emm_last_error()
    # empty work is a no-op that never reaches the device
    assert lib.emm_kv_pack(table, 1, 2, 4, 64, None, 0, None, None) == 0
    assert lib.emm_concat_rows(None, None, 0, None, 0, None) == 0
    assert lib.emm_concat_rows(None, None, 1000, None, 0, None) == -1
    with pytest.raises(_lib.EmmError, match="emm_concat_rows"):
        _lib.check(-1, "emm_concat_rows")
    rc = lib.emm_reshape_and_cache(0x1000, 0x1000, 0x1000, 0x1000, 0x1000, 4, 64, 32, 64, 16, None)
    assert rc == -1 and b"stride" in lib.emm_last_error()
    rc = lib.emm_kv_unpack_dequant_fp8(table, 1, 4, 24, 0x1000, 1, 0x1000, 0x1000, 0x1000, 0, None)
    assert rc == -1 and b"multiples of 16" in lib.emm_last_error()


def test_argument_errors_of_the_layout_variants_without_gpu():
    lib = _lib.load()
    P = 0x1000
    # paged-attention layout: head_size must be a multiple of x = 16 / cache element bytes
    rc = lib.emm_reshape_and_cache_paged(P, P, P, P, P, 4, 2, 20, 16, 8, 40, 40, 0, 2, None, None, None)
    assert rc == -1 and b"multiple of x" in lib.emm_last_error()
    rc = lib.emm_reshape_and_cache_paged(P, P, P, P, P, 4, 2, 32, 16, 8, 64, 64, 0, 3, None, None, None)
    assert rc == -1 and b"cache_elem_bytes" in lib.emm_last_error()
    rc = lib.emm_reshape_and_cache_paged(P, P, P, P, P, 4, 2, 32, 16, 8, 64, 64, 0, 1, None, None, None)
    assert rc == -1 and b"scale" in lib.emm_last_error()
    rc = lib.emm_reshape_and_cache_paged(P, P, P, P + 8, P, 4, 2, 32, 16, 8, 64, 64, 0, 2, None, None, None)
    assert rc == -1 and b"16-byte aligned" in lib.emm_last_error()
    rc = lib.emm_reshape_and_cache_paged(P, P, P, P, P, 4, 2, 32, 0, 8, 64, 64, 0, 2, None, None, None)
    assert rc == -1 and b"negative size" in lib.emm_last_error()
    assert lib.emm_reshape_and_cache_paged(P, P, P, P, P, 0, 2, 32, 16, 8, 64, 64, 0, 2, None, None, None) == 0
    t = _lib.ptr_table([P])
    rc = lib.emm_reshape_and_cache_paged_layers(t, t, t, t, 97, P, 4, 2, 32, 16, 8, 64, 64, 0, 2, None, None, None)
    assert rc == -1 and b"num_layers" in lib.emm_last_error()
    # strided flash layout: strides must cover a head row
    rc = lib.emm_reshape_and_cache_strided(t, t, t, t, 1, P, 4, 2, 64, 16, 8, 128, 128, 4096, 32, 64, None)
    assert rc == -1 and b"stride smaller than a head row" in lib.emm_last_error()
    rc = lib.emm_reshape_and_cache_strided(t, t, t, t, 1, P, 4, 2, 64, 16, 8, 100, 128, 4096, 128, 64, None)
    assert rc == -1 and b"token stride" in lib.emm_last_error()
    assert lib.emm_reshape_and_cache_strided(t, t, t, t, 0, P, 4, 2, 64, 16, 8, 128, 128, 4096, 128, 64, None) == 0


def test_argument_errors_of_the_host_table_moves_without_gpu():
    lib = _lib.load()
    P, t, none = 0x1000, _lib.ptr_table([0x1000]), _lib.ptr_table([0])

    def migrate(src=t, src_nb=4, dst=t, dst_nb=4, layers=1, kv=2, chunk=64, si=P, di=P, n=1):
        return lib.emm_kv_migrate_host_ids(src, src_nb, dst, dst_nb, layers, kv, chunk, si, di, n, None)

    def dequant(table=t, layers=1, nb=4, chunk=32, ids=P, n=1, packed=P, ks=P, vs=P, dtype=0):
        return lib.emm_kv_unpack_dequant_fp8_host_ids(table, layers, nb, chunk, ids, n, packed, ks, vs, dtype, None)

    for call, text, kw in [(migrate, b"num_layers", {"layers": 97}), (migrate, b"negative", {"chunk": -1}), (migrate, b"negative", {"dst_nb": -1}),
                           (migrate, b"negative", {"n": -1}), (migrate, b"exceeds", {"src_nb": 2 ** 31}), (migrate, b"exceeds", {"dst_nb": 2 ** 31}),
                           (migrate, b"null", {"src": None}), (migrate, b"null", {"dst": none}), (migrate, b"null index", {"si": None}),
                           (migrate, b"null index", {"di": None}),
                           (dequant, b"num_layers", {"layers": 97}), (dequant, b"negative", {"nb": -1}), (dequant, b"out_dtype", {"dtype": 2}),
                           (dequant, b"null", {"ids": None}), (dequant, b"null", {"packed": None}), (dequant, b"null", {"ks": None}),
                           (dequant, b"null", {"vs": None}), (dequant, b"multiples of 16", {"chunk": 24}),
                           (dequant, b"multiples of 16", {"packed": P + 8}), (dequant, b"aligned", {"table": _lib.ptr_table([P + 8])}),
                           (dequant, b"too large", {"chunk": 2 ** 31})]:
        assert call(**kw) == -1 and text in lib.emm_last_error() and b"host_ids" in lib.emm_last_error(), (kw, lib.emm_last_error())
    for empty in ({"n": 0}, {"layers": 0}, {"chunk": 0}):
        assert migrate(si=None, di=None, **empty) == 0 and dequant(ids=None, packed=None, **empty) == 0


def test_argument_errors_of_the_slot_mapping_without_gpu():
    """Whatever would make the kernel read past its words or write past `out` is refused before the launch."""
    import numpy as np

    lib = _lib.load()
    P, MAX = 0x1000, 2 ** 63 - 1

    def call(starts, offsets, firsts, blocks, bs=16, pad_to=None, out=P, seqs=None, num_blocks=None):
        a = [np.array(x, dtype=np.int64) for x in (starts, offsets, firsts, blocks)]
        return lib.emm_slot_mapping(a[0].ctypes.data, a[1].ctypes.data, a[2].ctypes.data, len(offsets) if seqs is None else seqs,
                                    a[3].ctypes.data, len(blocks) if num_blocks is None else num_blocks, bs,
                                    starts[-1] if pad_to is None else pad_to, out, None)

    def refused(text, *args, **kw):
        assert call(*args, **kw) == -1 and text in lib.emm_last_error(), (args, kw, lib.emm_last_error())

    for kw in ({"seqs": -1}, {"num_blocks": -1}, {"bs": 0}, {"pad_to": -1}):
        refused(b"negative size", [0, 100], [0], [0], [1] * 7, **kw)
    # `pad_to` is the size of `out`: never smaller than the tokens the sequences have
    refused(b"smaller than", [0, 100], [0], [0], [1] * 7, pad_to=99)
    refused(b"smaller than", [0, 100], [0], [0], [1] * 7, pad_to=0)
    refused(b"null pointer", [0, 100], [0], [0], [1] * 7, out=None)
    # counts of which the sum does not fit 64 bits
    refused(b"exceed", [0, 100], [0], [0], [1] * 7, num_blocks=MAX)
    refused(b"exceed", [0, 100], [0], [0], [1] * 7, seqs=2 ** 31 - 1)
    refused(b"exceed", [0, 1], [0], [0], [1] * (_lib.EMM_MAX_SLOT_WORDS - 3))
    for starts, off, first in (([0, 100], 0, 1), ([0, 100], 13, 0), ([0, 17], 0, MAX), ([0, 1], 0, 7), ([0, 1], 16, 0), ([0, 1], -1, 0),
                               ([0, 1], 0, -1), ([0, 0], 0, 0), ([5, 4], 0, 0), ([-1, 1], 0, 0), ([0, 2 ** 31], 0, 0),
                               ([0, MAX], 15, 0), ([MAX, -MAX - 1], 0, 0)):
        refused(b"", starts, [off], [first], [1] * 7, pad_to=max(0, starts[-1]))
    refused(b"too many tokens", [0], [], [], [], pad_to=2 ** 31)
    refused(b"too many tokens", [-1], [], [], [], pad_to=5)
    refused(b"block id", [0, 1], [0], [0], [-1])
    refused(b"block id", [0, 1], [0], [0], [2 ** 32])
    assert call([0], [], [], []) == 0  # nothing to write: never reaches the device


def test_last_error_is_kept_per_thread():
    """Two host threads that fail in different ways each read their own message (the text lives in
    thread-local storage; the transfer manager calls the library from a thread of its own)."""
    import threading

    lib = _lib.load()
    table = _lib.ptr_table([0x1000])
    seen, start = {}, threading.Barrier(2)

    def worker(name, layers, want):
        start.wait()
        for _ in range(200):
            rc = lib.emm_kv_pack(table, layers, 2, 4, 64 if layers == 200 else -64, 0x1000, 1, 0x1000, None)
            msg = lib.emm_last_error()
            if rc != -1 or want not in msg:
                seen[name] = msg
                return
        seen[name] = b"ok"

    a = threading.Thread(target=worker, args=("a", 200, b"num_layers"))
    b = threading.Thread(target=worker, args=("b", 1, b"negative"))
    a.start(), b.start()
    a.join(), b.join()
    assert seen == {"a": b"ok", "b": b"ok"}
    assert lib.emm_kv_pack(table, 1, 2, 4, 64, None, 0, None, None) == 0


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "library_path", lambda: str(tmp_path / "nope.so"))
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        _lib.load()


def test_native_host_side_is_loaded_by_the_appends_only(monkeypatch, tmp_path):
    """pack, unpack and migrate work without the extension module; an append asks for it and says what is missing."""
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_frontend_module", None)
    monkeypatch.setattr(_lib, "frontend_path", lambda: str(tmp_path / "nope.so"))
    lib = _lib.load()
    assert lib.emm_kv_pack(_lib.ptr_table([0x1000]), 1, 2, 4, 64, None, 0, None, None) == 0
    with pytest.raises(RuntimeError, match="native host side"):
        lib.frontend
    monkeypatch.undo()
    assert _lib.load().frontend is _lib.load().frontend


def test_native_host_side_of_another_build_is_refused(monkeypatch):
    """An extension compiled against another header would call the entry points with other signatures; one compiled
    against another torch would read other tensors."""
    module = _lib._load_frontend()
    for version in (0, _lib.EMM_KV_ABI_VERSION - 1, _lib.EMM_KV_ABI_VERSION + 1):
        with pytest.raises(RuntimeError, match="ABI version"):
            module.Frontend(version, 0x1000, 0x1000, 0x1000)
    with pytest.raises(ValueError, match="null entry point"):
        module.Frontend(_lib.EMM_KV_ABI_VERSION, 0x1000, 0, 0x1000)
    with pytest.raises(TypeError):
        module.Frontend(0x1000, 0x1000, 0x1000)
    import torch

    monkeypatch.setattr(_lib, "_frontend_module", None)
    monkeypatch.setattr(torch, "__version__", "1.0.0+rocm0")
    with pytest.raises(RuntimeError, match="built for torch"):
        _lib._load_frontend()
