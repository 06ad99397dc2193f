"""The C-ABI library builds for gfx950 without a GPU, loads, and exports every symbol the header declares
(no compute calls here: those are the -m gpu tests)."""
import ctypes
import os
import re

from nanollama_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "nanollama_hip.h")).read()
    return sorted(set(re.findall(r"NL_API\s+[\w\s\*]+?\b(nl_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    _lib.build()
    L = ctypes.CDLL(_lib.LIB_PATH)
    names = _declared()
    assert len(names) >= 25, names
    missing = [n for n in names if not hasattr(L, n)]
    assert not missing, missing
    assert set(_lib.EXPORTS) <= set(names)


def test_probes_work_without_a_gpu():
    L = _lib.lib()
    assert L.nl_abi_version() == 1
    assert L.nl_device_count() >= 0
    assert L.nl_kernel_kind_name(6) == b"lm_head" and L.nl_kernel_kind_name(99) == b""


def test_create_without_gpu_fails_loudly_or_succeeds_with_one():
    L = _lib.lib()
    cfg = _lib.NlConfig(2, 128, 4, 2, 32, 512, 512, 64, 1e-5, 10000.0, 0, 0, 1, 0, 0, 1, 0)
    h = ctypes.c_void_p()
    rc = L.nl_create(ctypes.byref(cfg), ctypes.byref(h))
    if L.nl_device_count() == 0:
        assert rc == -3 and b"no HIP device" in L.nl_last_error(None)   # NL_ERR_HIP, never a CPU fallback
    else:
        assert rc == 0
        L.nl_destroy(h)
    bad = _lib.NlConfig(2, 100, 4, 2, 25, 512, 512, 64, 1e-5, 10000.0, 0, 0, 1, 0, 0, 1, 0)
    assert L.nl_create(ctypes.byref(bad), ctypes.byref(h)) in (-1, -2, -3)


def test_create_group_without_gpu_fails_loudly():
    # nl_create_group (one process, N GPUs): argument errors are reported before any device is touched; with no device the
    # rank engines cannot be created -- NL_ERR_HIP, never a CPU fallback
    L = _lib.lib()
    cfg = _lib.NlConfig(2, 256, 4, 4, 64, 512, 512, 64, 1e-5, 10000.0, 0, 0, 1, 0, 0, 1, 0)
    h = ctypes.c_void_p()
    ids = (ctypes.c_int * 8)(0, 0, 0, 0, 0, 0, 0, 0)
    assert L.nl_create_group(ctypes.byref(cfg), ids, 3, ctypes.byref(h)) == -2 and b"2, 4 or 8" in L.nl_last_error(None)
    assert L.nl_create_group(ctypes.byref(cfg), None, 2, ctypes.byref(h)) == -1
    rc = L.nl_create_group(ctypes.byref(cfg), ids, 2, ctypes.byref(h))
    if L.nl_device_count() == 0:
        assert rc == -3 and b"no HIP device" in L.nl_last_error(None) and not h.value
    else:
        assert rc == 0
        L.nl_destroy(h)


# What "using the oracle" looks like in source: an import, an include, a dlopen / CDLL of the checker's library, or a path
# into oracle/.  (A comment that merely names the oracle as the thing a kernel is held to is not a use; an earlier tree
# went red on exactly such a comment.)
_ORACLE_USE = [
    re.compile(r"^\s*(from|import)\s+oracle\b", re.M),                 # import oracle / from oracle import ...
    re.compile(r"import_module\(\s*['\"]oracle"), re.compile(r"__import__\(\s*['\"]oracle"),
    re.compile(r"#\s*include\s*[<\"][^>\"]*oracle"),                   # #include "…oracle…"
    re.compile(r"libnl_oracle|nl_oracle\.(c|h|so)|oracle\.py"),          # the checker's files by name
    re.compile(r"(dlopen|CDLL|LoadLibrary)\s*\([^)]*oracle"),
    re.compile(r"['\"][^'\"\n]*\boracle/[^'\"\n]*['\"]"),             # a string literal holding a path into oracle/
]


def _oracle_uses(src):
    return [m.group(0) for rx in _ORACLE_USE for m in rx.finditer(src)]


def test_oracle_use_detector_sees_real_uses_and_ignores_prose():
    assert _oracle_uses("from oracle import oracle\n") and _oracle_uses("    import oracle\n")
    assert _oracle_uses('#include "../../oracle/nl_oracle.c"') and _oracle_uses('dlopen("x/oracle/lib.so", 2)')
    assert _oracle_uses('p = os.path.join(ROOT, "oracle/libnl_oracle.so")') and _oracle_uses("ctypes.CDLL(oracle_path)")
    assert not _oracle_uses("// held to the oracle's logits within 1e-4 (tests/test_gpu_parity.py)")
    assert not _oracle_uses("# the CPU oracle (oracle/) is test infrastructure")


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "nanollama_amd")
    seen = 0
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".cpp", ".c")):
                src = open(os.path.join(dirpath, f), errors="ignore").read()
                assert not _oracle_uses(src), (f, _oracle_uses(src))
                seen += 1
    assert seen >= 20
