"""The C-ABI library loads and exports every symbol include/neus2_amd.h declares (no GPU needed)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "neus2_amd.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(n2_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    assert "n2_grid_forward" in syms and "n2_last_error" in syms and len(syms) >= 10


def test_library_exports_every_declared_symbol():
    from neus2_amd import capi
    if not os.path.exists(capi.LIB_PATH):
        from neus2_amd.build import build_library
        build_library()
    lib = ctypes.CDLL(capi.LIB_PATH)
    missing = [s for s in declared_symbols() if not hasattr(lib, s)]
    assert not missing, missing


def test_nobody_sees_the_library_before_its_signatures_are_set(monkeypatch):
    """A thread that calls lib() meanwhile must not get it: Python's numbers go in as 32 bits where a function has no argtypes."""
    from neus2_amd import capi
    seen, real = [], capi.C.CDLL

    class Watched(real):
        def __getattr__(self, name):
            seen.append(capi._lib)
            return super().__getattr__(name)

    monkeypatch.setattr(capi, "_lib", None)
    monkeypatch.setattr(capi.C, "CDLL", Watched)
    L = capi.lib()
    assert len(seen) > len(capi._SIGNATURES) and not any(seen)
    assert capi.lib() is L and L.n2_grid_forward.argtypes[2] is ctypes.c_void_p


def test_signatures_are_the_headers():
    from neus2_amd import capi
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "neus2_amd.h")).read(), flags=re.S)
    kind = lambda a: "p" if "*" in a or "n2_stream_t" in a or "[" in a else {"uint32_t": "u", "float": "f", "uint64_t": "q"}.get(a.split()[0], "i")
    for name, signature in capi._SIGNATURES.items():
        arguments = re.search(r"\b%s\s*\((.*?)\)" % name, text, re.S).group(1).split(",")
        assert "".join(kind(a.replace("const ", "").strip()) for a in arguments) == signature, name


def test_host_only_entry_points_work_without_gpu():
    """Object creation and the level table are pure host code."""
    import numpy as np
    from neus2_amd import capi
    L = capi.lib()
    h = ctypes.c_void_p()
    assert L.n2_grid_create(16, 2, 19, 16, ctypes.c_float(1.447), ctypes.byref(h)) == 0
    assert L.n2_grid_n_params(h) == 12599920 and L.n2_grid_output_width(h) == 32
    res = np.zeros(16, np.uint32)
    off = np.zeros(17, np.uint32)
    assert L.n2_grid_level_table(h, None, capi.ptr(res), None, capi.ptr(off)) == 0
    assert res.tolist() == [16, 24, 34, 49, 71, 102, 147, 213, 308, 445, 644, 932, 1349, 1951, 2823, 4085]
    assert int(off[-1]) == 6299960
    L.n2_grid_destroy(h)
    # error behaviour: unsupported feature count, message available
    assert L.n2_grid_create(16, 4, 19, 16, ctypes.c_float(1.447), ctypes.byref(h)) == 3
    assert b"n_features_per_level" in L.n2_last_error()
    assert L.n2_grid_create(0, 2, 19, 16, ctypes.c_float(1.447), ctypes.byref(h)) == 1


def test_level_table_matches_oracle(oracle):
    import numpy as np
    from neus2_amd import capi
    L = capi.lib()
    for cfg in [(16, 19, 16, 1.447), (14, 19, 16, 1.4472692012786865), (8, 14, 4, 2.0), (5, 4, 2, 1.5)]:
        h = ctypes.c_void_p()
        assert L.n2_grid_create(cfg[0], 2, cfg[1], cfg[2], ctypes.c_float(cfg[3]), ctypes.byref(h)) == 0
        g = oracle.Grid(*cfg)
        sc, res, ent, off = (np.zeros(cfg[0], np.float32), np.zeros(cfg[0], np.uint32), np.zeros(cfg[0], np.uint32),
                             np.zeros(cfg[0] + 1, np.uint32))
        assert L.n2_grid_level_table(h, capi.ptr(sc), capi.ptr(res), capi.ptr(ent), capi.ptr(off)) == 0
        assert np.array_equal(sc, g.scale) and np.array_equal(res, g.resolution)
        assert np.array_equal(ent, g.entries) and np.array_equal(off, g.offset)
        L.n2_grid_destroy(h)


@pytest.mark.parametrize("res", [(2, 32, 64), (2, 1 << 15, 1 << 15), (3, 6, 1000), (16, 16, 16), (16, 512, 512), (17, 9, 33), (33, 5, 7), (63, 512, 512), (65, 64, 64), (512, 512, 512)])
def test_marching_cubes_workspace_of_short_rows(res):
    """A word of bits takes 72 bytes and has at least sixteen points where a plane has them; 4 KiB for what is per block."""
    from neus2_amd import capi
    L = capi.lib()
    L.n2_marching_cubes_workspace_bytes.restype = ctypes.c_uint64
    n = res[0] * res[1] * res[2]
    assert 0 < L.n2_marching_cubes_workspace_bytes((ctypes.c_uint32 * 3)(*res)) <= 4.6 * n + 4096


def test_cpp_shim_host_checks():
    """The header-only C++ shim (tcnn method names over the C ABI) compiles with the host compiler and its
    host-only behaviour holds: shapes, parameter counts, matrix views, errors as std::runtime_error."""
    import subprocess
    from neus2_amd.build import build_library, build_shim_check
    build_library()
    exe = build_shim_check()
    r = subprocess.run([exe, "host"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    assert "shim host checks ok" in r.stdout
