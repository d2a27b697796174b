"""The C-ABI library loads and exports every entry point include/*.h declares (no GPU needed:
nothing here launches device work)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    names = []
    inc = os.path.join(ROOT, "include")
    for fn in sorted(os.listdir(inc)):
        if not fn.endswith(".h"):
            continue
        text = open(os.path.join(inc, fn)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        text = re.sub(r"//[^\n]*", "", text)
        for m in re.finditer(r"^\s*(?:const\s+)?[A-Za-z_][A-Za-z0-9_]*\s*\**\s*(sg_[A-Za-z0-9_]+)\s*\(", text, re.M):
            names.append(m.group(1))
    return names


def test_header_declares_entry_points():
    names = declared_functions()
    assert "sg_uniform_cycle_dev" in names and "sg_last_error" in names
    assert len(names) == len(set(names))


def test_library_exports_every_declared_symbol():
    from code_only_amd import _lib
    lib = _lib.load()
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, missing
    # the Python binding covers the same set
    assert set(declared_functions()) == set(_lib.SIGNATURES)


def test_default_params_are_the_reference_values():
    from code_only_amd import _lib
    p = _lib.default_params()
    assert (p.tol, p.maxit, p.ncycle, p.npre, p.npost) == (1e-2, 10, 2, 2, 2)
    assert p.stop_mode == _lib.SG_STOP_REFERENCE
    assert _lib.load().sg_version() >= 1


def test_create_rejects_bad_sizes_without_touching_the_gpu():
    from code_only_amd import _lib
    lib = _lib.load()
    ctx = ctypes.c_void_p()
    for n in (0, 3, 96, 4096):
        rc = lib.sg_uniform_create(ctypes.byref(ctx), n, 1.0, _lib.SG_PREC_FP64)
        assert rc == _lib.SG_ERR_ARG
        assert b"power of two" in lib.sg_last_error()


def test_amr_create_rejects_improper_tables_without_touching_the_gpu():
    import numpy as np
    from code_only_amd import _lib
    from code_only_amd import amr_hierarchy as ah
    lib = _lib.load()
    h = ah.nested(base=4, levels=2, bc=ah.SPHERE)
    ip = lambda a: np.ascontiguousarray(a, np.int32).ctypes.data_as(ctypes.POINTER(ctypes.c_int))
    x0 = np.asarray(h.x0, np.float64)
    keep = [np.ascontiguousarray(a, np.int32) for a in (h.level, h.ijk, h.parent, h.child, h.nbr, h.base_dims)]

    def create(level=None, nbr=None, bc=_lib.SG_BC_SPHERE):
        arrs = list(keep)
        if level is not None:
            arrs[0] = np.ascontiguousarray(level, np.int32)
        if nbr is not None:
            arrs[4] = np.ascontiguousarray(nbr, np.int32)
        ctx = ctypes.c_void_p()
        return lib.sg_amr_create(ctypes.byref(ctx), h.nblk, h.nlev, *[ip(a) for a in arrs], h.h0,
                                 x0.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), bc)

    lvl = h.level.copy()
    lvl[[0, -1]] = lvl[[-1, 0]]         # not ordered by level
    assert create(level=lvl) == _lib.SG_ERR_ARG
    assert b"ordered by level" in lib.sg_last_error() or b"parent" in lib.sg_last_error()
    h3 = ah.nested(base=4, levels=3, bc=ah.SPHERE)
    b3 = int(np.nonzero(h3.level == 2)[0][0])
    nb3 = h3.nbr.copy()
    nb3[b3, 0] = 0                      # level 2 next to level 0
    keep3 = [np.ascontiguousarray(a, np.int32) for a in (h3.level, h3.ijk, h3.parent, h3.child, nb3, h3.base_dims)]
    ctx = ctypes.c_void_p()
    rc = lib.sg_amr_create(ctypes.byref(ctx), h3.nblk, h3.nlev, *[ip(a) for a in keep3], h3.h0,
                           np.asarray(h3.x0, np.float64).ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                           _lib.SG_BC_SPHERE)
    assert rc == _lib.SG_ERR_ARG and b"properly nested" in lib.sg_last_error()
    # a periodic hierarchy may not have open faces
    assert create(bc=_lib.SG_BC_PERIODIC) == _lib.SG_ERR_ARG
    assert b"open face" in lib.sg_last_error()


def test_amr_create_rejects_block_positions_outside_the_level_box():
    """ijk must lie in [0, base_dims << level) before any table built from it is indexed."""
    import numpy as np
    from code_only_amd import _lib
    from code_only_amd import amr_hierarchy as ah
    lib = _lib.load()
    h = ah.nested(base=4, levels=2, bc=ah.SPHERE)
    ip = lambda a: np.ascontiguousarray(a, np.int32).ctypes.data_as(ctypes.POINTER(ctypes.c_int))
    x0 = np.asarray(h.x0, np.float64).ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    for b, bad in ((0, -1), (0, 4), (int(np.nonzero(h.level == 1)[0][0]), 8)):
        ijk = np.ascontiguousarray(h.ijk, np.int32).copy()
        ijk[b, 0] = bad
        arrs = [np.ascontiguousarray(a, np.int32) for a in (h.level, ijk, h.parent, h.child, h.nbr, h.base_dims)]
        ctx = ctypes.c_void_p()
        rc = lib.sg_amr_create(ctypes.byref(ctx), h.nblk, h.nlev, *[ip(a) for a in arrs], h.h0, x0,
                               _lib.SG_BC_SPHERE)
        assert rc == _lib.SG_ERR_ARG and b"out of [0" in lib.sg_last_error(), (b, bad, lib.sg_last_error())


def test_fused_mode_is_only_turned_on_by_its_scope_guard():
    """Every turn-on of the AMR solver's fused launch structure sits in the guard whose destructor turns it
    off, so that a solve that fails half way does not leave the context in it (a HIP error cannot be
    forced from outside without harming the device, so the source is what is checked)."""
    text = open(os.path.join(ROOT, "code_only_amd", "csrc", "amr.hip")).read()
    guard = re.search(r"struct FusedScope \{.*?\n\};", text, re.S).group(0)
    assert "~FusedScope() { s.fused_on = 0; }" in guard
    rest = text.replace(guard, "")
    assert re.findall(r"fused_on = (?!0;)", rest) == []
    assert text.count("struct FusedScope") == 1 and len(re.findall(r"FusedScope fused_scope\(", rest)) == 3
