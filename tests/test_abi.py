"""The C-ABI library loads and exports every symbol include/moe_mi355.h declares
(no compute calls: this runs without a GPU)."""
import os
import re

import pytest

from moe_gen_amd import _native as N

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "moe_mi355.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = re.findall(r"\b(moe_[a-z0-9_]+)\s*\(", text)
    return sorted(set(names))


def test_header_declares_the_expected_entry_points():
    names = declared_functions()
    for must in ("moe_router", "moe_dispatch", "moe_grouped_swiglu_bf16", "moe_grouped_swiglu_w8a16",
                 "moe_combine", "moe_stage_create", "moe_stage_acquire", "moe_stage_release", "moe_last_error"):
        assert must in names


def test_library_exports_every_declared_symbol():
    lib = N.lib()
    for name in declared_functions():
        assert hasattr(lib, name), f"{name} is declared in moe_mi355.h but not exported"


def test_binding_covers_header_exactly():
    assert sorted(N.SIGNATURES) == declared_functions()


def test_version_and_error_string():
    lib = N.lib()
    assert b"gfx950" in lib.moe_version()
    assert isinstance(N.last_error(), str)


def test_argument_validation_needs_no_gpu():
    """Entry points reject bad arguments on the host before touching the device."""
    import ctypes
    lib = N.lib()
    p = N.RouterParams(4, 12, 8, 2, 1, 1, 0, 0, 0, 1, 0, 0, 1e-20, 1.0)      # hidden not a multiple of 8
    rc = lib.moe_router(1, 1, None, ctypes.byref(p), 1, 1, None, None)
    assert rc == -1 and "hidden" in N.last_error()
    p = N.RouterParams(4, 16, 8, 2, 1, 1, 7, 0, 0, 1, 0, 0, 1e-20, 1.0)       # unknown scoring function
    assert lib.moe_router(1, 1, None, ctypes.byref(p), 1, 1, None, None) == -1
    assert "scoring" in N.last_error()
    assert lib.moe_router_rmsnorm(1, 1, 1e-6, 1, None, ctypes.byref(p), 2, 1, 1, None, None) == -1     # (before the norm is launched)
    assert "scoring" in N.last_error()
    assert lib.moe_combine(1, 1, None, 1, None, 4, 99, 64, 0, 1, None) == -1 and "top_k" in N.last_error()
    assert lib.moe_grouped_swiglu_bf16(1, 8, None, 1, 1, 1, 1, 8, 2, 100, 64, 1, 1, 3, None, 0, None) == -1
    assert "hidden" in N.last_error()
    assert lib.moe_dispatch(1, 4, 2, 300, 1, 1, 1, 1, None, None, 0, None, None, 0, None) == -1


def test_joint_calls_check_their_groups_first():
    """No expert, or fewer than no rows: an error code (a division by zero would end the process), and a bad second group
    is refused before the first one is launched.  In a process of its own, which reports how it ended."""
    import subprocess
    import sys
    code = """
import ctypes
from moe_gen_amd import _native as N
lib = N.lib()
group = lambda rows, E, inter: N.MlpGroup(1, 8, rows, None, 1, 1, 1, 1, 1, 1, 1, E, inter, 0, 0, 1, 1, None, 0)
good, none = group(8, 2, 64), group(8, 1, 64)
for bad in (group(8, 0, 64), group(-1, 2, 64), group(8, -1, 64)):
    assert lib.moe_shared_joins(ctypes.byref(bad), ctypes.byref(none), 64) == 0
    for fp8 in (0, 1):
        assert lib.moe_grouped_swiglu_joint(ctypes.byref(bad), ctypes.byref(none), 64, fp8, 3, None) == -1, N.last_error()
assert lib.moe_grouped_swiglu_joint(ctypes.byref(good), ctypes.byref(group(8, 1, 65)), 64, 0, 3, None) == -1 and "intermediate" in N.last_error()
assert lib.moe_grouped_swiglu_joint(ctypes.byref(good), ctypes.byref(none), 64, 0, 9, None) == -1 and "phases" in N.last_error()
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stderr)


@pytest.mark.parametrize("fp8", [0, 1])
def test_a_layer_call_holds_tile_counters_only_where_it_can_claim_tiles(fp8):
    """4 KiB that the dispatch would clear: from a mean of 128 rows per expert on (64 experts, each with every token), or, with a
    shared expert, from 128 tokens on.  Of these sizes every other buffer grows by a multiple of 256 bytes a token."""
    import ctypes
    lib, first = N.lib(), 128

    def need(n, k, shared):
        p = N.RouterParams(n, 128, 64, k, 1, 1, 0, 0, 0, 1, 0, 0, 1e-20, 1.0)
        group = lambda E: N.MlpGroup(1, 1, 0, None, 1, 1, 1, 1, 1, 1, None, E, 128, 0, fp8, None, None, None, 0)
        r, s = group(64), group(1)
        a = N.LayerArgs(1, None, 1, None, ctypes.addressof(p), ctypes.addressof(r), ctypes.addressof(s) if shared else None, 1, 1, 1, None, 1,
                        None, 0, 0.0, 0, 1)
        size = lib.moe_layer_workspace_bytes(ctypes.byref(a))
        assert size > 0, N.last_error()
        return size - lib.moe_dispatch_workspace_bytes(n, k, 64)

    for k, shared in ((64, False), (64, True), (32, True)):
        step = [need(n + 1, k, shared) - need(n, k, shared) for n in range(first - 4, first + 4)]
        assert [d - min(step) >= 4096 for d in step] == [n + 1 == first for n in range(first - 4, first + 4)], (k, shared, step)
    assert len({need(n + 8, 32, False) - need(n, 32, False) for n in range(120, 136, 8)}) == 1          # a mean of 64
