"""The native caller of the C ABI (umdk_amd/_camcall.so) on the CPU: argument conversion, the library's errors, and the
workspace it asks for.  Nothing launches: every call fails in its validation or in its allocation."""
import shutil
import subprocess
import sys

import numpy as np
import pytest

from umdk_amd import _lib


def raw(name, *args, alloc=None, ws=None, have=0):
    return getattr(_lib._calls(), name)(alloc, ws, have, 0, *args)


def test_library_errors_keep_their_type_and_text():
    with pytest.raises(_lib.CamHipError, match=r"^camhipMoeRouteGetWorkspaceSize failed \(\d+\): moe_route: numExperts 0"):
        raw("camhipMoeRoute", 16, None, 4, 0, 1, 16, 16, None)
    with pytest.raises(_lib.CamHipError, match="logits must not be NULL"):
        raw("camhipMoeRoute", None, None, 4, 8, 2, 16, 16, None)
    # the launch phase: a workspace too small (checked before anything runs)
    with pytest.raises(_lib.CamHipError, match=r"^camhipDispatchLayout failed \(\d+\): dispatch_layout: workspace of 8 bytes"):
        raw("camhipDispatchLayout", 16, 64, 1, 8, 2, None, 16, None, 16, ws=16, have=8)


@pytest.mark.parametrize("args", [(16, None, 4.0, 8, 2, 16, 16, None), (16, None, None, 8, 2, 16, 16, None),
                                  ("x", None, 4, 8, 2, 16, 16, None), (16, None, 4, 8, 2, 16, 16)])
def test_wrong_arguments_are_type_errors(args):
    with pytest.raises(TypeError):
        raw("camhipMoeRoute", *args)


@pytest.mark.parametrize("kind", [np.int64, np.int32, np.uint8, np.array])
def test_sizes_of_any_integer_type(kind):
    sizes = [kind(v) for v in (64, 1, 8, 2)]
    want = _lib.workspace_size("camhipDispatchLayout", 1, 64, 1, 8, 2, None, 1, None, 1)
    seen = []

    def alloc(n):
        seen.append(n)
        raise MemoryError("no room")

    with pytest.raises(MemoryError):
        raw("camhipDispatchLayout", 16, *sizes, None, 16, None, 16, alloc=alloc)
    assert seen == [want]


def test_every_entry_point_is_there():
    for name in _lib.SIGNATURES:
        with pytest.raises(TypeError, match=name):
            raw(name)


def test_workspace_size_and_failed_allocation():
    want = _lib.workspace_size("camhipDispatchLayout", 1, 64, 1, 8, 2, None, 1, None, 1)
    seen = []

    def alloc(n):
        seen.append(n)
        raise MemoryError("no room")

    with pytest.raises(MemoryError, match="no room"):
        raw("camhipDispatchLayout", 16, 64, 1, 8, 2, None, 16, None, 16, alloc=alloc)
    assert seen == [want]


def test_calls_go_to_the_loaded_library(tmp_path):
    # a library chosen through LIB_PATH (a diagnostic build) takes the calls too, and no other one is loaded
    copy = tmp_path / "libother.so"
    shutil.copy(_lib.LIB_PATH, copy)
    code = f"""
from umdk_amd import _lib
_lib.LIB_PATH = {str(copy)!r}
try:
    _lib.call("camhipMoeRoute", None, None, 4, 8, 2, 16, 16, None, stream=0)
except _lib.CamHipError as e:
    assert "logits must not be NULL" in str(e)
maps = open("/proc/self/maps").read()
assert {str(copy)!r} in maps and "libcamhip.so" not in maps, "two libraries"
"""
    subprocess.run([sys.executable, "-c", code], check=True, cwd=_lib._HERE + "/..")
