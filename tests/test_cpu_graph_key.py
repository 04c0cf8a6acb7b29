"""A path tracer's captured frame is replayed while the bytes of its kernel
arguments are the same (wf_graph), so what view_of fills by value must have no
bytes that no member owns: a copy takes them from whatever the stack held, and
the frame would be captured again by chance."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include <type_traits>
#include "kernels.h"
static_assert(std::has_unique_object_representations_v<solhip::%s>, "bytes outside any member");
"""


@pytest.mark.parametrize("name", ["SceneView", "DevTables"])
def test_no_bytes_outside_members(tmp_path, name):
    src = tmp_path / "key.hip"
    src.write_text(SOURCE % name)
    r = subprocess.run(["/opt/rocm/bin/hipcc", "--cuda-host-only", "-fsyntax-only", "-std=c++17",
                        "-I" + os.path.join(ROOT, "sol-rs_amd", "csrc"), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
