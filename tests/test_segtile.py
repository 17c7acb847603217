"""The entry numbers of the segmented reduce's tiles (csrc/segtile.hpp) at the
largest triplet counts an assembly accepts, 2^31 - 1, compiled on the CPU."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "libuipc_amd", "csrc")


@pytest.mark.parametrize("m", [0, 1, 256, 257, 2**31 - 353, 2**31 - 352, 2**31 - 256, 2**31 - 255, 2**31 - 2, 2**31 - 1])
def test_entries_at_the_limits(tmp_path, m):
    """constant expressions, so that an overflow does not compile: the tiles of m
    entries, their first and last entries, the staged ones past them, and those of
    the tile past the last (which a workgroup asks for too)"""
    nt = -(-m // 256)
    checks = [f"mi::seg_tiles({m}u) == {nt}"]
    for t in {max(nt - 1, 0), nt}:
        for k in (0, 255, 256, 256 + 95):
            checks.append(f"(mi::seg_entry({t}u, {k}) < {m}u) == {str(256 * t + k < m).lower()}")
            checks.append(f"mi::seg_entry({t}u, {k}) == {256 * t + k}ll")
    src = tmp_path / "limits.cpp"
    src.write_text('#include "segtile.hpp"\n' + "".join(f"static_assert({c});\n" for c in checks))
    r = subprocess.run(["g++", "-std=c++17", "-Wall", "-Wno-sign-compare", "-fsyntax-only", "-I", CSRC, str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
