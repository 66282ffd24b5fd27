"""Answers of the library's host code (kernel selection, offsets) without a GPU.

The launch rules are functions inside the kernel sources.  query() compiles
such a source for the host alone together with a main() and returns what that
prints: the rule itself answers, not a copy of it.  No device code is built
(the reference to it stays unresolved) and nothing is launched."""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

from conftest import import_submodule


def query(tmp: Path, source: str, body: str) -> list[str]:
    """The lines printed by `body`, the statements of a main() that sees
    csrc/<source>."""
    build = import_submodule("build")
    try:
        hipcc = build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    src, obj, exe = tmp / "query.cpp", tmp / "query.o", tmp / "query"
    src.write_text(f'#include "{source}"\n#include <cstdio>\nint main() {{\n{body}\n}}\n')
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", *build.common_flags(), "-O1", "-c", str(src), "-o", str(obj)],
                   check=True, capture_output=True, text=True, timeout=300)
    rocm = Path(build.clangxx()).parents[2]
    subprocess.run([build.clangxx(), str(obj), "-o", str(exe), "-Wl,--unresolved-symbols=ignore-all",
                    f"-L{rocm}/lib", "-lamdhip64", f"-Wl,-rpath,{rocm}/lib"],
                   check=True, capture_output=True, text=True, timeout=120)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120).stdout.splitlines()
