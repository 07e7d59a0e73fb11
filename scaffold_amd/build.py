"""Builds ``libscaffold_hip.so`` in-tree with hipcc for gfx950 (``make -C scaffold_amd/csrc``) and the C++ host path
``_native.so`` that links it (``make -C scaffold_amd/csrc/host``)."""

from __future__ import annotations

import os
import subprocess
import sys

_HERE = os.path.dirname(os.path.abspath(__file__))


def build(jobs: int = 8, force: bool = False) -> str:
    """Compile every HIP source and link the shared library, then the host path; returns the library's path."""
    csrc = os.path.join(_HERE, "csrc")
    for directory, name in ((csrc, "libscaffold_hip.so"), (os.path.join(csrc, "host"), "_native.so")):
        if force:
            subprocess.run(["make", "-C", directory, "clean"], check=True, stdout=subprocess.DEVNULL)
        proc = subprocess.run(["make", "-C", directory, f"-j{int(jobs)}", f"PY={sys.executable}"], stdout=subprocess.PIPE,
                              stderr=subprocess.STDOUT, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"building {name} failed:\n" + proc.stdout[-8000:])
        if not os.path.exists(os.path.join(_HERE, name)):
            raise RuntimeError(f"make succeeded but {os.path.join(_HERE, name)} is missing")
    return os.path.join(_HERE, "libscaffold_hip.so")


if __name__ == "__main__":
    print(build())
