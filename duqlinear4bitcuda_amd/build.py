"""Build libduq_hip.so (kernels and C ABI, hipcc for gfx950) and _duq_host.so (the Python ops' host side in native code, g++,
for the Python and the torch that run this) in-tree: ``python -m duqlinear4bitcuda_amd.build``.  The package runs with the
first alone (``make -C duqlinear4bitcuda_amd/csrc lib``)."""
from __future__ import annotations

import os
import subprocess
import sys

_HERE = os.path.dirname(os.path.abspath(__file__))


def build(clean: bool = True, jobs: int = 8, verbose: bool = False) -> str:
    csrc = os.path.join(_HERE, "csrc")
    if clean:
        subprocess.run(["make", "-C", csrc, "clean"], check=True, capture_output=not verbose)
    res = subprocess.run(["make", "-C", csrc, f"-j{jobs}"], capture_output=not verbose, text=True)
    if res.returncode != 0:
        sys.stderr.write((res.stdout or "") + (res.stderr or ""))
        missing = [n for n in ("libduq_hip.so", "_duq_host.so") if not os.path.exists(os.path.join(_HERE, n))]
        raise RuntimeError(f"build failed, missing: {', '.join(missing) or 'nothing, but a file could not be renewed'}")
    return os.path.join(_HERE, "libduq_hip.so")


if __name__ == "__main__":
    print(build(verbose=True))
