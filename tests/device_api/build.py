"""Builds the test libraries of this folder (test infrastructure, gfx950, header-only library):
libwc_device_api.so, user kernels that call the tables' device API,
libwc_per_thread.so, host threads whose null stream is their own,
libwc_value_types.so, values of several words, and libwc_host_memory.so, an
operator new that throws."""
from __future__ import annotations

import concurrent.futures
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
REPO = HERE.parents[1]
SOURCES = {"device_api": [], "per_thread": ["-fgpu-default-stream=per-thread"], "value_types": [],
           "host_memory": ["-Wl,-Bsymbolic"]}   # and their own flags
LIB = HERE / "libwc_device_api.so"


def _build(name: str) -> Path:
    from warpcore_amd.build import HIPCC, HIP_FLAGS
    lib = HERE / f"libwc_{name}.so"
    tmp = lib.with_suffix(".so.tmp")
    cmd = [HIPCC, *HIP_FLAGS, *SOURCES[name], "-shared", str(HERE / f"{name}.hip"), "-o", str(tmp)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {name}.hip:\n{proc.stdout}{proc.stderr}")
    tmp.replace(lib)
    return lib


def build() -> Path:
    with concurrent.futures.ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        list(ex.map(_build, SOURCES))
    return LIB


if __name__ == "__main__":
    sys.path.insert(0, str(REPO))
    print(build())
