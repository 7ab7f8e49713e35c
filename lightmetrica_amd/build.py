"""In-tree build of the native libraries.

* ``lightmetrica_amd/liblmgpu.so`` -- the HIP kernels for gfx950 and the C ABI of
  ``include/lmgpu.h``.
* ``lightmetrica_amd/plugin.hip.so`` -- the component plugin (host C++ over the C ABI)
  that registers the GPU scene / renderer / scheduler under the reference's names.

Run ``python -m lightmetrica_amd.build`` (or ``__graft_entry__.build()``).
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
BUILD = ROOT / "_build"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# Packed FP32 instructions are disabled for all device code.
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-result",
    "-I", str(ROOT / "include"),
]
HOST_FLAGS = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-I", str(ROOT / "include")]

LIB_SOURCES = ["lmgpu_api.hip", "trace_kernels.hip", "pt_kernels.hip", "ray_order.hip", "bvh_build.cpp"]
LIB = PKG / "liblmgpu.so"


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError("build failed:\n" + " ".join(cmd) + "\n" + proc.stdout)
    if proc.stdout.strip():
        # Keep compiler diagnostics visible, minus the known host-pass note on the packed-fp32 feature.
        lines = [l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l]
        if lines:
            print("\n".join(lines), file=sys.stderr)


def _compile(src: Path) -> Path:
    obj = BUILD / (src.name + ".o")
    if src.suffix == ".hip":
        cmd = [HIPCC, *HIP_FLAGS, "-c", str(src), "-o", str(obj)]
    else:
        cmd = [HIPCC, *HOST_FLAGS, "-c", str(src), "-o", str(obj)]
    _run(cmd)
    return obj


def build_lib(jobs: int = 4) -> Path:
    BUILD.mkdir(exist_ok=True)
    srcs = [CSRC / s for s in LIB_SOURCES]
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB.with_suffix(".so.tmp")
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs), "-lpthread"])
    os.replace(tmp, LIB)
    return LIB


PLUGIN = PKG / "plugin.hip.so"
DRIVER = ROOT / "tests" / "native" / "plugin_driver"


def build_plugin() -> Path:
    """plugin.hip.so: host C++ over the C ABI, linked against liblmgpu.so next to it."""
    tmp = PLUGIN.with_suffix(".so.tmp")
    _run(["g++", *HOST_FLAGS, "-shared", str(CSRC / "plugin" / "plugin_hip.cpp"), "-o", str(tmp),
          "-L", str(PKG), "-llmgpu", "-Wl,-rpath,$ORIGIN", "-ldl"])
    os.replace(tmp, PLUGIN)
    return PLUGIN


def build_driver() -> Path:
    """The C++ host that loads plugins from a directory like the reference's tests do."""
    tmp = DRIVER.with_name(DRIVER.name + ".tmp")
    _run(["g++", *HOST_FLAGS, str(ROOT / "tests" / "native" / "plugin_driver.cpp"), "-o", str(tmp), "-ldl", "-lpthread"])
    os.replace(tmp, DRIVER)
    return DRIVER


BVH_CHECK = ROOT / "tests" / "native" / "bvh_check"


def build_bvh_check() -> Path:
    """The host-side BVH invariant checker (builder source compiled in, no GPU)."""
    tmp = BVH_CHECK.with_name(BVH_CHECK.name + ".tmp")
    _run(["g++", *HOST_FLAGS, str(ROOT / "tests" / "native" / "bvh_check.cpp"), str(CSRC / "bvh_build.cpp"), "-o",
          str(tmp), "-lpthread"])
    os.replace(tmp, BVH_CHECK)
    return BVH_CHECK


PACKED_CHECK = ROOT / "tests" / "native" / "packed_check"


def build_packed_check() -> Path:
    """The host-side checker of the packed nodes (the kernels' box arithmetic compiled in, no GPU)."""
    tmp = PACKED_CHECK.with_name(PACKED_CHECK.name + ".tmp")
    _run(["g++", *HOST_FLAGS, str(ROOT / "tests" / "native" / "packed_check.cpp"), str(CSRC / "bvh_build.cpp"), "-o",
          str(tmp), "-lpthread"])
    os.replace(tmp, PACKED_CHECK)
    return PACKED_CHECK


HOST_IO_CHECK = ROOT / "tests" / "native" / "host_io_check"


def build_host_io_check() -> Path:
    """The checker of the host copy team (no GPU)."""
    tmp = HOST_IO_CHECK.with_name(HOST_IO_CHECK.name + ".tmp")
    _run(["g++", *HOST_FLAGS, str(ROOT / "tests" / "native" / "host_io_check.cpp"), "-o", str(tmp), "-lpthread"])
    os.replace(tmp, HOST_IO_CHECK)
    return HOST_IO_CHECK


def build_all(jobs: int = 4) -> None:
    build_lib(jobs)
    build_plugin()
    build_driver()
    build_bvh_check()
    build_packed_check()
    build_host_io_check()


if __name__ == "__main__":
    build_all()
    print(f"built {LIB}")
