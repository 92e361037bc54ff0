"""Builds the HIP shared library in-tree: ``liteinfer_amd/_lib/libliteinfer_amd.so``.

Every ``csrc/*.hip`` file is compiled for gfx950 by ``hipcc`` and linked into
one shared library with a plain C ABI (``include/liteinfer_amd.h``). The
library is loaded with ctypes and depends on no torch; it links the HIP runtime
by soname, which resolves to the copy the process already has loaded when
torch was imported first. Beside it the host compiler builds
``csrc/fast_calls.cpp``, a Python extension against this interpreter and its
torch, whose file name carries a digest of both.

Run as ``python -m liteinfer_amd._build``.
"""

from __future__ import annotations

import concurrent.futures
import hashlib
import os
import shutil
import subprocess
import sys
import tempfile
from pathlib import Path

PACKAGE_DIR = Path(__file__).resolve().parent
CSRC_DIR = PACKAGE_DIR / "csrc"
LIB_DIR = PACKAGE_DIR / "_lib"
LIB_PATH = LIB_DIR / "libliteinfer_amd.so"
INCLUDE_DIR = PACKAGE_DIR.parent / "include"

OFFLOAD_ARCH = "gfx950"

# Packed fp32 instructions stay off: some of their forms have given wrong
# results on these machines with no error raised.
DEVICE_FLAGS = [
    f"--offload-arch={OFFLOAD_ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fno-honor-nans",
    "-Wall",
    "-Wno-unused-function",
]


# Per-source extra flags. prefill_mfma.hip: its persistent kernel claims the
# next unit with an atomic whose old value it reads only at the unit's end;
# the wave-level atomic optimizer would read it back at once, stalling the
# wave on every load in flight.
SOURCE_FLAGS = {
    "prefill_mfma.hip": ["-mllvm", "-amdgpu-atomic-optimizer-strategy=None"],
}


def source_hash() -> str:
    """16 hex digits of SHA-256 over every source and header and the compile flags.

    The build passes it into the library (``li_build_id``); the loader
    recomputes it from the files beside the package and refuses a mismatch.
    """
    h = hashlib.sha256()
    files = sorted(p for p in CSRC_DIR.iterdir() if p.is_file() and p.suffix in (".hip", ".h", ".cpp"))
    files += sorted(INCLUDE_DIR.glob("*.h"))
    for path in files:
        h.update(path.name.encode() + b"\0" + path.read_bytes() + b"\0")
    h.update(repr((DEVICE_FLAGS, sorted(SOURCE_FLAGS.items()))).encode())
    return h.hexdigest()[:16]


def hipcc() -> str:
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    path = Path(rocm) / "bin" / "hipcc"
    if path.exists():
        return str(path)
    found = shutil.which("hipcc")
    if found is None:
        raise RuntimeError("hipcc not found: set ROCM_PATH or put hipcc on PATH")
    return found


def sources() -> list[Path]:
    return sorted(CSRC_DIR.glob("*.hip"))


def _compile(src: Path, obj: Path, build_id: str) -> None:
    cmd = [hipcc(), *DEVICE_FLAGS, *SOURCE_FLAGS.get(src.name, []), f'-DLI_BUILD_ID="{build_id}"',
           "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass does not know the packed-fp32 feature and says so; that
    # warning is harmless and is the only output dropped.
    noise = "is not a recognized feature for this target"
    err = "\n".join(line for line in proc.stderr.splitlines() if noise not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)


# Host flags and libraries of csrc/fast_calls.cpp.
FAST_CALLS_FLAGS = ["-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", "-w"]
FAST_CALLS_LIBS = ["-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10"]


def fast_calls_path() -> Path:
    """Where the extension for this interpreter and this torch lies.

    Its code reads torch's and Python's objects at offsets fixed when it was
    compiled, so the name carries a digest of what these depend on: an
    extension built for others is not found.
    """
    import sysconfig

    import torch

    abi = (torch.__version__, torch.version.git_version, torch._C._GLIBCXX_USE_CXX11_ABI, sys.implementation.cache_tag,
           sysconfig.get_config_var("SOABI"), FAST_CALLS_FLAGS, FAST_CALLS_LIBS)
    return LIB_DIR / f"_fast_calls.{hashlib.sha256(repr(abi).encode()).hexdigest()[:16]}.so"


def _compile_fast_calls(build_id: str) -> None:
    """csrc/fast_calls.cpp, the eager calls' host side: a Python extension against this interpreter's torch."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    path = fast_calls_path()
    for stale in LIB_DIR.glob("_fast_calls*"):
        stale.unlink()
    torch_lib = Path(torch.__file__).resolve().parent / "lib"
    out_tmp = LIB_DIR / (path.name + ".tmp")
    cmd = [shutil.which("g++") or "c++", *FAST_CALLS_FLAGS,
           f'-DLI_BUILD_ID="{build_id}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-I{p}" for p in (*cpp_extension.include_paths(), sysconfig.get_paths()["include"])),
           str(CSRC_DIR / "fast_calls.cpp"), "-o", str(out_tmp), f"-L{torch_lib}", *FAST_CALLS_LIBS]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on fast_calls.cpp:\n{proc.stderr}")
    os.replace(out_tmp, path)


def build(verbose: bool = False) -> Path:
    """Compile every source and link the libraries. Always rebuilds.

    Without the eager calls' extension (no host compiler, no headers of torch
    or Python) the library still serves every call, so its failure is reported
    and does not end the build.
    """
    LIB_DIR.mkdir(parents=True, exist_ok=True)
    build_id = source_hash()
    with tempfile.TemporaryDirectory(prefix="liteinfer_amd_build_") as tmp:
        objs = []
        jobs = []
        with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
            fast_calls = pool.submit(_compile_fast_calls, build_id)
            for src in sources():
                obj = Path(tmp) / (src.stem + ".o")
                objs.append(obj)
                jobs.append(pool.submit(_compile, src, obj, build_id))
            for job in jobs:
                job.result()
        try:
            fast_calls.result()
        except (ImportError, OSError, RuntimeError) as e:
            print(f"the eager calls' C++ host side is not built, they will run through Python: {e}", file=sys.stderr)
        out_tmp = LIB_DIR / (LIB_PATH.name + ".tmp")
        cmd = [hipcc(), f"--offload-arch={OFFLOAD_ARCH}", "-shared", "-fPIC", "-o", str(out_tmp), *map(str, objs)]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"link failed:\n{proc.stderr}")
        os.replace(out_tmp, LIB_PATH)
    if verbose:
        print(f"built {LIB_PATH}")
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
