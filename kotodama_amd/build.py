"""Build libattnres_hip.so in-tree: gfx950 code objects + the C-ABI host library.

Steps (all outputs under ``kotodama_amd/lib/``):

1. ``hipcc --genco --offload-arch=gfx950`` compiles ``csrc/attnres_kernels.hip``
   once per code-object part (``-DATTNRES_PART=0..11``, in parallel).
2. ``gcc`` assembles ``csrc/attnres_blob.S``, which ``.incbin``s the parts.
3. ``hipcc -c -fPIC`` compiles ``csrc/attnres_noalloc.hip`` (the no-alloc
   entry point; its device array needs HIP device code of its own).
4. ``g++`` links ``csrc/attnres_capi.cpp``, the blob and that object into the
   shared library, linked against ROCm's ``libamdhip64.so.7``.  Loaded after ``import torch``,
   the dynamic linker binds that soname to the HIP runtime torch already
   loaded, so streams and device memory are shared with torch.
5. Where a ROCm torch is importable, ``g++`` compiles ``csrc/attnres_torch.cpp``
   against its headers into ``_attnres_torch`` (with this Python's extension
   suffix), the CPython extension through which the eager torch layer calls
   that library.  The library needs no torch and is in place before this step
   can fail; an extension of an earlier build does not stay beside it.

Run ``python -m kotodama_amd.build`` or call :func:`build`.
"""

from __future__ import annotations

import os
import subprocess
import sys
import tempfile
from importlib.machinery import EXTENSION_SUFFIXES
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIBDIR = PKG / "lib"
INCLUDE = PKG.parent / "include"
LIB_NAME = "libattnres_hip.so"
NATIVE_NAME = "_attnres_torch" + EXTENSION_SUFFIXES[0]  # as _native.py looks it up
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
ARCH = "gfx950"
NUM_PARTS = 12

# Packed-fp32 VALU ops are disabled for every HIP compile (the kernels are
# written with scalar fp32 arithmetic).
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "--genco",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
]


def _rocm_torch():
    """The torch module the extension can be built against, or None (no torch, or not a ROCm one)."""
    try:
        import torch
    except ImportError:
        return None
    return torch if torch.version.hip is not None else None


def _native_cmd(torch, out: Path) -> list[str]:
    """Compile the torch layer's extension to an object file (the link follows the C-ABI library's)."""
    import sysconfig

    from torch.utils.cpp_extension import include_paths

    incs = [f"-isystem{p}" for p in [*include_paths(), ROCM / "include", sysconfig.get_paths()["include"]]]
    return ["g++", "-c", "-fPIC", "-O2", "-std=c++17", "-Wall", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__",
            "-DUSE_ROCM", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
            f'-DATTNRES_TORCH_VERSION="{torch.__version__}"', f"-I{INCLUDE}", f"-I{CSRC}", *incs,
            str(CSRC / "attnres_torch.cpp"), "-o", str(out)]


def _run(cmd: list[str], cwd: Path | None = None) -> None:
    res = subprocess.run(cmd, cwd=cwd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"build step failed ({res.returncode}): {' '.join(cmd)}\n{res.stdout}\n{res.stderr}")


def _wait(cmd: list[str], proc: subprocess.Popen) -> None:
    so, se = proc.communicate()
    if proc.returncode != 0:
        raise RuntimeError(f"{Path(cmd[0]).name} failed ({proc.returncode}): {' '.join(cmd)}\n{so}\n{se}")


def build(verbose: bool = False, out_dir: Path | None = None, defines: tuple = ()) -> Path:
    """Compile everything; returns the path of the built shared library.

    ``out_dir`` (default ``kotodama_amd/lib``) and extra ``-D`` ``defines``
    (e.g. ``("ATTNRES_NT_LOADS=0",)``) allow side-by-side variant builds.
    """
    hipcc = str(ROCM / "bin" / "hipcc")
    libdir = Path(out_dir) if out_dir is not None else LIBDIR
    libdir.mkdir(parents=True, exist_ok=True)
    extra = [f"-D{d}" for d in defines]
    with tempfile.TemporaryDirectory(prefix="attnres_build_", dir=libdir) as tmp:
        tmpd = Path(tmp)
        procs = []
        native_o = tmpd / "attnres_torch.o"
        torch = _rocm_torch()
        if torch is not None:
            native = _native_cmd(torch, native_o)
            native_proc = subprocess.Popen(native, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
        for part in range(NUM_PARTS):
            out = tmpd / f"attnres_gfx950_part{part}.hsaco"
            cmd = [hipcc, *HIP_FLAGS, *extra, f"-DATTNRES_PART={part}", f"-I{CSRC}", str(CSRC / "attnres_kernels.hip"),
                   "-o", str(out)]
            if verbose:
                print(" ".join(cmd), flush=True)
            procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)))
        for cmd, p in procs:
            _wait(cmd, p)
        blob_o = tmpd / "attnres_blob.o"
        _run(["gcc", "-c", f"-I{tmpd}", str(CSRC / "attnres_blob.S"), "-o", str(blob_o)])
        noalloc_o = tmpd / "attnres_noalloc.o"
        noalloc_cmd = [hipcc, *[f for f in HIP_FLAGS if f != "--genco"], *extra, "-c", "-fPIC", f"-I{INCLUDE}",
                       str(CSRC / "attnres_noalloc.hip"), "-o", str(noalloc_o)]
        if verbose:
            print(" ".join(noalloc_cmd), flush=True)
        _run(noalloc_cmd)
        so_tmp = tmpd / LIB_NAME
        _run(
            [
                "g++",
                "-shared",
                "-fPIC",
                "-O2",
                "-std=c++17",
                "-Wall",
                "-D__HIP_PLATFORM_AMD__",
                *extra,
                f"-I{INCLUDE}",
                f"-I{CSRC}",
                f"-I{ROCM / 'include'}",
                str(CSRC / "attnres_capi.cpp"),
                str(blob_o),
                str(noalloc_o),
                f"-L{ROCM / 'lib'}",
                "-lamdhip64",
                f"-Wl,-rpath,{ROCM / 'lib'}",
                "-o",
                str(so_tmp),
            ]
        )
        final = libdir / LIB_NAME
        os.replace(so_tmp, final)  # atomic: a reader never sees a half-written library
        for old in libdir.glob("_attnres_torch*.so"):
            old.unlink()  # made for the library that was here before
        if torch is not None:
            _wait(native, native_proc)
            torch_lib = Path(torch.__file__).parent / "lib"
            native_tmp = tmpd / NATIVE_NAME
            _run(["g++", "-shared", str(native_o), f"-L{libdir}", "-lattnres_hip", f"-L{torch_lib}", "-ltorch_python",
                  "-ltorch_cpu", "-ltorch_hip", "-lc10_hip", "-lc10", "-Wl,-rpath,$ORIGIN",
                  f"-Wl,-rpath,{torch_lib}", "-o", str(native_tmp)])
            os.replace(native_tmp, libdir / NATIVE_NAME)
    if verbose:
        print(f"built {final}", flush=True)
    return final


if __name__ == "__main__":
    build(verbose="-q" not in sys.argv)
