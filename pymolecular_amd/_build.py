"""Build recipe for the HIP library ``libpymolecular_egnn.so`` (gfx950).

Each ``csrc/*.hip`` file is compiled with ``hipcc --offload-arch=gfx950`` in
parallel and linked into one shared library next to this file, so that it
travels with the source tree.  ``python -m pymolecular_amd._build`` runs it.

Next to the library the build writes ``libpymolecular_egnn.so.srchash``: a
SHA-256 over the sources it was built from (``csrc/``, ``include/egnn.h``)
and the compiler flags.  ``_capi.lib()`` recomputes it and refuses a library
built from other sources, so a run always exercises the current tree.

The layer's native autograd node ``_egnn_torch.so`` (``csrc/egnn_torch.cpp``,
host code against torch's headers) has a stamp of its own, which also holds
the versions of torch, its C++ ABI and Python: ``_capi.ext()`` refuses a
module built against others.
"""
from __future__ import annotations

import concurrent.futures as cf
import hashlib
import os
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
HEADER = PKG.parent / "include" / "egnn.h"
LIB = PKG / "libpymolecular_egnn.so"
STAMP = LIB.with_name(LIB.name + ".srchash")
EXT = PKG / "_egnn_torch.so"   # the layer's native autograd node, linked to LIB
EXT_SRC = CSRC / "egnn_torch.cpp"
EXT_STAMP = EXT.with_name(EXT.name + ".srchash")
OBJ = PKG / "_objs"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed fp32 VALU forms are kept out of all device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


# per-file flags: the edge-parallel kernels keep their MFMA accumulators in VGPRs (the VALU reads
# every product's result; the AGPR form would copy each one back)
FILE_FLAGS = {
    "egnn_mpnn.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "egnn_eqfwd.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "egnn_wfwd.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "egnn_wbwd.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "egnn_f32.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "egnn_f32s.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
}


def source_files() -> list:
    return sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")) + [HEADER]


EXT_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
             "-DTORCH_API_INCLUDE_EXTENSION_H"]
EXT_LIBS = ["-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]


def _ext_commands(out: Path):
    """(compile, link) of the autograd node, linked to ``out``: host code against torch's headers, no device code."""
    import sysconfig

    import torch
    root = Path(torch.__file__).resolve().parent
    obj = OBJ / "egnn_torch.o"
    inc = [root / "include", root / "include/torch/csrc/api/include", sysconfig.get_paths()["include"],
           os.environ.get("ROCM_PATH", "/opt/rocm") + "/include"]
    cc = ["g++", *EXT_FLAGS, f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
          *(x for p in inc for x in ("-isystem", str(p))), "-c", str(EXT_SRC), "-o", str(obj)]
    ld = ["g++", "-shared", "-o", str(out), str(obj), f"-L{PKG}", "-l:" + LIB.name, f"-L{root / 'lib'}", *EXT_LIBS]
    return cc, ld


def ext_hash() -> str:
    """SHA-256 over what the autograd node is made of: its source, the C-ABI's header, the flags, and the versions
    of torch, its C++ ABI and Python it is compiled against."""
    import sysconfig

    import torch
    h = hashlib.sha256()
    for part in (*EXT_FLAGS, *EXT_LIBS, torch.__version__, str(torch.compiled_with_cxx11_abi()),
                 sysconfig.get_config_var("SOABI") or sys.version):
        h.update(part.encode() + b"\0")
    for p in (EXT_SRC, HEADER):
        h.update(b"\0" + p.name.encode() + b"\0")
        h.update(p.read_bytes())
    return h.hexdigest()


def _run(cmd, what) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n" + r.stderr[-6000:])
    if r.stderr.strip():
        print(r.stderr.strip(), file=sys.stderr)


def source_hash() -> str:
    """SHA-256 over the flags and the (relative name, content) of every source file."""
    h = hashlib.sha256()
    h.update("\0".join(FLAGS).encode())
    for name in sorted(FILE_FLAGS):
        h.update(("\0" + name + "\0" + "\0".join(FILE_FLAGS[name])).encode())
    for p in source_files():
        h.update(b"\0" + p.name.encode() + b"\0")
        h.update(p.read_bytes())
    return h.hexdigest()


def _compile(src: Path) -> Path:
    obj = OBJ / (src.stem + ".o")
    cmd = [HIPCC, *FLAGS, *FILE_FLAGS.get(src.name, []), "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        msg = "\n".join(l for l in r.stderr.splitlines() if "not a recognized feature" not in l)
        raise RuntimeError(f"hipcc failed for {src.name}:\n{msg}")
    return obj


def build(verbose: bool = True) -> Path:
    OBJ.mkdir(exist_ok=True)
    digest, ext_digest = source_hash(), ext_hash()
    srcs = sorted(CSRC.glob("*.hip"))
    jobs = min(len(srcs), max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        ext_tmp = EXT.with_suffix(".so.tmp")
        ext_cc, ext_ld = _ext_commands(ext_tmp)
        ext = ex.submit(_run, ext_cc, "compiling egnn_torch.cpp")   # the longest single file
        objs = list(ex.map(_compile, srcs))
        ext.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    for stamp in (STAMP, EXT_STAMP):
        stamp.unlink(missing_ok=True)
    os.replace(tmp, LIB)
    STAMP.write_text(digest + "\n")
    _run(ext_ld, "linking " + EXT.name)
    os.replace(ext_tmp, EXT)
    EXT_STAMP.write_text(ext_digest + "\n")
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources (sources sha256 {digest[:16]})")
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
