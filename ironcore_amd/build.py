"""Build recipe for the HIP library: hipcc, gfx950 only, in-tree output.

    python -m ironcore_amd.build

compiles every translation unit under ironcore_amd/csrc/ and links
ironcore_amd/lib/libironcore_paged.so, then the torch-side call path
ironcore_amd/lib/_host.so.  Cross-compiles without a GPU.
"""
from __future__ import annotations

import concurrent.futures
import os
import re
import shutil
import subprocess
import sys
import tempfile
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIB_DIR = PKG / "lib"
LIB_PATH = LIB_DIR / "libironcore_paged.so"
HOST_PATH = LIB_DIR / "_host.so"   # native call path (csrc/host_binding.cpp), links LIB_PATH
OBJ_DIR = PKG / "build" / "obj"

SOURCES = ["ic_api.hip", "kv_append.hip", "rope_kv_append.hip", "paged_decode.hip", "paged_decode_mfma.hip", "paged_prefill.hip",
           "paged_prefill_short.hip", "paged_prefill_f32.hip", "mask_pack.hip", "linear_rows.hip", "step_linear.hip", "step_stack.hip", "choose_token.hip", "mfma_probe.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Wall",
    "-Wno-unused-function",
    # the staging loads set m0 by hand and say so in their clobber lists
    "-Wno-inline-asm",
    # hipcc -O3 must not form packed-fp32 VALU ops on its own.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def csrc_digest() -> str:
    """SHA-256 over the names and contents of the kernel sources (csrc/*.hip,
    *.h): identifies the code a profiler figure was measured on."""
    import hashlib
    h = hashlib.sha256()
    for path in sorted(CSRC.glob("*")):
        if path.suffix in (".hip", ".h"):
            h.update(path.name.encode())
            h.update(b"\0")
            h.update(path.read_bytes())
            h.update(b"\0")
    return h.hexdigest()


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the HIP library cannot be built")
    return exe


# Per-file flags.  The prefill kernel keeps its MFMA accumulators in ordinary
# VGPRs: the softmax rescales them with VALU instructions, and the AGPR form
# costs a register copy each way per tile.
_VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]
PER_SOURCE_FLAGS = {"paged_prefill.hip": _VGPR_FORM, "paged_prefill_short.hip": _VGPR_FORM,
                    "paged_prefill_f32.hip": _VGPR_FORM, "paged_decode_mfma.hip": _VGPR_FORM}


# Sources whose kernels keep registers in scratch: their assembly is looked at, see masked_spills.
_SPILLING = {"step_stack.hip"}


def masked_spills(asm: str) -> list[str]:
    """Labels of blocks that move registers to or from scratch and only then switch on the lanes that a branch had
    switched off.  The compiler does that where a whole value is meant (it takes the block's start for the place behind
    ``s_or_b64 exec``): the other lanes' part is then lost, and a kernel that counts on it ends wrong or never."""
    found, kernel, label, moved = [], "", "", False
    for line in asm.splitlines():
        name = re.match(r"(\w+):|; (%bb\.\d+):|(\.LBB\w+):", line)
        if name:
            kernel, label, moved = name[1] or kernel, name[2] or name[3] or "entry", False
        elif re.match(r"\ts_\w+ exec, exec|\ts_mov_b64 exec|\ts_\w+_saveexec", line):
            if moved and line.startswith("\ts_or_b64 exec, exec"):
                found.append(f"{kernel} {label}")
            moved = False
        elif "Folded" in line and "scratch_" in line:
            moved = True
    return found


def _compile(src: str, extra: list[str]) -> Path:
    obj = OBJ_DIR / (src + ".o")
    with tempfile.TemporaryDirectory(dir=OBJ_DIR) as temps:
        out = Path(temps) / obj.name
        cmd = [_hipcc(), *HIPCC_FLAGS, *PER_SOURCE_FLAGS.get(src, []), *extra, "-c", str(CSRC / src), "-o", str(out)]
        if src in _SPILLING:
            cmd.append("-save-temps=obj")
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{res.stdout}\n{res.stderr}")
        if src in _SPILLING:
            (asm,) = Path(temps).glob("*-gfx950.s")
            if found := masked_spills(asm.read_text()):
                raise RuntimeError(f"{src}: registers go to scratch before all lanes are on again, in {found}")
        os.replace(out, obj)
    noise = "is not a recognized feature for this target"
    warn = "\n".join(line for line in res.stderr.splitlines() if noise not in line)
    if warn.strip():
        sys.stderr.write(warn + "\n")
    return obj


def _compile_host() -> Path:
    """The torch-side call path: host code only, torch's headers, the system compiler."""
    import sysconfig
    from torch.utils import cpp_extension
    obj = OBJ_DIR / "host_binding.cpp.o"
    includes = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-DTORCH_EXTENSION_NAME=_host",
           "-DTORCH_API_INCLUDE_EXTENSION_H", *(f"-I{p}" for p in includes), "-c", str(CSRC / "host_binding.cpp"),
           "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on host_binding.cpp:\n{res.stdout}\n{res.stderr}")
    return obj


def _link_host(obj: Path) -> None:
    from torch.utils import cpp_extension
    tmp = HOST_PATH.with_suffix(".so.tmp")
    cmd = ["g++", "-shared", str(obj), "-o", str(tmp), f"-L{LIB_DIR}", f"-l:{LIB_PATH.name}", "-Wl,-rpath,$ORIGIN",
           *(f"-L{p}" for p in cpp_extension.library_paths()), "-lc10", "-ltorch_cpu", "-ltorch", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, HOST_PATH)


def build(verbose: bool = True, extra_flags: list[str] | None = None) -> Path:
    """Compile and link; returns the path of the shared library."""
    extra = list(extra_flags or [])
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    LIB_DIR.mkdir(parents=True, exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(SOURCES) + 1)) as pool:
        host = pool.submit(_compile_host)
        objs = list(pool.map(lambda s: _compile(s, extra), SOURCES))
        host_obj = host.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc",
           *map(str, objs), "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    _link_host(host_obj)
    if verbose:
        print(f"built {LIB_PATH} ({LIB_PATH.stat().st_size} bytes)")
    return LIB_PATH


if __name__ == "__main__":
    build()
