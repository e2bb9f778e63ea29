"""Build recipe for the in-tree HIP library ``libw4g64_hip.so`` (gfx950 only)
and the CPython module ``_host.so`` that calls it.

Compiles every ``csrc/*.hip`` translation unit with hipcc (in parallel) and
links them into ``qwen_int4_hip/libw4g64_hip.so``; ``csrc/host_linear.cpp``
(host code only) is compiled against torch's headers.  Always rebuilds: the
caller (``__graft_entry__.build``) wants a fresh compile every time.

``build(timeline=True)`` compiles the same sources with ``-DW4G64_TIMELINE``
into ``libw4g64_hip_timeline.so``: a profiling build whose instrumented
kernels record per-workgroup phase timestamps (``bench.py --timeline``).  The
product never loads it.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PACKAGE_DIR = Path(__file__).resolve().parent
SOURCE_ROOT = PACKAGE_DIR.parent
CSRC = SOURCE_ROOT / "csrc"
REPO_ROOT = SOURCE_ROOT.parent
LIBRARY = PACKAGE_DIR / "libw4g64_hip.so"
TIMELINE_LIBRARY = PACKAGE_DIR / "libw4g64_hip_timeline.so"
HOST_MODULE = PACKAGE_DIR / "_host.so"
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # Keep fp32 math unpacked (no v_pk_*_f32 generated by the compiler).
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{REPO_ROOT / 'include'}",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found; the W4G64 HIP library needs ROCm's hipcc")
    return path


# Per-source flags.  The pipelined GEMV keeps its MFMA results in VGPRs: its
# scaling FMAs read them straight away, and AGPR results cost a copy each.
SOURCE_FLAGS = {
    "w4g64_gemv_pipe.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
}


def _compile(source: Path, obj: Path, extra: tuple = ()) -> None:
    cmd = [hipcc(), *HIPCC_FLAGS, *SOURCE_FLAGS.get(source.name, []), *extra, "-c", str(source), "-o", str(obj)]
    result = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    stderr = "\n".join(line for line in result.stderr.splitlines() if noise not in line)
    if result.returncode != 0:
        raise RuntimeError(f"hipcc failed for {source.name}:\n{stderr}")
    if stderr.strip():
        print(stderr, file=sys.stderr)


def build_host() -> Path:
    """Compile ``_host.so`` (the library has to be built: it is linked)."""
    import sysconfig

    import torch

    root = Path(torch.__file__).resolve().parent
    tmp = HOST_MODULE.with_suffix(".so.tmp")
    compiler = shutil.which("g++") or str(Path(hipcc()).resolve().parent / "amdclang++")
    cmd = [compiler, "-std=c++17", "-O2", "-fPIC", "-shared", "-w",
           "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{sysconfig.get_paths()['include']}", f"-I{root / 'include'}",
           f"-I{root / 'include/torch/csrc/api/include'}", f"-I{Path(hipcc()).resolve().parents[1] / 'include'}",
           str(CSRC / "host_linear.cpp"), "-o", str(tmp), f"-L{root / 'lib'}",
           "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip",
           f"-L{PACKAGE_DIR}", f"-l:{LIBRARY.name}", "-Wl,-rpath,$ORIGIN"]
    result = subprocess.run(cmd, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for host_linear.cpp:\n{result.stderr}")
    os.replace(tmp, HOST_MODULE)
    return HOST_MODULE


def build(verbose: bool = True, timeline: bool = False) -> Path:
    """Compile and link the library (or its timeline build); returns its path."""
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    obj_dir = SOURCE_ROOT / ("_build_timeline" if timeline else "_build")
    obj_dir.mkdir(exist_ok=True)
    objects = [obj_dir / (src.stem + ".o") for src in sources]
    extra = ("-DW4G64_TIMELINE",) if timeline else ()
    workers = min(len(sources), int(os.environ.get("MAX_JOBS", "8")) or 1)
    with ThreadPoolExecutor(max_workers=workers) as pool:
        list(pool.map(lambda pair: _compile(*pair, extra), zip(sources, objects)))
    target = TIMELINE_LIBRARY if timeline else LIBRARY
    tmp = target.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objects)]
    result = subprocess.run(cmd, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"link failed:\n{result.stderr}")
    os.replace(tmp, target)
    if not timeline:
        build_host()
    if verbose:
        print(f"built {target} from {len(sources)} sources", file=sys.stderr)
    return target


if __name__ == "__main__":
    build(timeline="--timeline" in sys.argv)
