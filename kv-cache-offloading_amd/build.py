"""Builds libkvx.so (HIP kernels + C ABI) for gfx950 and the CPython binding into the kvx package directory.

Run: python kv-cache-offloading_amd/build.py [--arch gfx950] [--verbose]
"""

import argparse
import os
import shutil
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent
SOURCES = [HERE / "csrc" / "kvx_kernels.hip", HERE / "csrc" / "kvx_capi.hip"]
OUTPUT = HERE / "kvx" / "libkvx.so"
BIND_SOURCE = HERE / "csrc" / "kvx_bind.cpp"
BIND_OUTPUT = HERE / "kvx" / "_bind.so"

# fp-contract=off keeps every multiply and add separately rounded, as the
# FP8 codec's bit-exact contract assumes; packed FP32 instructions are
# disabled (they have produced wrong results on this hardware).
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "-shared",
    "-ffp-contract=off", "-fno-fast-math",
    "-mcode-object-version=5",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found; libkvx needs ROCm's compiler")
    return path


def build(arch: str = "gfx950", verbose: bool = False) -> Path:
    """Compiles both, then puts both in place: a failed step leaves the pair that was there."""
    _run([hipcc(), f"--offload-arch={arch}", *FLAGS, f"-I{ROOT / 'include'}", f"-I{HERE / 'csrc'}",
          *map(str, SOURCES), "-o", _tmp(OUTPUT)], verbose)
    _run(_bind_command(), verbose)
    for output in (OUTPUT, BIND_OUTPUT):
        os.replace(_tmp(output), output)
    return OUTPUT


def _bind_command() -> list[str]:
    """kvx/_bind.so: host code only, against the installed torch's headers; it calls libkvx by address."""
    import sysconfig

    import torch

    torch_dir = Path(torch.__file__).parent
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
            "-DUSE_ROCM", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            f'-DKVX_TORCH_VERSION="{torch.__version__}"', f"-I{ROOT / 'include'}",
            f"-isystem{torch_dir / 'include'}", "-isystem/opt/rocm/include",
            f"-I{sysconfig.get_paths()['include']}", str(BIND_SOURCE), "-o", _tmp(BIND_OUTPUT),
            f"-L{torch_dir / 'lib'}", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]


def _tmp(output: Path) -> str:
    return str(output) + ".tmp"


def _run(cmd: list[str], verbose: bool):
    if verbose:
        print(" ".join(cmd), flush=True)
    result = subprocess.run(cmd, capture_output=True, text=True, env=dict(os.environ))
    if result.returncode != 0:
        sys.stderr.write(result.stdout + result.stderr)
        raise RuntimeError(f"{cmd[0]} failed with exit code {result.returncode}")
    if verbose and result.stderr.strip():
        sys.stderr.write(result.stderr)


def main():
    parser = argparse.ArgumentParser(description=__doc__)
    parser.add_argument("--arch", default="gfx950")
    parser.add_argument("--verbose", action="store_true")
    args = parser.parse_args()
    print(build(args.arch, args.verbose))


if __name__ == "__main__":
    main()
