"""Compiles tests/host/*.hip for the host alone: the index rules that kernels and host code share, run on the CPU."""
import os
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def build(name: str, out_dir: Path) -> Path:
    exe = Path(out_dir) / name
    cmd = [HIPCC, "--cuda-host-only", "-O1", "-std=c++17", "-Wall", "-Wno-unused-function",
           "-I", str(ROOT / "tasktorrent_amd" / "csrc"), str(ROOT / "tests" / "host" / f"{name}.hip"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"host build of {name} failed:\n{r.stderr}")
    return exe


def run(exe: Path, *args) -> str:
    r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
