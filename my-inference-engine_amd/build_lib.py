"""Build libmi_fa2.so and libmi_model.so (the HIP kernels + C ABIs) in-tree with hipcc for gfx950.

    python my-inference-engine_amd/build_lib.py

Compiles every source of csrc/ in parallel into _build/ and links kernels/libmi_fa2.so (attention,
sampling, step metadata; loaded by kernels/_lib.py) and kernels/libmi_model.so (the projections of
few rows; loaded by kernels/few_rows.py).  Always rebuilds (a few seconds per file).
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
OUT = PKG / "kernels" / "libmi_fa2.so"
LIBS = {
    OUT: ["fa2_prefill.hip", "fa2_decode.hip", "fa2_general.hip", "fa2_prefill_dims.hip", "fa2_merge.hip",
          "rope_kv.hip", "sample.hip", "step_meta.hip", "model_ops.hip", "fa2_capi.cpp"],
    PKG / "kernels" / "libmi_model.so": ["linear_rows.hip", "model_capi.cpp"],
}

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    # Packed fp32 VALU ops stay off: hipcc would otherwise emit v_pk_{add,mul,fma}_f32.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{ROOT / 'include'}",
    f"-I{CSRC}",
]


def _compile(src: str) -> Path:
    obj = BUILD / (Path(src).stem + ".o")
    cmd = [HIPCC, *FLAGS, "-c", str(CSRC / src), "-o", str(obj)]
    if src.endswith(".cpp"):
        cmd.insert(1, "-xhip")
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{' '.join(cmd)}\n{proc.stdout}{proc.stderr}")
    return obj


def build(verbose: bool = True) -> Path:
    BUILD.mkdir(exist_ok=True)
    sources = [src for srcs in LIBS.values() for src in srcs]
    with ThreadPoolExecutor(max_workers=len(sources)) as ex:
        objs = dict(zip(sources, ex.map(_compile, sources)))
    for out, srcs in LIBS.items():
        tmp = out.with_suffix(".so.tmp")
        cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *(str(objs[x]) for x in srcs),
               "-o", str(tmp)]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{proc.stdout}{proc.stderr}")
        os.replace(tmp, out)
        if verbose:
            print(f"built {out.relative_to(ROOT)}")
    return OUT


if __name__ == "__main__":
    try:
        build()
    except RuntimeError as e:
        print(e, file=sys.stderr)
        sys.exit(1)
