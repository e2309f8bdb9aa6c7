"""Build libpippin_hip.so in-tree with hipcc for gfx950.

Every source is compiled with -ffp-contract=off so the device arithmetic keeps
the reference's unfused multiply/add order, and with packed-FP32 instructions
disabled. Device code is scheduled with LLVM's iterative ILP strategy: the step
kernels run one wavefront per SIMD, so their latency is hidden only by
independent instructions within the wavefront (the Ant step kernel measured
about 7 % faster than with the default scheduler; scheduling moves no rounding).
"""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
OUT = HERE / "libpippin_hip.so"
# the step kernels' instances, one object each (step_kernels.hpp)
INSTANCES = {"k1": (1, "DModel"), "k2": (2, "DModel"), "k4": (4, "DModel"), "ant": (4, "SpecAnt")}
# (source, object name, extra flags), the slowest to compile first
UNITS = [
    (src, f"{src[:-4]}_{tag}.o", [f"-DPH_K={k}", f"-DPH_MT={mt}", f"-DPH_TAG={tag}"])
    for src in ("step_inst.hip", "step_mlp_inst.hip", "pgs_inst.hip") for tag, (k, mt) in INSTANCES.items()
    if src != "pgs_inst.hip" or mt == "DModel"
] + [(src, src + ".o", []) for src in
     ("runtime.hip", "mlp.hip", "host_model.cpp", "mjcf.cpp", "meshes.cpp", "urdf.cpp")]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("PIPPIN_HIP_ARCH", "gfx950")
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"--offload-arch={ARCH}",
    "-mllvm", "-amdgpu-sched-strategy=iterative-ilp",
]


# Models whose kernels are also built with compile-time sizes and LDS layout
# (struct name, MJCF file); any other model runs the generic kernel.
SPECIALISED = [("SpecAnt", HERE / "assets" / "ant.xml")]


def generate_specs(bdir: Path, verbose: bool = False) -> None:
    """Build the host-only generator and write _build/spec_models.hpp."""
    gen = bdir / "spec_gen"
    srcs = [CSRC / "spec_gen.cpp", CSRC / "host_model.cpp", CSRC / "mjcf.cpp", CSRC / "meshes.cpp"]
    cmd = [HIPCC, "-O1", "-std=c++17", "-x", "hip", f"--offload-arch={ARCH}", *map(str, srcs), "-o", str(gen)]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True, stderr=subprocess.DEVNULL if not verbose else None)
    args = [str(gen)]
    for name, path in SPECIALISED:
        args += [name, str(path)]
    out = subprocess.run(args, check=True, capture_output=True, text=True).stdout
    (bdir / "spec_models.hpp").write_text(out)


def build(verbose: bool = False) -> Path:
    from concurrent.futures import ThreadPoolExecutor

    bdir = HERE / "_build"
    bdir.mkdir(exist_ok=True)
    generate_specs(bdir, verbose)

    def compile_unit(unit) -> str:
        src, name, extra = unit
        lang = ["-x", "hip"] if src.endswith(".cpp") else []
        cmd = [HIPCC, *FLAGS, *extra, *lang, "-I", str(bdir), "-c", str(CSRC / src), "-o", str(bdir / name)]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)
        return str(bdir / name)

    with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:  # side by side
        objs = list(pool.map(compile_unit, UNITS))
    tmp = OUT.with_suffix(".so.tmp")
    cmd = [HIPCC, *FLAGS, "-shared", "-o", str(tmp), *objs]
    subprocess.run(cmd, check=True)
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
