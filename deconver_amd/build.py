"""In-tree build of the HIP library (and, on request, of the host checker).

    python -m deconver_amd.build            # libdeconver_ndc.so for gfx950, _native.so (autograd nodes)
    python -m deconver_amd.build --hostcheck  # + libndc_hostcheck.so (CPU test-suite)
"""

from __future__ import annotations

import argparse
import concurrent.futures
import os
import subprocess
import sys
import tempfile

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, "csrc")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-ffp-contract=fast",
    # packed-fp32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # LLVM's VectorCombine widens scalar loads of the per-thread state into overlapping
    # two-element loads, which pins that state in private memory instead of registers
    "-mllvm", "-disable-vector-combine",
]


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines()
                    if "packed-fp32-ops" not in l and "is not a recognized feature" not in l)
    if proc.returncode != 0:
        sys.stderr.write(out + "\n")
        raise RuntimeError("build failed: " + " ".join(cmd))
    return out


HIP_SOURCES = ("ndc_capi.hip", "ndc_fused_bf16.hip", "ndc_fused_f32.hip", "ndc_gemm.hip", "ndc_mlp.hip")


def build_hip(extra_flags=(), out: str = os.path.join(_HERE, "libdeconver_ndc.so"), csrc: str = CSRC) -> str:
    """The HIP library: its translation units side by side, then one link."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    with tempfile.TemporaryDirectory() as tmp, concurrent.futures.ThreadPoolExecutor() as pool:
        objects = [os.path.join(tmp, name + ".o") for name in HIP_SOURCES]
        list(pool.map(lambda so: _run([hipcc, *HIPCC_FLAGS, *extra_flags, "-c", os.path.join(csrc, so[0]), "-o", so[1]]),
                      zip(HIP_SOURCES, objects)))
        _run([hipcc, "--offload-arch=gfx950", "-fPIC", "-shared", "-o", out, *objects])
    return out


def build_native() -> str:
    """The autograd nodes (``csrc/ndc_torch.cpp``): host code against PyTorch and the HIP library,
    which it finds next to itself."""
    import sysconfig

    import torch

    out = os.path.join(_HERE, "_native.so")
    base = os.path.dirname(torch.__file__)
    include = [os.path.join(base, "include"), os.path.join(base, "include", "torch", "csrc", "api", "include"),
               os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    libs = ["c10", "c10_hip", "torch_cpu", "torch_hip", "torch", "torch_python"]
    _run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-w", "-DTORCH_EXTENSION_NAME=_native",
          "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
          *["-isystem" + d for d in include], os.path.join(CSRC, "ndc_torch.cpp"), "-o", out,
          "-L" + _HERE, "-ldeconver_ndc", "-L" + os.path.join(base, "lib"), *["-l" + n for n in libs],
          "-Wl,-rpath,$ORIGIN"])
    return out


def build_hostcheck(sanitize: bool = False) -> str:
    out = os.path.join(_HERE, "libndc_hostcheck.so")
    flags = ["-O1", "-g", "-fsanitize=address,undefined"] if sanitize else ["-O2"]
    _run(["g++", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-unknown-pragmas", *flags, "-o", out,
          os.path.join(CSRC, "ndc_hostcheck.cpp")])
    return out


def main(argv=None) -> None:
    ap = argparse.ArgumentParser()
    ap.add_argument("--hostcheck", action="store_true")
    ap.add_argument("--no-hip", action="store_true")
    args = ap.parse_args(argv)
    if not args.no_hip:
        print(build_hip())
        print(build_native())
    if args.hostcheck:
        print(build_hostcheck())


if __name__ == "__main__":
    main()
