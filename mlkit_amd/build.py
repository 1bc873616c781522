"""Builds ``libmlkit_amd.so`` for gfx950 with hipcc (cross-compiles without a GPU), and the layers' native call from Python.

``python -m mlkit_amd.build`` compiles every translation unit under ``csrc/`` in
parallel and links the shared library beside this file.  Nothing here runs at import
time: loading a prebuilt library is ``mlkit_amd.native``'s job.
"""

import concurrent.futures
import os
import pathlib
import subprocess
import sys
import sysconfig
import time

ROOT = pathlib.Path(__file__).resolve().parent
CSRC = ROOT / "csrc"
OBJECTS = CSRC / "_build"
LIBRARY = ROOT / "libmlkit_amd.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

COMMON_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    # hipcc may not form packed fp32 arithmetic on its own (flag for the device pass;
    # the host pass prints a harmless "not a recognized feature" warning).
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# Kernels whose results are compared bit for bit keep multiply and add separate.
EXACT_FLAGS = ["-ffp-contract=off"]

HOST_EXTENSION = ROOT / "_packed_call.so"   # the layers' native call: host code against torch's headers

MATVEC_WIDTHS = range(2, 9)
MATMUL_FORMATS = range(5)


def translation_units() -> list[tuple[str, pathlib.Path, list[str]]]:
    units: list[tuple[str, pathlib.Path, list[str]]] = []
    for width in MATVEC_WIDTHS:
        units.append((f"packed_matvec_b{width}", CSRC / "packed_matvec_bits.hip",
                      [f"-DMK_MATVEC_BITS={width}"]))
    for code_format in MATMUL_FORMATS:
        units.append((f"packed_matmul_f{code_format}", CSRC / "packed_matmul_kernels.hip",
                      [f"-DMK_MATMUL_FORMAT={code_format}"]))
    exact = {"packed_decode", "scalar_codec", "scalar_round", "error_feedback", "hadamard", "vector_feedback", "column_transforms"}
    for source in sorted(CSRC.glob("*.hip")):
        if source.name in ("packed_matvec_bits.hip", "packed_matmul_kernels.hip"):
            continue
        units.append((source.stem, source, EXACT_FLAGS if source.stem in exact else []))
    return units


def _compile(unit: tuple[str, pathlib.Path, list[str]]) -> tuple[str, float, str]:
    name, source, extra = unit
    target = OBJECTS / f"{name}.o"
    started = time.time()
    command = [HIPCC, *COMMON_FLAGS, *extra, "-c", str(source), "-o", str(target)]
    result = subprocess.run(command, capture_output=True, text=True)
    log = "\n".join(line for line in (result.stdout + result.stderr).splitlines()
                    if "packed-fp32-ops' is not a recognized feature" not in line)
    if result.returncode != 0:
        raise RuntimeError(f"hipcc failed for {source.name}:\n{log}")
    return name, time.time() - started, log


def _compile_host_extension() -> tuple[str, float, str]:
    import torch
    from torch.utils import cpp_extension

    started = time.time()
    libraries = pathlib.Path(torch.__file__).parent / "lib"
    includes = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include"]
    command = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
               f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{path}" for path in includes),
               str(CSRC / "packed_call.cpp"), "-o", str(HOST_EXTENSION), f"-L{libraries}",
               "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    result = subprocess.run(command, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"{command[0]} failed for packed_call.cpp:\n{result.stdout}{result.stderr}")
    return "packed_call", time.time() - started, result.stdout + result.stderr


def build(verbose: bool = True, jobs: int | None = None, only: list[str] | None = None) -> pathlib.Path:
    """Compile all units (or, while developing, just the units named in ``only``, reusing the
    other objects of an earlier full build) and link the library; returns its path."""
    OBJECTS.mkdir(exist_ok=True)
    units = translation_units()
    chosen = [unit for unit in units if not only or unit[0] in only]
    jobs = jobs or min(len(units), os.cpu_count() or 4, 16)
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_compile_host_extension) if not only or "packed_call" in only else None
        for name, seconds, log in pool.map(_compile, chosen):
            if verbose:
                print(f"[mlkit_amd.build] {name}.o  {seconds:6.1f}s", flush=True)
                if log.strip():
                    print(log)
        if host is not None:
            name, seconds, log = host.result()
            if verbose:
                print(f"[mlkit_amd.build] {name}  {seconds:6.1f}s", flush=True)
                if log.strip():
                    print(log)
    objects = [str(OBJECTS / f"{name}.o") for name, _, _ in units]
    link = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", "-o", str(LIBRARY), *objects]
    result = subprocess.run(link, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"link failed:\n{result.stdout}{result.stderr}")
    if verbose:
        print(f"[mlkit_amd.build] linked {LIBRARY}", flush=True)
    return LIBRARY


if __name__ == "__main__":
    build(verbose=True, only=sys.argv[1:] or None)   # e.g. `python -m mlkit_amd.build hadamard`
    sys.exit(0)
