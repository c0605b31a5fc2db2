"""Build libiris_hip.so for gfx950 with hipcc, and the Python module that calls it with g++.

    python -m iris_amd.csrc.build [--force]

The library lands in iris_amd/lib/ next to the package so that it travels with the source tree.
"""

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
# One translation unit per input type of the MFMA kernel, of the kernel for small outputs and of the any-shape kernel (they
# hold most of the compile time and are compiled side by side), the entry points, and the stand-alone collectives.
SOURCES = [os.path.join(HERE, f) for f in (
    "iris_hip_mfma_bf16.hip", "iris_hip_mfma_f16.hip", "iris_hip_mfma_fp8.hip", "iris_hip_any_bf16.hip",
    "iris_hip_any_f16.hip", "iris_hip_any_fp8.hip", "iris_hip_any_f32.hip", "iris_hip_decode_bf16.hip",
    "iris_hip_decode_f16.hip", "iris_hip_decode_fp8.hip", "iris_hip_rows_bf16.hip", "iris_hip_rows_f16.hip", "iris_hip_rows_fp8.hip",
    "iris_hip.hip", "iris_ccl.hip")]
HEADERS = [os.path.join(HERE, h) for h in ("fused_kernel.h", "decode_kernel.h", "any_kernel.h", "any_epilogue.h", "fused_params.h", "pack_kernel.h", "layout.h", "device_util.h",
                                           "host_common.h")] + [
    os.path.join(ROOT, "include", "iris_hip.h")]
OUTPUT = os.path.join(os.path.dirname(HERE), "lib", "libiris_hip.so")
# The Python module through which the operators call the library's entry points (host code only; it reads torch's
# tensors without going through their Python attributes).
LAUNCHER_SOURCE = os.path.join(HERE, "launcher.cpp")
LAUNCHER_OUTPUT = os.path.join(os.path.dirname(HERE), "lib", "_launch.so")

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # Keep hipcc from forming packed fp32 instructions out of scalar float code.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unknown-warning-option",
    "-I" + os.path.join(ROOT, "include"),
    "-I" + HERE,
]


def launcher_tag():
    """What _launch.so is tied to, as the text that its build puts into it: it reads the tensors of one torch for one
    Python, and another one's differ without a symbol missing."""
    import torch

    return f"iris_amd launcher for torch {torch.__version__}, {sysconfig.get_config_var('SOABI')};"


def launcher_fits(path):
    """True when the module at `path` was built for the torch and the Python that run."""
    with open(path, "rb") as f:
        return launcher_tag().encode() in f.read()


def up_to_date():
    if not (os.path.exists(OUTPUT) and os.path.exists(LAUNCHER_OUTPUT) and launcher_fits(LAUNCHER_OUTPUT)):
        return False
    built = min(os.path.getmtime(OUTPUT), os.path.getmtime(LAUNCHER_OUTPUT))
    return all(os.path.getmtime(f) <= built for f in SOURCES + HEADERS + [LAUNCHER_SOURCE, os.path.abspath(__file__)])


def _build_launcher(verbose):
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    tmp = LAUNCHER_OUTPUT + ".tmp"
    includes = [sysconfig.get_paths()["include"]] + include_paths() + [os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")]
    _run([shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", f'-DIRIS_LAUNCHER_TAG="{launcher_tag()}"', "-I" + os.path.join(ROOT, "include")]
         + [flag for path in includes for flag in ("-isystem", path)] + ["-o", tmp, LAUNCHER_SOURCE]
         + ["-L" + path for path in library_paths()] + ["-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", "-ldl"], verbose)
    os.replace(tmp, LAUNCHER_OUTPUT)


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # hipcc's host pass does not know the packed-fp32 feature and says so; that line is noise.
    noise = "is not a recognized feature for this target"
    out = "\n".join(l for l in proc.stdout.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
    if verbose and out.strip():
        print(out)


STAMPS_OUTPUT = os.path.join(os.path.dirname(HERE), "lib", "libiris_hip_stamps.so")


def build(force=True, verbose=True, stamps=False):
    """Compile the library.  With force=False an up-to-date library is left alone.  stamps=True builds
    the diagnostic variant (kernels record time stamps at their phase boundaries; see
    iris_amd/bench/phase_stamps.py) as libiris_hip_stamps.so next to the regular library."""
    if stamps:
        return _build(STAMPS_OUTPUT, FLAGS + ["-DIRIS_HIP_PHASE_STAMPS"], verbose)
    if not force and up_to_date():
        return OUTPUT
    return _build(OUTPUT, FLAGS, verbose)


def _build(output, flags, verbose):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    os.makedirs(os.path.dirname(output), exist_ok=True)
    with tempfile.TemporaryDirectory(prefix="iris_hip_build_") as tmpdir:
        objects = [os.path.join(tmpdir, os.path.splitext(os.path.basename(src))[0] + ".o") for src in SOURCES]
        with concurrent.futures.ThreadPoolExecutor(max_workers=min(len(SOURCES), os.cpu_count() or 1)) as pool:
            jobs = [pool.submit(_build_launcher, verbose)]
            jobs += [pool.submit(_run, [hipcc] + flags + ["-c", "-o", obj, src], verbose)
                     for src, obj in zip(SOURCES, objects)]
            for job in jobs:
                job.result()
        tmp = output + ".tmp"
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-o", tmp] + objects, verbose)
        os.replace(tmp, output)
    return output


if __name__ == "__main__":
    print(build(force=True, stamps="--stamps" in sys.argv))
