"""Builds libminicompiler_hip.so (and the mcc driver) in-tree.

Host C++ (the compiler core, the HIP backend's host side and the C ABI) is
compiled with g++ and sees no HIP header except in the thin layer
csrc/hip/hip_rt.cpp. The matmul kernels (csrc/hip/*.hip) are compiled
ahead of time for gfx950 with hipcc. Everything links into one shared
library against libamdhip64 and libhiprtc. Always rebuilds everything (the
"does it build" check must compile), in parallel.

    python -m minicompiler_amd.build            # library + mcc
    python -m minicompiler_amd.build --sanitize # host C++ with ASan + UBSan (below)

--sanitize builds a second copy of the library, for CPU-side checks of the
host code: the host objects compiled by g++ with AddressSanitizer and
UndefinedBehaviorSanitizer, linked (by g++) with the gfx950 kernel objects
of the normal build, into _build/sanitize/libminicompiler_hip.so. Run the
CPU tests against it with

    MINICOMPILER_HIP_LIBRARY=_build/sanitize/libminicompiler_hip.so \
    LD_PRELOAD="$(gcc -print-file-name=libasan.so) $(gcc -print-file-name=libubsan.so)" \
    ASAN_OPTIONS=detect_leaks=0:halt_on_error=1 UBSAN_OPTIONS=halt_on_error=1:print_stacktrace=1 \
    python -m pytest tests -m "not gpu"

(the GPU kernels themselves are never built with a sanitizer).
"""

from __future__ import annotations

import concurrent.futures as futures
import os
import shlex
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
INCLUDE = ROOT / "include"
BUILD = ROOT / "_build" / "minicompiler_amd"
LIBDIR = PKG / "lib"
LIBRARY = LIBDIR / "libminicompiler_hip.so"
MCC = PKG / "bin" / "mcc"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
ARCH = "gfx950"

CXXFLAGS = ["-std=c++17", "-O2", "-fPIC", "-Wall", "-Wextra", "-Wno-unused-parameter", "-ffp-contract=off",
            f"-I{INCLUDE}", f"-I{CSRC}"]
# Kernels: gfx950 only; packed FP32 instructions off (see the build notes).
HIPFLAGS = ["-std=c++17", "-O3", "-fPIC", f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang",
            "-packed-fp32-ops", "-Wno-unused-command-line-argument", f"-I{INCLUDE}", f"-I{CSRC}"]


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature.
    lines = [l for l in proc.stdout.splitlines() if "packed-fp32-ops' is not a recognized feature" not in l]
    if proc.returncode != 0:
        raise RuntimeError("build step failed:\n" + " ".join(shlex.quote(c) for c in cmd) + "\n" + "\n".join(lines))
    if lines:
        print("\n".join(lines), file=sys.stderr)


# Headers whose text the library embeds, to compile them at run time with
# generated epilogues (csrc/hip/rtc_sources.hpp declares the strings).
EMBEDDED = {"kGemmF32MfmaSource": CSRC / "hip" / "gemm_f32_mfma.h",
            "kGemmF32RingSource": CSRC / "hip" / "gemm_f32_ring.h",
            "kGemmF32NarrowSource": CSRC / "hip" / "gemm_f32_narrow.h",
            "kGemmSplitArrivalSource": CSRC / "hip" / "gemm_split_arrival.h",
            "kGemm16FastSource": CSRC / "hip" / "gemm_mfma16_fast.h",
            "kGemm16FragSource": CSRC / "hip" / "gemm_mfma16_frag.h"}


def _embed() -> Path:
    out = BUILD / "gen" / "rtc_sources.cpp"
    out.parent.mkdir(parents=True, exist_ok=True)
    text = "// Generated by minicompiler_amd/build.py from the embedded headers.\n"
    text += '#include "hip/rtc_sources.hpp"\n\nnamespace minicompiler::hip {\n\n'
    for name, path in EMBEDDED.items():
        body = path.read_text()
        if ")mc_embedded" in body:
            raise RuntimeError(f"{path} contains the raw-string delimiter")
        text += f'const char* const {name} = R"mc_embedded({body})mc_embedded";\n\n'
    text += "}  // namespace minicompiler::hip\n"
    out.write_text(text)
    return out


def _sources() -> tuple[list[Path], list[Path], Path]:
    host = sorted((CSRC / "core").glob("*.cpp")) + sorted((CSRC / "hip").glob("*.cpp")) + [CSRC / "capi.cpp"]
    host.append(_embed())
    kernels = sorted((CSRC / "hip").glob("*.hip"))
    return host, kernels, CSRC / "tools" / "mcc.cpp"


def _object(src: Path) -> Path:
    rel = src.relative_to(CSRC) if src.is_relative_to(CSRC) else src.relative_to(BUILD)
    return BUILD / (str(rel).replace("/", "__") + ".o")


def _compile(src: Path) -> Path:
    obj = _object(src)
    obj.parent.mkdir(parents=True, exist_ok=True)
    if src.suffix == ".hip":
        cmd = [str(ROCM / "bin" / "hipcc"), *HIPFLAGS, "-c", str(src), "-o", str(obj)]
    else:
        cmd = ["g++", *CXXFLAGS]
        if src.name == "hip_rt.cpp":  # the one host file that includes HIP headers
            cmd += [f"-I{ROCM / 'include'}", "-D__HIP_PLATFORM_AMD__"]
        elif src.name == "engine_clock.cpp":  # AMD SMI's header (types only; the library is dlopen'ed)
            cmd += [f"-I{ROCM / 'include'}"]
        cmd += ["-c", str(src), "-o", str(obj)]
    _run(cmd)
    return obj


def build(jobs: int | None = None, verbose: bool = True) -> Path:
    host, kernels, mcc = _sources()
    jobs = jobs or min(16, os.cpu_count() or 4)
    # Kernel TUs first in the queue: they take the longest.
    order = kernels + host
    with futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(_compile, order))
    LIBDIR.mkdir(parents=True, exist_ok=True)
    tmp = LIBRARY.with_suffix(".so.tmp")
    _run([str(ROCM / "bin" / "hipcc"), "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", str(tmp), *map(str, objs),
          f"-L{ROCM / 'lib'}", "-lamdhip64", "-lhiprtc", "-ldl", f"-Wl,-rpath,{ROCM / 'lib'}", "-Wl,--no-undefined"])
    os.replace(tmp, LIBRARY)
    MCC.parent.mkdir(parents=True, exist_ok=True)
    _run(["g++", *CXXFLAGS, str(mcc), "-o", str(MCC), f"-L{LIBDIR}", "-lminicompiler_hip",
          "-Wl,-rpath,$ORIGIN/../lib", f"-Wl,-rpath,{ROCM / 'lib'}"])
    if verbose:
        print(f"built {LIBRARY.relative_to(ROOT)} and {MCC.relative_to(ROOT)}")
    return LIBRARY


SANITIZE_DIR = ROOT / "_build" / "sanitize"
SANITIZE_FLAGS = ["-O1", "-g", "-fno-omit-frame-pointer", "-fsanitize=address,undefined"]


def build_sanitized(jobs: int | None = None) -> Path:
    """The host code with ASan + UBSan, linked with the normal build's kernel
    objects (built first when missing)."""
    host, kernels, _ = _sources()
    kobjs = [_object(k) for k in kernels]
    if not all(o.exists() for o in kobjs):
        build(jobs, verbose=False)
    SANITIZE_DIR.mkdir(parents=True, exist_ok=True)
    flags = [f for f in CXXFLAGS if f != "-O2"] + SANITIZE_FLAGS

    def host_object(src: Path) -> Path:
        obj = SANITIZE_DIR / (src.name + ".o")
        cmd = ["g++", *flags]
        if src.name == "hip_rt.cpp":
            cmd += [f"-I{ROCM / 'include'}", "-D__HIP_PLATFORM_AMD__"]
        elif src.name == "engine_clock.cpp":
            cmd += [f"-I{ROCM / 'include'}"]
        _run(cmd + ["-c", str(src), "-o", str(obj)])
        return obj

    with futures.ThreadPoolExecutor(max_workers=jobs or min(16, os.cpu_count() or 4)) as pool:
        objs = list(pool.map(host_object, host))
    out = SANITIZE_DIR / "libminicompiler_hip.so"
    _run(["g++", "-shared", "-fsanitize=address,undefined", "-o", str(out), *map(str, objs), *map(str, kobjs),
          f"-L{ROCM / 'lib'}", "-lamdhip64", "-lhiprtc", "-ldl", f"-Wl,-rpath,{ROCM / 'lib'}"])
    print(f"built {out.relative_to(ROOT)}")
    return out


if __name__ == "__main__":
    if "--sanitize" in sys.argv[1:]:
        build_sanitized()
    else:
        build()
