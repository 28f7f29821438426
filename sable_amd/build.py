"""Build step of the native library (runs on machines without a GPU).

1. embeds the kernel headers as string literals for hipRTC
   (``csrc/_embedded_src.inc``);
2. compiles ``libsable_amd.so`` with hipcc for gfx950 (host runtime, plan
   builder and the ahead-of-time generic kernels);
3. compiles the hipRTC specialisations the benchmarks and tests use into the
   code-object cache next to the package (``_rtc_cache/``), so a fresh GPU
   host loads them instead of compiling.

``python -m sable_amd.build`` runs all three.
"""
from __future__ import annotations

import ctypes
import os
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG, "csrc")
LIB = os.path.join(PKG, "libsable_amd.so")
RTC_CACHE = os.path.join(PKG, "_rtc_cache")
ARCH = "gfx950"

EMBED = ["sable_device.h", "sable_kernels.h", "sable_mfma.h"]

HIPCC_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "-shared", f"--offload-arch={ARCH}",
    # packed FP32 instructions are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unused-value", "-Wno-unused-result",
]


def hipcc():
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found")


def write_embedded():
    out = os.path.join(CSRC, "_embedded_src.inc")
    parts = ["// generated by sable_amd/build.py: kernel sources for hipRTC\n"]
    for name in EMBED:
        text = open(os.path.join(CSRC, name)).read()
        if ")SBSRC\"" in text:
            raise RuntimeError(f"{name} contains the raw-string delimiter")
        var = "k_src_" + name.replace(".", "_")
        parts.append(f'static const char *{var} = R"SBSRC({text})SBSRC";\n')
    new = "".join(parts)
    if not os.path.exists(out) or open(out).read() != new:
        with open(out, "w") as f:
            f.write(new)
    return out


def build_library(verbose=False):
    write_embedded()
    srcs = [os.path.join(CSRC, "runtime.hip"), os.path.join(CSRC, "plan.cpp"), os.path.join(CSRC, "vbr_text.cpp")]
    tmp = LIB + ".tmp"
    cmd = [hipcc(), *HIPCC_FLAGS, "-o", tmp, *srcs, "-lhiprtc"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("hipcc failed building libsable_amd.so")
    if verbose:
        sys.stderr.write(r.stderr)
    os.replace(tmp, LIB)
    return LIB


# (kind, wg, unroll, xcap, nrhs, rtmax): the specialisations used by the
# benchmarks and tests.  Others are compiled on first use on the GPU host.
PRECOMPILE = [
    (0, wg, u, xcap, 0, 8) for wg in (256, 512) for u in (2, 4) for xcap in (64, 256, 512, 1024, 2048, 4096)
] + [
    (0, 256, 8, xcap, 0, 8) for xcap in (1024, 4096)
] + [
    (1, 128 if n < 64 else 256, 4, 0, n, 1) for n in (4, 8, 12, 16, 32, 48, 64, 72, 80, 128, 256, 512)
] + [
    (k, 256, 4, xcap, n, 8) for k in (2, 3) for n in (16, 32, 64, 128, 256) for xcap in (256, 512, 1024, 2048)
] + [
    (k, wg, 4, 256, n, 8) for k, wg, n in ((2, 128, 96), (2, 256, 96), (3, 256, 96), (2, 256, 144), (2, 128, 160),
                                           (2, 256, 160), (2, 256, 224), (2, 256, 240))
] + [
    (k, 512, 4, xcap, n, 8) for k in (2, 3) for n in (16, 128) for xcap in (512, 1024, 2048)
] + [
    # the 256-matrix batch's SpMM members (N = 16, 128-thread workgroups)
    (k, 128, 4, xcap, 16, 8) for k in (2, 3) for xcap in (256, 512, 1024, 2048)
]


def precompile(specs=PRECOMPILE, jobs=8, prune=True):
    """Compile hipRTC specialisations into RTC_CACHE (in parallel processes).
    With ``prune``, code objects this build did not produce or reuse (stale
    sources or specs) are deleted afterwards."""
    import time
    os.makedirs(RTC_CACHE, exist_ok=True)
    t0 = time.time() - 2.0
    code = (
        "import ctypes,sys\n"
        f"lib=ctypes.CDLL({LIB!r})\n"
        f"lib.sable_set_cache_dir({RTC_CACHE.encode()!r})\n"
        "k,wg,u,xc,n,rt=map(int,sys.argv[1:7])\n"
        f"rc=lib.sable_rtc_precompile(k,wg,u,xc,n,rt,{ARCH.encode()!r})\n"
        "lib.sable_last_error.restype=ctypes.c_char_p\n"
        "sys.exit(0 if rc==0 else print(lib.sable_last_error().decode()) or 1)\n"
    )
    procs, failed = [], []
    for spec in specs:
        procs.append((spec, subprocess.Popen([sys.executable, "-c", code, *map(str, spec)],
                                             stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        if len(procs) >= jobs:
            spec0, p0 = procs.pop(0)
            out, _ = p0.communicate()
            if p0.returncode:
                failed.append((spec0, out.decode()[-2000:]))
    for spec0, p0 in procs:
        out, _ = p0.communicate()
        if p0.returncode:
            failed.append((spec0, out.decode()[-2000:]))
    if failed:
        for spec, msg in failed:
            sys.stderr.write(f"precompile {spec} failed:\n{msg}\n")
        raise RuntimeError("hipRTC precompilation failed")
    if prune:
        for name in os.listdir(RTC_CACHE):
            path = os.path.join(RTC_CACHE, name)
            if name.startswith("sb_") and os.path.getmtime(path) < t0:
                os.remove(path)


def build_all(verbose=False, with_precompile=True):
    build_library(verbose)
    if with_precompile:
        precompile()
    return LIB


if __name__ == "__main__":
    build_all(verbose="-v" in sys.argv, with_precompile="--no-rtc" not in sys.argv)
    print(LIB)
