"""Builds libsrx_hip.so (HIP kernels + C-ABI runtime) in-tree for gfx950 with hipcc.

Numerics flags: no FMA contraction, IEEE fp32 division and square root, fp32 denormals kept,
so every fp32 expression rounds like the reference's x86 SSE code.  Packed-fp32 instructions are
disabled (they are not needed and some forms misbehave on this platform).
"""
import os
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG, "csrc")
OUT_DIR = os.path.join(PKG, "lib")
OUT = os.path.join(OUT_DIR, "libsrx_hip.so")
SOURCES = ["srx_runtime.cpp", "srx_batch.cpp", "srx_server.cpp", "srx_sasl.cpp", "srx_sasl_jit.cpp", "srx_noalloc.hip",
           "srx_kernels.hip", "srx_raster.hip", "srx_inorder.hip",
           "srx_vis.hip"]
# device headers the SASL shading kernels compiled at run time include (embedded in the library)
JIT_HEADERS = ["srx_device.h", "srx_sampler.h", "srx_sasl_program.h", "srx_shade_common.h", "srx_sasl_exec.h"]
JIT_GEN = os.path.join(OUT_DIR, "srx_jit_sources.gen.h")
ARCH = "gfx950"

FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-ffp-contract=off", "-fno-fast-math",
    "-fno-gpu-flush-denormals-to-zero", "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for c in ("/opt/rocm/bin/hipcc", shutil.which("hipcc") or ""):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found")


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{' '.join(cmd)}\n{res.stdout}\n{res.stderr}")


def write_jit_sources():
    """The text of the device headers as C string literals, for hiprtc at run time."""
    delim = "SRXJIT"
    names, texts = [], []
    for h in JIT_HEADERS:
        with open(os.path.join(CSRC, h)) as f:
            text = f.read()
        assert f"){delim}\"" not in text
        names.append(f'"{h}"')
        texts.append(f'R"{delim}({text}){delim}"')
    body = ("// generated by build.py from the headers in csrc/\n#pragma once\n"
            f"static const int kJitHeaderCount = {len(names)};\n"
            f"static const char* const kJitHeaderName[] = {{{', '.join(names)}}};\n"
            f"static const char* const kJitHeaderText[] = {{\n" + ",\n".join(texts) + "};\n")
    tmp = JIT_GEN + ".tmp"
    with open(tmp, "w") as f:
        f.write(body)
    os.replace(tmp, JIT_GEN)


def build(verbose: bool = False) -> str:
    os.makedirs(OUT_DIR, exist_ok=True)
    write_jit_sources()
    objs = [os.path.join(OUT_DIR, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    cmds = [[hipcc(), *FLAGS, "-I", OUT_DIR, "-c", os.path.join(CSRC, s), "-o", o] for s, o in zip(SOURCES, objs)]
    with ThreadPoolExecutor(len(cmds)) as ex:
        list(ex.map(lambda c: _run(c, verbose), cmds))
    tmp = OUT + ".tmp"
    _run([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs, "-lhiprtc"], verbose)
    os.replace(tmp, OUT)
    for o in objs:
        os.remove(o)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
