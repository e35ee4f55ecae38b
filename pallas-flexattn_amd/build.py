"""Build libflexattn.so (HIP kernels + C ABI) for gfx950, in-tree.

    python pallas-flexattn_amd/build.py
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
OUT = os.path.join(HERE, "pallas_flexattn", "libflexattn.so")
CSRC = os.path.join(HERE, "csrc")
# translation units: (source, extra defines, object name).  kernels.hip holds
# the tile-kernel instantiations and is compiled once per head dim and
# direction, so the objects build in parallel.
UNITS = [(os.path.join(CSRC, "capi.hip"), [], "capi"), (os.path.join(CSRC, "kernels_fp8.hip"), [], "kernels_fp8"),
         (os.path.join(CSRC, "host.cpp"), [], "host")] + [
    (os.path.join(CSRC, "kernels.hip"), [f"-DFA_KERNELS_D={d}", f"-DFA_KERNELS_BWD={bwd}"],
     f"kernels_d{d}_{'bwd' if bwd else 'fwd'}")
    for d in (128, 64, 32) for bwd in (1, 0)]
SOURCES = sorted({u[0] for u in UNITS})
# CPython extension over torch tensors (host code, links against torch)
LAUNCH_SRC = os.path.join(CSRC, "torch_launch.cpp")
LAUNCH_OUT = os.path.join(HERE, "pallas_flexattn", "_launch.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CXX = os.environ.get("CXX", "g++")  # host-only units (.cpp)
HOST_FLAGS = ["-O3", "-std=c++17", "-fPIC", "-pthread", "-Wall"]

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-shared", "-fPIC",
    # keep packed-fp32 VALU instructions out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA accumulators in VGPRs where they fit: fewer AGPR<->VGPR copies in
    # the backward kernels (about 3% faster there, forward unchanged)
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",
    # the hand-ordered tiles are fully unrolled step sequences; past the default
    # size limit a partly unrolled loop indexes the register arrays dynamically
    # and they go to scratch
    "-mllvm", "-pragma-unroll-threshold=200000",
    "-I" + os.path.join(REPO, "include"),
    # generated: the kernel headers as strings for run-time compiles (write_rtc_sources)
    "-I" + os.path.join(HERE, "_build"),
]


# kernel headers the library embeds for run-time compiles of user mods
RTC_HEADERS = ["index.h", "common.h", "dma.h", "kargs.h", "fwd.h", "fwd_bf16.h", "bwd.h", "bwd_bf16.h", "f32_split.h"]
GEN_DIR = os.path.join(HERE, "_build")


def write_rtc_sources() -> str:
    """_build/rtc_sources.inc: the kernel headers as string literals (names,
    sources, count) for hiprtcCreateProgram."""
    import hashlib
    os.makedirs(GEN_DIR, exist_ok=True)
    delim = "FA_RTC_SRC"
    names, texts = [], []
    digest = hashlib.sha256()
    for h in RTC_HEADERS:
        with open(os.path.join(HERE, "csrc", h)) as f:
            text = f.read()
        if f"){delim}\"" in text:
            raise RuntimeError(f"{h} contains the raw-string delimiter")
        names.append(f'"{h}"')
        texts.append(f'R"{delim}({text}){delim}"')
        digest.update(h.encode() + b"\0" + text.encode() + b"\0")
    out = os.path.join(GEN_DIR, "rtc_sources.inc")
    # identifies the embedded headers: a code blob compiled from other headers
    # (other kernel argument layouts) is refused by fa_mods_load
    body = ("// generated by build.py from csrc/ -- do not edit\n"
            f"static const unsigned long long kRtcHash = 0x{digest.hexdigest()[:16]}ULL;\n"
            f"static const int kRtcHeaders = {len(names)};\n"
            f"static const char* const kRtcHeaderNames[] = {{{', '.join(names)}}};\n"
            "static const char* const kRtcHeaderSources[] = {\n" + ",\n".join(texts) + "\n};\n")
    with open(out, "w") as f:
        f.write(body)
    return out


def _run(cmd):
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    errs = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    return res.returncode, errs


def compile_units(extra_flags=(), suffix=".o", out_dir=None, jobs=None):
    """Compile every unit with FLAGS (minus -shared) plus extra_flags; returns
    the output paths.  Raises with hipcc's messages on the first failure."""
    out_dir = out_dir or GEN_DIR
    os.makedirs(out_dir, exist_ok=True)
    base = [f for f in FLAGS if f != "-shared"]
    cmds, outs = [], []
    for src, defs, name in UNITS:
        if src.endswith(".cpp"):  # host code: no device pass (skipped for device-only outputs)
            if "--cuda-device-only" in extra_flags:
                continue
            cmd = [CXX, *HOST_FLAGS, *defs, *[f for f in extra_flags if f in ("-c", "-S")], src]
        else:
            cmd = [HIPCC, *base, *defs, *extra_flags, src]
        out = os.path.join(out_dir, name + suffix)
        cmds.append(cmd + ["-o", out])
        outs.append(out)
    jobs = jobs or min(len(cmds), max(1, (os.cpu_count() or 2) - 1))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        results = list(ex.map(_run, cmds))
    for (rc, errs), out in zip(results, outs):
        if rc != 0:
            raise RuntimeError(f"compile failed on {os.path.basename(out)} ({rc}):\n{errs}")
    return outs, [e for _, e in results]


def build_launch() -> str:
    """pallas_flexattn/_launch.so against the installed torch's headers and libraries."""
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    lib = os.path.join(root, "lib")
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           sysconfig.get_paths()["include"]]
    tmp = LAUNCH_OUT + ".tmp"
    rc, errs = _run([CXX, "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                     *[f"-isystem{d}" for d in inc], LAUNCH_SRC, "-o", tmp, "-L" + lib, "-ltorch_python", "-ltorch_cpu",
                     "-lc10", "-Wl,-rpath," + lib])
    if rc != 0:
        raise RuntimeError(f"compile failed on {os.path.basename(LAUNCH_SRC)} ({rc}):\n{errs}")
    os.replace(tmp, LAUNCH_OUT)
    return LAUNCH_OUT


def build(verbose: bool = False) -> str:
    tmp = OUT + ".tmp"
    launch = ThreadPoolExecutor(max_workers=1).submit(build_launch)
    write_rtc_sources()
    objs, logs = compile_units(["-c"])
    rc, errs = _run([HIPCC, "-shared", "-fPIC", "-pthread", *objs, "-o", tmp, "-L/opt/rocm/lib", "-lhiprtc",
                     "-Wl,-rpath,/opt/rocm/lib"])
    if rc != 0:
        raise RuntimeError(f"link failed ({rc}):\n{errs}")
    if verbose:
        for e in logs + [errs]:
            if e.strip():
                print(e, file=sys.stderr)
    os.replace(tmp, OUT)
    launch.result()
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
