"""Builds libhs.so (the HIP runtime of the hip_standalone device) in-tree for gfx950.

Usage: python -m brian2cuda_amd.build   (or brian2cuda_amd.build.build())

Flags that carry the numerical contract:
  -ffp-contract=off       no fused multiply-add: the expression text fixes every rounding
  -Xclang -target-feature -Xclang -packed-fp32-ops
                          no packed FP32 instructions (v_pk_*_f32) anywhere
  -munsafe-fp-atomics     hardware global FP atomics (effects are additions)
"""
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libhs.so")
SOURCES = ["hs_runtime.hip", "hs_engine.hip", "hs_ops.hip", "hs_hines.hip", "hs_connect.hip", "hs_plastic.hip",
           "hs_sort.hip", "hs_codegen.hip", "hs_resident.hip"]
# the engine sources compiled again at run time for code models (hs_codegen.hip),
# by the names their #include lines use
RTC_SOURCES = [("hs_engine.hip", "hs_engine.hip"), ("hs_device.h", "hs_device.h"), ("hs_internal.h", "hs_internal.h"),
               ("hs_model_exprs.h", "hs_model_exprs.h"), ("hs_model_body.inc", "hs_model_body.inc"),
               ("hs_philox.h", "hs_philox.h"), ("hs_detmath.h", "hs_detmath.h"), ("hs_syncode.h", "hs_syncode.h"),
               ("hs_conndev.h", "hs_conndev.h"), ("hs_cgconn.h", "hs_cgconn.h"),
               ("hs_cgfuncs.h", "hs_cgfuncs.h"),
               ("../../include/hs_models.h", os.path.join("..", "..", "include", "hs_models.h"))]
ARCH = os.environ.get("HS_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fno-fast-math",
    "-munsafe-fp-atomics",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-result",
]

# hs_resident.hip, hs_hines.hip: the polynomials' 64-bit constants stay where they are used (two
# scalar moves) instead of being hoisted out of the step loop, where they exceed
# the scalar registers and are spilled (231 -> 52 spills in the FP64 plain noise model)
SOURCE_FLAGS = {f: ["-mllvm", "-disable-machine-licm"] for f in ("hs_resident.hip", "hs_hines.hip")}


def hipcc_path():
    p = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(p):
        raise RuntimeError("hipcc not found: the HIP runtime cannot be built")
    return p


def write_rtc_sources(path):
    """hs_rtc_sources.inc: the engine sources as C string literals (raw strings,
    split below the compilers' literal limits and joined by adjacency)."""
    names, texts = [], []
    for name, rel in RTC_SOURCES:
        with open(os.path.join(CSRC, rel)) as f:
            text = f.read()
        if ")HSRTC\"" in text:
            raise RuntimeError(f"{rel}: holds the raw-string delimiter")
        parts = [text[k:k + 16000] for k in range(0, len(text), 16000)] or [""]
        names.append(f'"{name}"')
        texts.append("\n".join(f'R"HSRTC({p})HSRTC"' for p in parts))
    out = ["/* generated by brian2cuda_amd/build.py from the engine sources: do not edit */",
           f"static const int hs_rtc_count = {len(names)};",
           "static const char *hs_rtc_names[] = {" + ", ".join(names) + "};",
           "static const char *hs_rtc_texts[] = {"]
    out += [t + "," for t in texts]
    out.append("};")
    with open(path, "w") as f:
        f.write("\n".join(out) + "\n")


def build(verbose=False):
    """Compile every source to an object, then link libhs.so. Always recompiles."""
    hipcc = hipcc_path()
    objs, cmds = [], []
    build_dir = os.path.join(HERE, "_build")
    os.makedirs(build_dir, exist_ok=True)
    write_rtc_sources(os.path.join(build_dir, "hs_rtc_sources.inc"))
    for src in SOURCES:
        path = os.path.join(CSRC, src)
        if not os.path.exists(path):
            continue
        obj = os.path.join(build_dir, src.replace(".hip", ".o"))
        cmd = [hipcc, *HIPCC_FLAGS, *SOURCE_FLAGS.get(src, []), "-I", build_dir, "-c", path, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        cmds.append(cmd)
        objs.append(obj)
    with ThreadPoolExecutor(min(len(cmds), os.cpu_count() or 1, 8)) as pool:
        list(pool.map(lambda c: subprocess.run(c, check=True), cmds))
    tmp = LIB + ".tmp"
    cmd = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs, "-lhiprtc"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    build(verbose="-v" in sys.argv)
    print(LIB)
