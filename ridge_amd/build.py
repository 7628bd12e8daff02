"""Builds the native parts of ridge_amd in-tree.

    python -m ridge_amd.build            # libridge_gemm.so (gfx950) + model + tools
    python -m ridge_amd.build --no-gate  # keep going when a variant spills

Outputs (git-ignored, shipped with the tree):
    ridge_amd/lib/libridge_gemm.so   GEMM kernel table, fills, hipBLASLt comparator
    ridge_amd/lib/libridge_model.so  the cost model behind a C ABI
    ridge_amd/bin/ridge-predict      the model CLI (reference tools/ridge-predict.cpp)
    ridge_amd/bin/ridge-check        correctness + throughput harness (bench/check-gemm.cu)
    ridge_amd/bin/ridge-measure      ground-truth sweep (bench/measure.cu)
    ridge_amd/bin/cal-*              calibration microbenchmarks (bench/calibrate/)

The kernel translation unit is compiled once with the compiler's
kernel-resource-usage remarks; the per-variant VGPR/AGPR/scratch counts are parsed
from them into a generated table, the way the reference copies ptxas -v output
into its variant table (bench/kernels/gemm-mma.cu:377-381). A variant that spills
fails the build (the reference's gate, setup-box.sh:96-104).
"""

import argparse
import os
import re
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
BUILD = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "lib")
BIN = os.path.join(PKG, "bin")
INCLUDE = os.path.join(ROOT, "include")

ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CXX = os.environ.get("CXX", "g++")

# Packed FP32 VALU forms are kept out of every code object built here.
HIP_FLAGS = [
    "--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + INCLUDE, "-I" + CSRC,
]

# Kernel arguments of the library's kernels arrive in scalar registers instead of by
# a load that every workgroup waits for: 0.22 us off each launch (1024^3 5.91 -> 5.69
# us). Not for the calibration benches, whose constants were measured without it.
LIB_HIP_FLAGS = HIP_FLAGS + ["-mllvm", "-amdgpu-kernarg-preload-count=16"]

_RESOURCE_KEYS = {
    "VGPRs": "vgprs",
    "AGPRs": "agprs",
    "TotalSGPRs": "sgprs",
    "ScratchSize [bytes/lane]": "scratch",
    "Occupancy [waves/SIMD]": "occupancy",
    "SGPRs Spill": "sgpr_spill",
    "VGPRs Spill": "vgpr_spill",
    "LDS Size [bytes/block]": "lds",
}


def _run(cmd, capture=False):
    print("  $ " + " ".join(cmd), flush=True)
    if capture:
        p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
        if p.returncode != 0:
            sys.stderr.write(p.stdout + p.stderr)
            raise SystemExit("build step failed: %s" % cmd[0])
        return p.stdout + p.stderr
    subprocess.run(cmd, check=True)
    return ""


def read_variant_list():
    """The registered table, in order, from gemm_variants.def: one key per row,
    (BM,BN,BK,WM,WN,S,G) plus a trailing 1 for RIDGE_VARIANT_PERSISTENT rows
    (0 otherwise), which run a different kernel template."""
    rows = []
    pat = re.compile(r"^\s*RIDGE_VARIANT(_PERSISTENT)?\(([^)]*)\)")
    with open(os.path.join(CSRC, "gemm_variants.def")) as f:
        for line in f:
            m = pat.match(line)
            if m:
                rows.append(tuple(int(x) for x in m.group(2).split(",")) + (1 if m.group(1) else 0,))
    return rows


def parse_resource_remarks(text):
    """Maps (BM,BN,BK,WM,WN,S,G,persistent) -> resource dict from -Rpass-analysis
    output; a row's kernel with non-temporal stores has "nt" behind its key, and the
    small-grid kernel of block n is ("part", n)."""
    out = {}
    cur = None
    name_re = re.compile(r"Function Name: (\S+)")
    tmpl_re = re.compile(
        r"gemmMfma(PingPong|Persistent)?KernelILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E(?:Lb([01])E)?")
    part_re = re.compile(r"gemmMfmaSmallGridKernelILi(\d+)E")
    field_re = re.compile(r"remark:\s+([A-Za-z][A-Za-z /\[\]]*?):\s*(\S+)")
    for line in text.splitlines():
        m = name_re.search(line)
        if m:
            t = tmpl_re.search(m.group(1))
            cur = (tuple(int(x) for x in t.groups()[1:8]) + (1 if t.group(1) == "Persistent" else 0,)
                   if t else None)
            if cur is not None and t.group(9) == "1":
                cur += ("nt",)  # the non-temporal form of a row: gated, not in the table
            part = part_re.search(m.group(1))
            if part:
                cur = ("part", int(part.group(1)))  # likewise
            if cur is not None:
                out[cur] = {}
            continue
        if cur is None:
            continue
        f = field_re.search(line)
        if f and f.group(1).strip() in _RESOURCE_KEYS:
            val = f.group(2)
            key = _RESOURCE_KEYS[f.group(1).strip()]
            out[cur][key] = int(val) if val.isdigit() else val
    return out


def write_resource_table(variants, res, path):
    lines = [
        "// Generated by ridge_amd/build.py from kernel-resource-usage remarks. Do not edit.",
        '#include "gemm_resources.h"',
        "extern \"C\" const ridge_gemm_resources_t ridge_gemm_resource_table[] = {",
    ]
    for v in variants:
        r = res[v]
        lines.append("    {%d, %d, %d, %d, %d},  // %s" % (
            r["vgprs"], r["agprs"], r["sgprs"], r["scratch"], r["occupancy"], v))
    lines.append("};")
    lines.append("extern \"C\" const int ridge_gemm_resource_count = %d;" % len(variants))
    with open(path, "w") as f:
        f.write("\n".join(lines) + "\n")


def build_gemm(gate=True):
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIB, exist_ok=True)
    variants = read_variant_list()
    kobj = os.path.join(BUILD, "gemm_kernels.o")
    remarks = _run([HIPCC] + LIB_HIP_FLAGS + ["-Rpass-analysis=kernel-resource-usage", "-c",
                                          os.path.join(CSRC, "gemm_kernels.hip"), "-o", kobj], capture=True)
    res = parse_resource_remarks(remarks)
    missing = [v for v in variants if v not in res]
    if missing:
        raise SystemExit("no resource remarks for variants %s" % missing)
    spilling = [v for v in res
                if res[v]["scratch"] != 0 or res[v]["vgpr_spill"] != 0 or res[v]["sgpr_spill"] != 0]
    print("  %d variants, %d spilling" % (len(variants), len(spilling)))
    for v in spilling:
        print("    SPILL %s: %s" % (v, res[v]))
    if spilling and gate:
        raise SystemExit("spill gate: %d variant(s) use scratch; a spilling kernel is not a fair "
                         "ground truth" % len(spilling))
    gen = os.path.join(BUILD, "gemm_resources.gen.cpp")
    write_resource_table(variants, res, gen)
    objs = [kobj]
    for src in ("fill.hip", "blaslt.cpp"):
        o = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
        lang = ["-x", "hip"] if src.endswith(".hip") else []
        _run([HIPCC] + (LIB_HIP_FLAGS if lang else HIP_FLAGS) + lang + ["-c", os.path.join(CSRC, src), "-o", o])
        objs.append(o)
    o = os.path.join(BUILD, "gemm_resources.gen.o")
    _run([CXX, "-O2", "-fPIC", "-std=c++17", "-I" + INCLUDE, "-I" + CSRC, "-c", gen, "-o", o])
    objs.append(o)
    so = os.path.join(LIB, "libridge_gemm.so")
    tmp = so + ".tmp"
    _run([HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp] + objs +
         ["-L/opt/rocm/lib", "-lhipblaslt", "-Wl,-rpath,/opt/rocm/lib"])
    os.replace(tmp, so)
    return so


MODEL_SRCS = ["model/model.cpp", "model/hardware.cpp"]


def build_model():
    """libridge_model.so and the ridge-predict CLI: plain C++17, no GPU code."""
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIB, exist_ok=True)
    os.makedirs(BIN, exist_ok=True)
    flags = ["-O2", "-std=c++17", "-fPIC", "-Wall", "-Wextra", "-I" + INCLUDE, "-I" + CSRC]
    objs = []
    for src in MODEL_SRCS + ["model/model_capi.cpp"]:
        o = os.path.join(BUILD, os.path.basename(src).replace(".cpp", ".o"))
        _run([CXX] + flags + ["-c", os.path.join(CSRC, src), "-o", o])
        objs.append(o)
    so = os.path.join(LIB, "libridge_model.so")
    _run([CXX, "-shared", "-o", so + ".tmp"] + objs)
    os.replace(so + ".tmp", so)
    exe = os.path.join(BIN, "ridge-predict")
    _run([CXX] + flags + ["-o", exe + ".tmp", os.path.join(CSRC, "tools", "ridge_predict.cpp")] + objs[:2])
    os.replace(exe + ".tmp", exe)
    return so


CAL_BENCHES = ["cal_mma", "cal_smem_bw", "cal_hbm_bw", "cal_latency"]


def build_tools():
    """Host harnesses over the C ABI (ridge-measure, ridge-check) and the four
    calibration microbenchmarks, all for gfx950."""
    os.makedirs(BIN, exist_ok=True)
    rpath = "-Wl,-rpath,$ORIGIN/../lib,-rpath,/opt/rocm/lib"
    for tool in ("ridge_measure", "ridge_check"):
        src = os.path.join(CSRC, "tools", tool + ".cpp")
        if not os.path.exists(src):
            continue
        exe = os.path.join(BIN, tool.replace("_", "-"))
        _run([HIPCC] + HIP_FLAGS + ["-fopenmp", "-I" + os.path.join(CSRC, "tools"), "-o", exe + ".tmp", src,
                                    "-L" + LIB, "-lridge_gemm", rpath])
        os.replace(exe + ".tmp", exe)
    for bench in CAL_BENCHES:
        exe = os.path.join(BIN, bench.replace("_", "-"))
        _run([HIPCC] + HIP_FLAGS + ["-I" + os.path.join(CSRC, "calibrate"), "-o", exe + ".tmp",
                                    os.path.join(CSRC, "calibrate", bench + ".hip")])
        os.replace(exe + ".tmp", exe)


def build_oracle():
    """The CPU checker (test infrastructure) and, when the reference tree is
    present, the reference's own model build under oracle/_ref/."""
    odir = os.path.join(ROOT, "oracle")
    _run(["make", "-C", odir, "-s"])
    if os.path.isdir("/root/reference/src"):
        _run(["make", "-C", odir, "-s", "ref"])


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--no-gate", action="store_true", help="do not fail on spilling variants")
    ap.add_argument("--only", default="all", choices=["all", "gemm", "model", "tools", "oracle"])
    args = ap.parse_args(argv)
    print("ridge_amd build (%s)" % ARCH, flush=True)
    if args.only in ("all", "gemm"):
        build_gemm(gate=not args.no_gate)
    if args.only in ("all", "model"):
        build_model()
    if args.only in ("all", "tools"):
        build_tools()
    if args.only in ("all", "oracle"):
        build_oracle()
    print("ridge_amd build done", flush=True)


if __name__ == "__main__":
    main()
