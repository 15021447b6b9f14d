"""Build libMMFFmulti_lib.so (HIP kernels for gfx950 + host C++ + C-ABI) in-tree.

    python -m firecore_amd.build        # or firecore_amd.build.build()
"""
import json
import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libMMFFmulti_lib.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# packed FP32 instructions are disabled for all device code
COMMON = ["-O3", "-std=c++17", "-fPIC", "-Wno-unused-command-line-argument",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
HIP_FLAGS = ["-x", "hip", "--offload-arch=" + ARCH, "-munsafe-fp-atomics", "-fno-hip-fp32-correctly-rounded-divide-sqrt"]
# the compiler reports what each kernel uses (registers, scratch, LDS): see check_scratch
RES_FLAGS = ["-Rpass-analysis=kernel-resource-usage"]
RESOURCES = os.path.join(OBJ, "resources.json")
HOST_FLAGS = ["-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include"]

HIP_SOURCES = ["relax_persistent.hip", "split_kernels.hip", "sample_kernels.hip", "proposal_train.hip",
               "gridff_gen.hip"]
CPP_SOURCES = ["molgen.cpp", "topology.cpp", "gridff_host.cpp", "builder.cpp", "database.cpp", "world.cpp", "train.cpp", "capi.cpp"]


def kernel_resources(remarks):
    """{kernel: {quantity: value}} of the compiler's resource-usage remarks."""
    out, cur = {}, None
    for q, v in re.findall(r"remark: +([A-Z][\w ]*?)(?: \[[^\]]*\])?: (\S+) \[-Rpass-analysis=kernel-resource-usage\]",
                           remarks):
        if q == "Function Name":
            cur = out.setdefault(v, {})
        elif v.isdigit():
            cur[q] = int(v)
    return out


def check_scratch(res):
    """No kernel may use scratch memory.  In a build of the relaxation kernel that spilled, the
    compiler stored a spilled address at a loop exit before it restored the execution mask: the
    reload gave garbage and the GPU faulted.  Many instances use all 168 registers that three
    waves per SIMD leave them, so one more live value is enough."""
    if not res:
        raise RuntimeError("the compiler gave no resource-usage remarks: cannot tell whether kernels spill")
    bad = [k for k, r in res.items() if r["ScratchSize"] or r["VGPRs Spill"]]
    if bad:
        raise RuntimeError("kernels with scratch memory (register spills): " + ", ".join(
            "%s (%d B per lane, %d VGPRs)" % (k, res[k]["ScratchSize"], res[k]["VGPRs Spill"]) for k in bad))


def resources():
    """What the kernels of the last build use."""
    with open(RESOURCES) as f:
        return json.load(f)


def _compile(src):
    path = os.path.join(CSRC, src)
    obj = os.path.join(OBJ, src + ".o")
    if src.endswith(".hip"):
        cmd = [HIPCC] + COMMON + HIP_FLAGS + RES_FLAGS + ["-c", path, "-o", obj]
    else:
        cmd = [HIPCC] + COMMON + HOST_FLAGS + ["-c", path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("compile failed: %s\n%s\n%s" % (" ".join(cmd), r.stdout, r.stderr))
    if not src.endswith(".hip"):
        return obj, {}
    res = kernel_resources(r.stderr)
    check_scratch(res)
    return obj, res


def build(verbose=False):
    os.makedirs(OBJ, exist_ok=True)
    srcs = HIP_SOURCES + CPP_SOURCES
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        done = list(ex.map(_compile, srcs))
    objs = [obj for obj, _ in done]
    with open(RESOURCES, "w") as f:
        json.dump({k: r for _, res in done for k, r in res.items()}, f, indent=1)
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", "-fPIC", "--offload-arch=" + ARCH, "-o", tmp] + objs + ["-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed: %s\n%s\n%s" % (" ".join(cmd), r.stdout, r.stderr))
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
