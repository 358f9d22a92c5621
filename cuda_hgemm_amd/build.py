"""Builds the native pieces in-tree with hipcc for gfx950:

    cuda_hgemm_amd/lib/libhgemm.so            the kernels + C ABI (include/hgemm.h)
    cuda_hgemm_amd/lib/libhgemm_hipblaslt.so  vendor comparator (include/hgemm_hipblaslt.h)
    cuda_hgemm_amd/lib/_call.so               the Python calls' launcher for torch tensors (where torch is installed)
    cuda_hgemm_amd/bin/hgemm                  C++ benchmark / check driver

Run as ``python -m cuda_hgemm_amd.build`` (add ``--force`` to rebuild everything).
hipcc cross-compiles without a GPU, so this works on a CPU-only machine.
"""
from __future__ import annotations

import concurrent.futures as cf
import importlib.util
import os
import re
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "lib")
BIN = os.path.join(HERE, "bin")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
# -packed-fp32-ops is switched off on purpose: the packed FP32 forms the compiler would
# pick by itself are not trusted on this hardware pool.
# Kernel arguments are preloaded: the dispatcher writes the first 14 to 16 dwords of them into scalar registers before a wave
# starts, where it would otherwise begin with a load and its latency.  0.25 us of every launch that is short enough to show
# it: 256^3 3.07 -> 2.80 us, 512^3 4.01 -> 3.72, 1 x 4096 x 4096 7.08 -> 6.86; level from about 15 us on
# (the persistent decode kernel lost 0.8 % by it until its first copies were held back again, mfma_decode_resident.h).
DEVICE_FLAGS = ["--offload-arch=" + ARCH, "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                "-Xarch_device", "-mllvm=-amdgpu-kernarg-preload-count=16"]
CXXFLAGS = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wextra", "-Wno-unused-parameter", "-I" + INCLUDE]

LIB_SOURCES = ["basic_kernels.hip", "ladder_sync.hip", "ladder_async.hip", "ladder_stages.hip", "tiles_256.hip",
               "tiles_224.hip", "tiles_192.hip", "tiles_160.hip", "tiles_128.hip", "tiles_64.hip", "tiles_unaligned.hip", "dispatch.hip", "api.hip"]
VENDOR_SOURCES = ["vendor_hipblaslt.cpp"]
DRIVER_SOURCES = ["driver/main.cpp"]
PYTHON_CALL_SOURCE = "python_call.cpp"


def _headers():
    out = []
    for root, _, files in os.walk(CSRC):
        out += [os.path.join(root, f) for f in files if f.endswith(".h")]
    out += [os.path.join(INCLUDE, f) for f in os.listdir(INCLUDE)]
    return out


def _stale(target, deps):
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    lines = [l for l in r.stdout.splitlines() if "is not a recognized feature for this target" not in l]
    if r.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), "\n".join(lines)))
    return "\n".join(lines)


# Kernels whose operands and accumulators are handled from inline assembly in an order the
# compiler does not know: a register spill between an LDS read and its wait, or of an
# accumulator, would corrupt results silently, so the build fails if one appears.  The chained
# kernel keeps its accumulators in AGPRs a0 ... a(4*TM*TN-1) that only its asm statements name:
# it must use exactly that many AGPRs (one more would be an accumulator register the compiler
# took for itself) and fewer than 256 VGPRs (beyond them the allocator starts looking for AGPRs).
# (the decode kernel that keeps A in registers is here because a spill of those registers would put A in scratch
# memory and silently cost what the kernel exists to save; the kernel that reads unaligned rows because one of its tiles, with a
# helper that was not inlined, kept its operands in scratch memory and ran 20 times slower)
NO_SPILL_KERNELS = ("hgemm_pipelined_kernel", "hgemm_chained_kernel", "hgemm_decode_resident_kernel", "hgemm_unaligned_kernel")
# sources that must contain such kernels: a remark format the parser no longer understands
# must not turn the guard into a no-op
MUST_CHECK = {"dispatch.hip": NO_SPILL_KERNELS[:3], "tiles_unaligned.hip": NO_SPILL_KERNELS[3:], "tiles_256.hip": NO_SPILL_KERNELS[:2], "tiles_224.hip": NO_SPILL_KERNELS[:2], "tiles_192.hip": NO_SPILL_KERNELS[:2],
              "tiles_160.hip": NO_SPILL_KERNELS[:2], "tiles_128.hip": NO_SPILL_KERNELS[:1], "tiles_64.hip": NO_SPILL_KERNELS[:1]}


def _chained_accumulator_registers(mangled):
    """4 * PTM * PTN of a hgemm_chained_kernel instantiation, from the PipeConfig arguments in
    its mangled name (BM, BN, BK, WAVES_M, WAVES_N, STAGES, MI, ...): 16x16 tiles, 4 registers each."""
    m = re.search(r"PipeConfigI((?:Li\d+E)+)E", mangled)
    if not m:
        raise RuntimeError(f"cannot read the tile configuration out of {mangled}")
    bm, bn, _bk, waves_m, waves_n, _stages, mi = [int(v) for v in re.findall(r"Li(\d+)E", m.group(1))[:7]]
    return 4 * (bm // waves_m // mi) * (bn // waves_n // mi)


def _check_no_spills(src, remarks):
    """`remarks`: output of -Rpass-analysis=kernel-resource-usage for one source file.
    Returns the names of the guarded kernel templates that were seen and checked."""
    usage = {}  # kernel -> {key: value}
    name = None
    for line in remarks.splitlines():
        if "remark: Function Name:" in line:
            name = line.split("Function Name:")[1].split()[0]
            usage[name] = {}
            continue
        if name is None:
            continue
        for key in ("ScratchSize [bytes/lane]:", "VGPRs Spill:", "VGPRs:", "AGPRs:"):
            if "remark:     " + key in line or "remark: " + key in line:
                usage[name][key] = int(line.split(key)[1].split()[0])
    seen = set()
    for name, u in usage.items():
        kind = next((k for k in NO_SPILL_KERNELS if k in name), None)
        if kind is None:
            continue
        missing = [k for k in ("ScratchSize [bytes/lane]:", "VGPRs Spill:", "VGPRs:", "AGPRs:") if k not in u]
        if missing:
            raise RuntimeError(f"{src}: no {missing} remark for kernel {name}: the resource guard cannot check it")
        for key in ("ScratchSize [bytes/lane]:", "VGPRs Spill:"):
            if u[key] != 0:
                raise RuntimeError(f"{src}: kernel {name} has {key} {u[key]}; its inline-assembly schedule "
                                   "needs every operand and accumulator in registers")
        if kind == "hgemm_chained_kernel":
            want = _chained_accumulator_registers(name)
            if u["AGPRs:"] != want or u["VGPRs:"] >= 256:
                raise RuntimeError(f"{src}: kernel {name} uses {u['AGPRs:']} AGPRs and {u['VGPRs:']} VGPRs; its named "
                                   f"accumulators need exactly {want} AGPRs and fewer than 256 VGPRs")
        seen.add(kind)
    for kind in MUST_CHECK.get(os.path.basename(src), ()):
        if kind not in seen:
            raise RuntimeError(f"{src}: the resource guard found no {kind} in the compiler's remarks")
    return seen


def _compile(src, force):
    obj = os.path.join(OBJ, src.replace("/", "_") + ".o")
    path = os.path.join(CSRC, src)
    if force or _stale(obj, [path] + _headers()):
        flags = CXXFLAGS + (DEVICE_FLAGS if src.endswith(".hip") else [])
        if src.startswith("driver/"):
            flags = flags + ["-fopenmp"]
        if src.endswith(".hip"):
            flags = flags + ["-Rpass-analysis=kernel-resource-usage"]
        out = _run([HIPCC] + flags + ["-c", path, "-o", obj])
        if src.endswith(".hip"):
            with open(obj + ".resources.txt", "w") as f:  # registers, scratch and occupancy per kernel, for inspection
                f.write(out)
            try:
                _check_no_spills(src, out)
            except RuntimeError:
                os.remove(obj)
                raise
    return obj


def _torch_string_abi(root):
    """Which std::string the installed torch was built with (1: C++11's), from its CMake configuration; importing it takes seconds."""
    config = os.path.join(root, "share", "cmake", "Torch", "TorchConfig.cmake")
    found = re.search(r"_GLIBCXX_USE_CXX11_ABI=([01])", open(config).read()) if os.path.exists(config) else None
    return found.group(1) if found else "1"


def _build_python_call(force):
    """The module behind HgemmLibrary.call and hgemm() for torch tensors: host code only, against the installed torch."""
    torch = importlib.util.find_spec("torch")
    if torch is None or not torch.submodule_search_locations:
        return None  # a machine without torch: nobody there has a torch tensor either
    if not os.path.exists(os.path.join(sysconfig.get_path("include"), "Python.h")):
        print("Python's headers are not installed: calls on torch tensors will go through ctypes")
        return None
    root = list(torch.submodule_search_locations)[0]
    target, source = os.path.join(LIB, "_call.so"), os.path.join(CSRC, PYTHON_CALL_SOURCE)
    if force or _stale(target, [source, os.path.join(root, "version.py")]):
        _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D_GLIBCXX_USE_CXX11_ABI=" + _torch_string_abi(root), "-I" + os.path.join(root, "include"),
              "-I" + os.path.join(root, "include", "torch", "csrc", "api", "include"), "-I" + sysconfig.get_path("include"), source,
              "-o", target, "-L" + os.path.join(root, "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10"])
    return target


def build(force: bool = False, verbose: bool = False) -> dict:
    for d in (OBJ, LIB, BIN):
        os.makedirs(d, exist_ok=True)
    sources = LIB_SOURCES + VENDOR_SOURCES + DRIVER_SOURCES
    with cf.ThreadPoolExecutor(max_workers=min(8, len(sources))) as pool:
        python_call = pool.submit(_build_python_call, force)
        objs = dict(zip(sources, pool.map(lambda s: _compile(s, force), sources)))
        python_call.result()
    libhgemm = os.path.join(LIB, "libhgemm.so")
    vendor = os.path.join(LIB, "libhgemm_hipblaslt.so")
    driver = os.path.join(BIN, "hgemm")
    lib_objs = [objs[s] for s in LIB_SOURCES]
    if force or _stale(libhgemm, lib_objs):
        _run([HIPCC, "-shared", "-o", libhgemm] + lib_objs)
    ven_objs = [objs[s] for s in VENDOR_SOURCES]
    if force or _stale(vendor, ven_objs):
        _run([HIPCC, "-shared", "-o", vendor] + ven_objs + ["-L/opt/rocm/lib", "-lhipblaslt", "-ldl", "-Wl,-rpath,/opt/rocm/lib"])
    drv_objs = [objs[s] for s in DRIVER_SOURCES]
    if force or _stale(driver, drv_objs + [libhgemm, vendor]):
        _run([HIPCC, "-o", driver] + drv_objs + ["-L" + LIB, "-lhgemm", "-lhgemm_hipblaslt", "-fopenmp",
                                                  "-Wl,-rpath,$ORIGIN/../lib"])
    if verbose:
        print("built", libhgemm, vendor, driver)
    return {"libhgemm": libhgemm, "vendor": vendor, "driver": driver}


if __name__ == "__main__":
    build(force="--force" in sys.argv, verbose=True)
