"""Builds ``libfla_gfx950.so`` in-tree with hipcc (gfx950 only).

Run as ``python -m flashy_linear_attention_amd.build``.  hipcc cross-compiles
without a GPU.  One object per (dtype, DC, DO) kernel instantiation, compiled in
parallel, then linked with the C ABI into the package directory; ``_fla_torch.so`` beside it
is the operators' host path against PyTorch (no kernels in it).
"""

from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig
from typing import List

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_ROOT = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
INCLUDE = os.path.join(REPO_ROOT, "include")
OBJ_DIR = os.path.join(PKG_DIR, "csrc", "_obj")
LIB_NAME = "libfla_gfx950.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
BINDING_PATH = os.path.join(PKG_DIR, "_fla_torch.so")

DIMS = (32, 64, 128, 256)
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # hipcc may not form packed fp32 VALU ops on this target
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results in architectural VGPRs (operands may still sit in AGPRs): the S
    # accumulators are read by VALU right away, and the AGPR form costs 32 copies per sub-tile
    "-mllvm", "-amdgpu-mfma-vgpr-form",
    "-Wno-unused-command-line-argument",
    "-I" + INCLUDE,
    "-I" + CSRC,
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the HIP kernels cannot be built")
    return exe


def _run(cmd: List[str]) -> str:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(cmd) + "\n" + proc.stdout)
    return proc.stdout


def _check_no_scratch(report: str, kernel: str) -> None:
    """Fail the build if an instantiation of `kernel` spills registers.  The reverse walk keeps its
    running sums in accumulation registers through MFMAs issued from inline assembly, with the wait
    states they need placed by hand; a spill or reload the register allocator put between two of them
    would get none and read stale values without any error.  `report`: the compiler's
    -Rpass-analysis=kernel-resource-usage remarks."""
    name, seen = None, 0
    for line in report.splitlines():
        if "Function Name:" in line:
            name = line.split("Function Name:")[1].split()[0]
        elif "ScratchSize" in line and name and kernel in name:
            seen += 1
            size = int(line.split("ScratchSize [bytes/lane]:")[1].split()[0])
            if size != 0:
                raise RuntimeError(f"{name} uses {size} bytes of scratch per lane: its hand-placed MFMA wait states "
                                   "assume that no spill code sits between its MFMAs")
    if seen == 0:
        raise RuntimeError(f"no resource report for {kernel}: the spill check did not run")


def _check_waves(report: str, kernel: str, waves: int) -> None:
    """Fail the build if an instantiation of `kernel` (a part of the mangled name) leaves room for fewer than `waves` wavefronts on a
    SIMD: with many small workgroups the kernel's rate goes by how many of them are resident."""
    name, seen = None, 0
    for line in report.splitlines():
        if "Function Name:" in line:
            name = line.split("Function Name:")[1].split()[0]
        elif "Occupancy [waves/SIMD]:" in line and name and kernel in name:
            seen += 1
            if int(line.split("Occupancy [waves/SIMD]:")[1].split()[0]) < waves:
                raise RuntimeError(f"{name} uses registers for fewer than {waves} wavefronts per SIMD")
    if seen == 0:
        raise RuntimeError(f"no resource report for {kernel}: the occupancy check did not run")


def _check_scalar_spills(report: str, kernel: str, most: int) -> None:
    """Fail the build if an instantiation of `kernel` (a part of the mangled name) spills more than `most` scalar registers: each is a
    v_writelane or v_readlane, in the loop over the chunks where the allocator puts it there.  The map of workgroups to parts
    (xcd_item) with a division on either side of a branch cost the normalised forward walk 14 (64 columns) and 24 (32) of them and 3 to
    8 % of its time."""
    name, seen = None, 0
    for line in report.splitlines():
        if "Function Name:" in line:
            name = line.split("Function Name:")[1].split()[0]
        elif "SGPRs Spill:" in line and name and kernel in name:
            seen += 1
            spills = int(line.split("SGPRs Spill:")[1].split()[0])
            if spills > most:
                raise RuntimeError(f"{name} spills {spills} scalar registers, at most {most} so far")
    if seen == 0:
        raise RuntimeError(f"no resource report for {kernel}: the check of scalar spills did not run")


def _compile_inst(args) -> str:
    dtype, dc, do = args
    obj = os.path.join(OBJ_DIR, f"inst_t{dtype}_c{dc}_o{do}.o")
    _run([_hipcc(), *HIPCC_FLAGS, f"-DFLA_INST_DTYPE={dtype}", f"-DFLA_INST_DC={dc}", f"-DFLA_INST_DO={do}",
          "-c", os.path.join(CSRC, "fla_inst.hip"), "-o", obj])
    return obj


def _compile_walk(args) -> str:
    dtype, part = args
    obj = os.path.join(OBJ_DIR, f"walk_t{dtype}_p{part}.o")
    report = _run([_hipcc(), *HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", f"-DFLA_WALK_DTYPE={dtype}",
                   f"-DFLA_WALK_PART={part}", "-c", os.path.join(CSRC, "fla_walk_inst.hip"), "-o", obj])
    if part == 1:
        _check_no_scratch(report, "walk_bwd_rev_kernel")
        _check_no_scratch(report, "walk_bwd_rev_wide_kernel")
    else:  # (the plain forward walk at D = 32; the forward walks without a feature map up to 64 columns, the normalised one among them)
        walk = f"walk_fwd_kernelI{('DF16b', 'DF16_')[dtype]}"
        _check_waves(report, walk + "Li32ELb0ELi0ELb0", 4)
        for width, norm, most in ((32, 0, 0), (64, 0, 0), (32, 1, 4), (64, 1, 0), (32, 2, 0), (64, 2, 0)):
            _check_scalar_spills(report, f"{walk}Li{width}ELb0ELi{norm}ELb0", most)
    return obj


def _compile_other(name: str) -> str:
    obj = os.path.join(OBJ_DIR, f"{name}.o")
    # (the pair kernels without the VGPR form of MFMA: see that file's header)
    flags = [f for f in HIPCC_FLAGS if name != "fla_pair_inst" or f not in ("-mllvm", "-amdgpu-mfma-vgpr-form")]
    _run([_hipcc(), *flags, "-c", os.path.join(CSRC, f"{name}.hip"), "-o", obj])
    return obj


def _compile_torch(_=None) -> str:
    """The operators' host path against this PyTorch (host code only)."""
    import torch
    from torch.utils.cpp_extension import include_paths

    obj = os.path.join(OBJ_DIR, "fla_torch.o")
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I" + INCLUDE,
          *(flag for path in include_paths() for flag in ("-isystem", path)), "-isystem", "/opt/rocm/include",
          "-isystem", sysconfig.get_paths()["include"], "-c", os.path.join(CSRC, "fla_torch.cc"), "-o", obj])
    return obj


def build(jobs: int | None = None, verbose: bool = True) -> str:
    """Compile every kernel instantiation and link the shared library, and the extension module that binds it
    to PyTorch.  Always recompiles."""
    import torch

    os.makedirs(OBJ_DIR, exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 1)
    # (the slowest first)
    work = [(_compile_walk, (t, part)) for part in (1, 0) for t in (0, 1)]
    work += [(_compile_torch, None), (_compile_other, "fla_capi"), (_compile_other, "fla_pair_inst"),
             (_compile_other, "fla_poly_inst")]
    work += [(_compile_inst, (t, dc, do)) for dc in DIMS for do in DIMS for t in (0, 1)]
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(lambda w: w[0](w[1]), work))
    binding = next(o for o in objs if o.endswith("fla_torch.o"))
    objs.remove(binding)
    tmp = LIB_PATH + ".tmp"
    _run([_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-soname," + LIB_NAME, "-o", tmp, *objs])
    os.replace(tmp, LIB_PATH)
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = BINDING_PATH + ".tmp"
    _run(["g++", "-shared", "-o", tmp, binding, LIB_PATH, "-L" + torch_lib, "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu",
          "-ltorch_python", "-Wl,-rpath,$ORIGIN"])
    os.replace(tmp, BINDING_PATH)
    if verbose:
        print(f"built {LIB_PATH} ({os.path.getsize(LIB_PATH) / 1e6:.1f} MB, {len(objs)} objects) and {BINDING_PATH}")
    return LIB_PATH


TRACE_LIB_PATH = os.path.join(OBJ_DIR, "trace", "libfla_trace.so")


def build_trace(jobs: int | None = None) -> str:
    """The host-only trace build of the same sources (``-DFLA_TRACE_LAUNCHES``): a library with the
    same C ABI that makes no launch and writes every launch down instead (kernel, grid, LDS, every
    argument), plus ``fla_trace_take``.  Runs without a GPU; the launch-plan tests load it."""
    out_dir = os.path.dirname(TRACE_LIB_PATH)
    os.makedirs(out_dir, exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 1)
    flags = ["--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-DFLA_TRACE_LAUNCHES",
             "-Wno-unused-command-line-argument", "-I" + INCLUDE, "-I" + CSRC]

    def one(args) -> str:
        src, obj, defs = args
        _run([_hipcc(), *flags, *defs, "-c", os.path.join(CSRC, src), "-o", os.path.join(out_dir, obj)])
        return os.path.join(out_dir, obj)

    work = [("fla_inst.hip", f"inst_t{t}_c{dc}_o{do}.o",
             [f"-DFLA_INST_DTYPE={t}", f"-DFLA_INST_DC={dc}", f"-DFLA_INST_DO={do}"])
            for t in (0, 1) for dc in DIMS for do in DIMS]
    work += [("fla_walk_inst.hip", f"walk_t{t}_p{part}.o", [f"-DFLA_WALK_DTYPE={t}", f"-DFLA_WALK_PART={part}"])
             for t in (0, 1) for part in (0, 1)]
    work += [("fla_capi.hip", "fla_capi.o", []), ("fla_pair_inst.hip", "fla_pair_inst.o", []),
             ("fla_poly_inst.hip", "fla_poly_inst.o", []),
             ("fla_trace.cc", "fla_trace.o", ["-x", "c++"])]
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(one, work))
    # A host-only object still registers its (absent) device code with the HIP runtime when it is
    # loaded: it refers to a code-object symbol that the device link would have made, and calls the
    # runtime's registration hooks.  The trace library brings both itself -- empty code objects and
    # hooks that do nothing, bound inside the library -- so that loading it touches no HIP runtime.
    names = set()
    for obj in objs:
        out = subprocess.run(["nm", "-u", obj], stdout=subprocess.PIPE, text=True, check=True).stdout
        names.update(tok for tok in out.split() if tok.startswith("__hip_fatbin_"))
    stubs = os.path.join(out_dir, "registration_stubs.c")
    with open(stubs, "w") as f:
        for name in sorted(names):
            f.write(f"const char {name}[64] = {{0}};\n")
        f.write("void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }\n"
                "void __hipUnregisterFatBinary(void **h) { (void)h; }\n"
                "void __hipRegisterFunction(void **m, const void *f, char *a, const char *b, unsigned c, void *d,\n"
                "                           void *e, void *g, void *h, int *i) {}\n"
                "void __hipRegisterVar(void **m, void *v, char *a, const char *b, int c, unsigned long d, int e,\n"
                "                      int g) {}\n")
    stubs_obj = os.path.join(out_dir, "registration_stubs.o")
    _run(["gcc", "-O1", "-fPIC", "-c", stubs, "-o", stubs_obj])
    tmp = TRACE_LIB_PATH + ".tmp"
    _run([_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-o", tmp, *objs, stubs_obj])
    os.replace(tmp, TRACE_LIB_PATH)
    return TRACE_LIB_PATH


if __name__ == "__main__":
    if len(sys.argv) > 1 and sys.argv[1] == "trace":
        print(build_trace())
    else:
        build()
    sys.exit(0)
