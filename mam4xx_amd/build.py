"""Build recipe of the HIP library (gfx950) -- called by __graft_entry__.build().

Produces ``mam4xx_amd/lib/libmam4x.so`` in-tree (git-ignored; it travels to
the GPU box with the source tree).
"""
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libmam4x.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["mam4x.hip", "chain_consts.cpp"]
HIP_FLAGS = [
    "-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC", "-shared",
    # packed-FP32 VALU forms are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the FP64 drop-in performs the reference's IEEE operations one by one
    # (no a*b+c fusion), so it differs from the CPU build only in libm bits
    "-ffp-contract=off",
    "-Wall", "-Wno-unused-variable", "-Wno-unused-but-set-variable",
]


# Kernels that may keep values in accumulation registers, because they need more
# than 256 vector registers.  Copies there inside divergent branches have lost the
# lanes that were off (the diagnostics finish kernel's overcast cells, the
# sub-stepped tangent's), so each of these is compared with single-lane runs, bit
# for bit, in tests/test_gpu_lanes.py (gas_chem_kernel: cell by cell with the
# oracle, tests/test_gpu_gas_chem.py).  A kernel outside the list fails the build.
ACC_KERNELS = re.compile(r"gas_chem_kernel|chain_fused_kernel|chain_fused_order_kernel|"
                         r"chain_adjoint_kernel|chain_adjoint_sub_kernel|adj_post_kernel|"
                         r"chain_post_kernel.*Fp64Diag")
USAGE_FLAG = "-Rpass-analysis=kernel-resource-usage"
_DIAG = re.compile(r"^\S+:\d+:\d+: (remark|warning|error|note|fatal error): (.*)")


def split_remarks(text):
    """The compiler's messages without its register remarks, and {kernel's mangled
    name: accumulation registers} from those."""
    rest, regs, name, skip = [], {}, None, False
    for line in text.splitlines():
        m = _DIAG.match(line)
        if m:
            skip = m.group(1) == "remark"
        elif not line.startswith(" "):
            skip = False
        if not skip:
            rest.append(line)
        elif m:
            k, _, v = m.group(2).replace("[" + USAGE_FLAG + "]", "").strip().partition(": ")
            if k == "Function Name":
                name = v
            elif k == "AGPRs":
                regs[name] = int(v)
    return rest, regs


def check_registers(regs):
    """No kernels, or one outside ACC_KERNELS with accumulation registers, raise."""
    if not regs:
        raise RuntimeError("the compiler reported no kernel's registers")
    bad = ["%s: %d" % (n, a) for n, a in sorted(regs.items()) if a and not ACC_KERNELS.search(n)]
    if bad:
        raise RuntimeError("accumulation registers in kernels that tests/test_gpu_lanes.py does "
                           "not cover:\n  " + "\n  ".join(bad))


def build(verbose=False, extra_flags=()):
    os.makedirs(LIBDIR, exist_ok=True)
    srcs = [os.path.join(CSRC, s) for s in SOURCES]
    cmd = [HIPCC] + HIP_FLAGS + [USAGE_FLAG] + list(extra_flags) + ["-o", LIB + ".tmp"] + srcs
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, stderr=subprocess.PIPE, text=True)
    rest, regs = split_remarks(r.stderr)
    if rest:
        print("\n".join(rest), file=sys.stderr, flush=True)
    r.check_returncode()
    check_registers(regs)
    os.replace(LIB + ".tmp", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True, extra_flags=sys.argv[1:])
