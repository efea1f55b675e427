"""The build's check of accumulation registers (mam4xx_amd/build.py), on messages
in the compiler's form."""
import pytest

from mam4xx_amd import build as B

HEAD = "/x/mam4x.hip:253:1: remark: "
TAIL = " [" + B.USAGE_FLAG + "]\n"


def messages(kernel, agprs):
    return (HEAD + "Function Name: " + kernel + TAIL + "  253 | __global__ void f() {\n      | ^\n"
            + HEAD + "    VGPRs: 256" + TAIL + HEAD + "    AGPRs: %d" % agprs + TAIL
            + "/x/mam4x.hip:9:5: warning: loop not unrolled [-Wpass-failed]\n    9 |   for\n"
            + "1 warning generated when compiling for gfx950.\n")


@pytest.mark.parametrize("kernel,agprs,ok", [
    ("_ZN12_GLOBAL__N_117chain_post_kernelILb1EN5mam4x4Fp64ENS_9OneDomainEEEvT1_NS_4WorkE", 0, True),
    ("_ZN12_GLOBAL__N_117chain_post_kernelILb1EN5mam4x4Fp64ENS_9OneDomainEEEvT1_NS_4WorkE", 4, False),
    ("_ZN12_GLOBAL__N_117chain_post_kernelILb1EN5mam4x8Fp64DiagENS_9OneDomainEEEvT1_NS_4WorkE", 58,
     True),
    ("_ZN12_GLOBAL__N_116soa_queue_kernelENS_4WorkEPy", 1, False),
    ("_ZN12_GLOBAL__N_115adj_post_kernelILb0EEEvN5mam4x9ChainArgsENS_7AdjWorkE", 256, True),
])
def test_kernels_outside_the_list_are_refused(kernel, agprs, ok):
    rest, regs = B.split_remarks(messages(kernel, agprs))
    assert regs == {kernel: agprs}
    assert rest == ["/x/mam4x.hip:9:5: warning: loop not unrolled [-Wpass-failed]", "    9 |   for",
                    "1 warning generated when compiling for gfx950."]
    if ok:
        B.check_registers(regs)
    else:
        with pytest.raises(RuntimeError, match="accumulation"):
            B.check_registers(regs)


def test_a_build_without_remarks_is_refused():
    with pytest.raises(RuntimeError, match="no kernel"):
        B.check_registers({})
