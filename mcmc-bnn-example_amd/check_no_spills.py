#!/usr/bin/env python3
"""Build check: the kernels whose tile loads are issued from inline assembly must not spill.

Such a load lands in its register long after the compiler believes the register written; if the
register is spilled to scratch or re-used while the load is in flight, the kernel computes with, or
addresses memory through, corrupted values.  Reads the -Rpass-analysis=kernel-resource-usage remarks of
a compilation and fails if one of those kernels has VGPR spills or uses scratch memory, or if the
file holds none of them.  (Every other inline-assembly load of the library waits for its result inside
the same assembly statement, so the kernels that use only those may spill freely.)

The 64 -> 128 -> 1 kernel keeps 128 sums per lane and at 512 threads has 256 registers for everything: it spills, around
its loops rather than in them.  How much is bounded, so that more of it does not go unnoticed."""
import re
import sys

ASM_LOAD_KERNELS = ("MfmaLayerILi22ELi40ELi2EEE", "MfmaSplitLayer")
# kernel -> bytes of scratch per lane (168 and 152 bytes, 126 and 95 registers, for the two likelihoods)
SCRATCH_BUDGET = {r"hmc_kernel_wide.*ELi512EE": 176, r"hmc_kernel_wide.*ELi256EE": 0}


def budget(name):
    if any(k in name for k in ASM_LOAD_KERNELS):
        return 0
    return next((most for pattern, most in SCRATCH_BUDGET.items() if re.search(pattern, name)), None)


def main(path):
    text = open(path, errors="replace").read()
    blocks = re.split(r"remark: Function Name: ", text)[1:]
    checked, bad = 0, []
    for b in blocks:
        name = b.split()[0]
        most = budget(name)
        if most is None:
            continue
        checked += 1
        spill = int(re.search(r"VGPRs Spill: (\d+)", b).group(1))
        scratch = int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", b).group(1))
        if scratch > most or (spill and most == 0):
            bad.append("%s: %d VGPRs spilled, %d bytes of scratch per lane, at most %d" % (name, spill, scratch, most))
    for line in bad:
        print("check_no_spills: " + line, file=sys.stderr)
    if bad:
        return 1
    if checked == 0:
        print("check_no_spills: no kernel in %s has a bound: the check would be vacuous" % path, file=sys.stderr)
        return 1
    print("check_no_spills: %d kernel(s) in %s within their bounds" % (checked, path))
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1]))
