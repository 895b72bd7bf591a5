"""CPU: the decode kernels' loop as compiled for gfx950 asks for all of a step's cache rows before it waits for the first."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tscale_amd", "csrc")
HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_no_wait_between_a_steps_requests(tmp_path):
    out = tmp_path / "decode.s"
    flags = subprocess.check_output(["make", "-s", "-C", CSRC, "print-flags"], text=True).split()
    subprocess.check_call([HIPCC, *flags, "-S", "--cuda-device-only", os.path.join(CSRC, "decode.hip"), "-o", str(out)], stderr=subprocess.DEVNULL)
    requests, kernel, waited = {}, None, False
    for line in out.read_text().splitlines():
        label = re.match(r"(_ZN\w*decode_(?:split_kernelILi[01]ELi(?:64|128)ELb[01]ELb[01]|wide_kernelILi[01]ELi(?:64|128)ELb[01])ELb0E\w*):", line)  # (without a front)
        if label:
            kernel = label.group(1)
            requests[kernel] = 0
        elif line.startswith(".Lfunc_end"):
            kernel = None
        if kernel is None:
            continue
        if line.startswith(".LBB"):
            waited = False  # a block begins
        elif re.search(r"\ts_waitcnt .*vmcnt", line):
            waited = True
        elif "global_load_dwordx4" in line and line.rstrip().endswith(" nt"):  # a cache row
            assert not waited, kernel
            requests[kernel] += 1
    # two types, two widths, with and without bf16 queries: long and short steps of four waves, near and any stride; of sixteen
    assert sum("split" in k for k in requests) == 32 and sum("wide" in k for k in requests) == 16
    for kernel, n in requests.items():
        rows = int(re.search(r"ELi(\d+)EEEv", kernel).group(1))
        assert n == 2 * rows, (kernel, n)
