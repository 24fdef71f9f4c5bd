"""The streaming stores of the built library keep their non-temporal hint.  The
compiler may merge two stores of a kernel into one and then drops it without a
word, which costs a forward pass that is bound by memory 3 to 9 %."""
import collections
import os
import re
import shutil
import subprocess

import pytest

LIBRARY = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oslo_amd", "csrc", "liboslo_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# all 16-byte stores of these kernels are outputs that are written once
KERNELS = ("softmax_fwd_kernel", "softmax_bwd_kernel", "softmax_dropout_bwd_kernel", "norm_fwd_reg_kernel")


@pytest.mark.skipif(not os.path.exists(OBJDUMP) or not os.path.exists(LIBRARY), reason="needs the ROCm tools and the built library")
def test_wide_stores_are_non_temporal(tmp_path):
    shutil.copy(LIBRARY, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    images = [p for p in os.listdir(tmp_path) if "gfx950" in p]
    stores, plain = collections.Counter(), collections.Counter()
    for image in images:
        out = subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", image], cwd=tmp_path, stdout=subprocess.PIPE, text=True)
        family = build = None
        for line in out.stdout:
            if line.endswith(">:\n"):
                build = line.split("<", 1)[1][:-3]
                family = next((k for k in KERNELS if re.match(r"_ZN4oslo\d+%sI" % k, build)), None)
            elif family and "global_store_dwordx4" in line:
                stores[family] += 1
                if " nt" not in line.split("//")[0]:
                    plain[build] += 1
        assert out.wait() == 0
    assert set(stores) == set(KERNELS)
    assert not plain, sorted(plain)[:5]
