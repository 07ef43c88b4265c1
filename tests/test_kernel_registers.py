"""Kernels that keep their operands in registers do so: none of them lies in scratch memory, which a walk would read again at every block."""
import os
import re
import subprocess

import pytest

from minivllm_amd.csrc import build


@pytest.mark.parametrize("source, kernel, least", [("attention_latent_heads.hip", "attention_latent_heads_kernel", 2)])
def test_no_register_lies_in_memory(source, kernel, least):
    hipcc = build.find_hipcc()
    if hipcc is None:
        pytest.skip("no compiler")
    done = subprocess.run([hipcc, *build.BASE_FLAGS, *build.VARIANT_DEFINES["bf16"], "-Rpass-analysis=kernel-resource-usage", "-c",
                           os.path.join(build.CSRC, source), "-o", os.devnull], capture_output=True, text=True)
    assert done.returncode == 0, done.stderr[-2000:]
    scratch = re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", done.stderr, re.S)
    ours = {name: int(size) for name, size in scratch if kernel in name}
    assert len(ours) >= least and not any(ours.values()), ours
