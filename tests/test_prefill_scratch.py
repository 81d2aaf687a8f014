"""The prefill attention's kernels keep their registers: one that spills needs
scratch memory, which the runtime sets up on a stream at its first such launch
-- inside the first prompt of every engine.  Compiled here for the check."""
import os
import re
import shutil
import subprocess

import pytest

from ligguf_amd import build as B


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_attention_kernels_use_no_scratch(tmp_path):
    out = tmp_path / "k.s"
    subprocess.run([B.HIPCC, *B.HIP_FLAGS, "--cuda-device-only", "-S", os.path.join(B.CSRC, "lg_pfattn.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    asm = out.read_text()
    sizes = dict(zip(re.findall(r"^\s*\.name:\s+(_Z\S+)", asm, re.M), map(int, re.findall(r"\.private_segment_fixed_size:\s+(\d+)", asm))))
    assert len(sizes) >= 25 and not {k: v for k, v in sizes.items() if v}
