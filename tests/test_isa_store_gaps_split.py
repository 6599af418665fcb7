"""The store-data hazard check of test_isa_store_gaps.py over the split-bf16 fp32 kernels."""
import subprocess

import pytest

from my_own_cnn_amd import build as B
from tests.test_isa_store_gaps import store_gaps


@pytest.mark.parametrize("src", ["conv_f32_split.hip", "conv_f32_split_grad.hip"])
def test_every_wide_store_is_followed_by_two_wait_states(src, tmp_path):
    dst = tmp_path / "k.s"
    subprocess.run([B.hipcc(), *B.common_flags(), "--cuda-device-only", "-S", str(B.CSRC / src), "-o", str(dst)],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    lines = dst.read_text().splitlines()
    assert any("v_mfma_f32_16x16x32_bf16" in ln for ln in lines)
    short = [g for g in store_gaps(lines) if g[3] < 2]
    assert not short, short[:5]
