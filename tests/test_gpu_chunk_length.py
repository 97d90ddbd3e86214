"""Row chunks of over-full experts where the experts' tiles are several rounds of the chip: of at least 256 rows."""

import pytest
import torch

from tests import test_gpu_moe as moe

pytestmark = pytest.mark.gpu


# routes of the fullest expert: below the length from which it is cut, in chunks of 256, in more chunks than there are experts' even shares; E beyond the
# experts of the schedule (32) and within
@pytest.mark.parametrize("T,H,E,I,skew", [(900, 512, 64, 512, 0.25), (1200, 512, 64, 512, 0.5), (6000, 520, 65, 504, 0.9), (1500, 1024, 32, 512, 0.6)])
def test_weight_gradients(T, H, E, I, skew, monkeypatch):
    moe.test_weight_gradients_with_row_chunks(T, H, E, I, skew, monkeypatch)


@pytest.mark.parametrize("T,H,E,I,skew", [(1200, 512, 64, 512, 0.5), (1500, 1024, 32, 512, 0.6)])
@pytest.mark.parametrize("dtype,fp32_weights", [(torch.bfloat16, True), (torch.float16, False)])
def test_joint_launch_equals_separate_launches(T, H, E, I, skew, dtype, fp32_weights, monkeypatch):
    moe.test_joint_backward_launch_equals_separate_launches(T, H, E, I, dtype, fp32_weights, skew, monkeypatch)
