"""The matrix-core norm at the row lengths between its two register sets and at its largest, and the backward's ordered
sums at partial counts around their batches, against float64 autograd (the check of test_model_gpu)."""
import pytest
import torch

from test_model_gpu import test_norm_forget_kernel as check

F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


# rows of 832 and 1024: more than the 12 steps of the small register set, and all 16; 1, 8, 9, 40, 64, 65 and 73 row blocks of
# the dW_f partials (batches of 64, tails of 8) and as many dw partial rows per split from 1 to 19; long rows with few outputs
# at and below the row count from which they stay on the vector units (forward under 8 outputs, backward under 12)
@pytest.mark.gpu
@pytest.mark.parametrize("xd,yd,N,D,H", [(F32, BF16, 1, 1024, 16), (F32, BF16, 1024, 832, 16), (F32, F32, 1100, 896, 3),
                                         (BF16, BF16, 5000, 1024, 9), (F32, F16, 8192, 1024, 16),
                                         (F32, BF16, 8200, 768, 12), (F32, BF16, 9300, 1024, 1),
                                         (F32, BF16, 16383, 832, 11), (F32, BF16, 16384, 832, 11),
                                         (F32, BF16, 16384, 832, 7), (F32, BF16, 16384, 832, 8),
                                         (F32, BF16, 16384, 1024, 12)])
def test_norm_edges(xd, yd, N, D, H):
    check(xd, yd, N, D, H)
