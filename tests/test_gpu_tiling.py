"""Which workgroup shape a kernel takes follows from the grid, the type and the tap count: sizes on both
sides of each of those lines, against the float64 oracle at the parity tests' bounds."""
import pytest
import torch

from helpers import make_case
from test_gpu_parity import check

pytestmark = pytest.mark.gpu


# data gradient: workgroups (tiles x 16-channel slices x passes of up to nine taps) up to 512 take sixteen
# waves, more take eight (3D: always sixteen); sixteen waves on 16-bit operands hold a step's fragments of
# every tap, whatever the number of taps and of 32-channel steps
DATA_GRADIENT = [
    # dim, batch, cin, cout, size, kernel, transposed
    (1, 128, 64, 16, [5], [3], False),       # 512 workgroups
    (1, 129, 64, 16, [5], [3], False),       # 516
    (2, 16, 64, 24, [6, 7], [4, 4], False),  # two passes: 128
    (2, 43, 96, 16, [3, 5], [4, 3], False),  # two passes of six taps: 516
    (2, 2, 20, 72, [9, 17], [5, 5], False),  # three passes of nine, nine, seven; three steps of channels
    (2, 2, 72, 36, [9, 7], [4, 4], True),    # transposed: scatter alone, and offset / mask gradients alone
    (3, 1, 16, 40, [5, 9, 9], [3, 3, 3], False),
    (3, 2, 36, 16, [3, 4, 5], [2, 3, 2], True),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", DATA_GRADIENT, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_data_gradient_workgroups(case, dtype):
    dim, batch, cin, cout, size, kernel, transposed = case
    stride = 2 if transposed else 1
    check(make_case(dim, transposed, batch=batch, cin=cin, cout=cout, kernel=kernel, stride=[stride] * dim,
                    padding=[1] * dim, dilation=[1] * dim, out_pad=[0] * dim, in_size=size, seed=dim + batch), dtype)
