"""Which workgroup shape a kernel takes follows from the grid, the type and the tap count: sizes on both
sides of each of those lines, against the float64 oracle at the parity tests' bounds."""
import ctypes

import pytest
import torch

from helpers import make_case, rel_err
from test_gpu_parity import check
from test_zz_no_alloc import SCRATCH_BYTES, _desc, _lib, _run

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


# forward: the (pass, channel slice) units of a tile in one share, in several (whole and ragged last shares,
# shares that begin inside a pass) and one each; outputs in whole quads and not
FORWARD = [
    # dim, batch, cin, cout, size, kernel, transposed
    (2, 1, 16, 16, [3, 3], [1, 1], False),       # one unit: one share
    (2, 1, 16, 20, [5, 5], [4, 4], False),       # two passes of one slice
    (2, 3, 52, 132, [17, 33], [3, 3], False),    # four slices, a ragged one; 128-row tiles
    (2, 1, 84, 40, [9, 7], [5, 5], False),       # three passes of six slices
    (1, 5, 144, 24, [301], [5], False),
    (1, 33, 32, 300, [257], [3], False),         # 198 tiles of 128 rows
    (3, 1, 40, 16, [4, 9, 9], [3, 3, 3], False),  # four passes of three slices
    (2, 2, 36, 72, [9, 11], [4, 4], True),       # grad_input: two passes of five slices, strided
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", FORWARD, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_forward_shares(case, dtype):
    dim, batch, cin, cout, size, kernel, transposed = case
    stride = 2 if transposed else 1
    check(make_case(dim, transposed, batch=batch, cin=cin, cout=cout, kernel=kernel, stride=[stride] * dim,
                    padding=[k // 2 for k in kernel], dilation=[1] * dim, out_pad=[0] * dim, in_size=size,
                    seed=40 + dim + batch), dtype)


def test_forward_without_room_for_partial_sums():
    """The allocation-free forward takes a problem whose shares' partials alone exceed its scratch array: in
    one share, the same sum in another order. Its 4608 positive terms reach a float32 accumulator in at least
    144 additions (32 products each), each rounded to 2^-24 of the sum so far: at most 9e-6 of the result."""
    lib = _lib()
    case = make_case(2, batch=1, cin=512, cout=1536, kernel=[3, 3], stride=[1, 1], padding=[1, 1], dilation=[1, 1],
                     out_pad=[0, 0], in_size=[40, 40], seed=77)
    d = _desc(case, torch.float32)
    assert lib.tvdcn_deform_conv_forward_workspace_size(ctypes.byref(d)) > SCRATCH_BYTES
    y = _run(lib, case, torch.float32, noalloc=True)
    assert rel_err(y, _run(lib, case, torch.float32, noalloc=False)) < 9e-6
