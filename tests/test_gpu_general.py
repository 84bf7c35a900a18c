"""Seeded random problems of the general kernels (fwd_gather_gemm, bwd_data, bwd_weight) against the float64 oracle:
channel counts in no whole quads, or float64, with columns longer than the few-channel kernels take. test_launch_shapes.py
checks on the host that each problem takes them."""
import random

import pytest
import torch

import tvdcn
from helpers import make_case, rel_err
from test_gpu_blocks import _lib, _per_image
from test_gpu_parity import check, run_oracle

pytestmark = pytest.mark.gpu

SEEDS = range(1200, 1232)


def general_case(seed):
    """(dim, transposed, dtype, make_case arguments): columns of more than 200 values (few-channel kernels: up to 200)"""
    rnd = random.Random(seed)
    dim = rnd.choice((1, 2, 2, 3))
    transposed = rnd.random() < 0.4
    dtype = (torch.float32, torch.float32, torch.float16, torch.bfloat16, torch.float64)[seed % 5]
    groups = rnd.choice((1, 1, 2, 3))
    kernel = {1: [rnd.choice((7, 11))], 2: rnd.choice(([4, 4], [5, 3], [5, 5])), 3: rnd.choice(([3, 3, 2], [2, 4, 3]))}[dim]
    taps = 1
    for k in kernel:
        taps *= k
    # the sampled side: odd multiples, or (float64) whole quads too
    cols = -(-201 // taps)
    cols = -(-cols // (2 * groups)) * 2 * groups
    if dtype != torch.float64 and cols % 4 == 0 and (cols // groups) % 4 == 0:
        cols += 2 * groups
    other = groups * rnd.choice((1, 3, 8, 20, 34))
    cin, cout = (other, cols) if transposed else (cols, other)
    divs = [g for g in (1, 2, 3) if cin % g == 0 and cols % g == 0]
    stride = [rnd.choice((1, 2)) for _ in range(dim)]
    hi = {1: 40, 2: 12, 3: 7}[dim]
    return dim, transposed, dtype, dict(
        batch=rnd.choice((1, 2, 3)), cin=cin, cout=cout, groups=groups, og=rnd.choice(divs), mg=rnd.choice(divs),
        deformable=rnd.random() < 0.9, modulated=rnd.random() < 0.7, bias=rnd.random() < 0.7, kernel=kernel, stride=stride,
        padding=[1] * dim, dilation=[1] * dim, out_pad=[0] * dim, in_size=[rnd.randint(5, hi) for _ in range(dim)], seed=seed,
        offset_scale=rnd.choice((0.5, 2.0, 6.0)))


@pytest.mark.parametrize("seed", SEEDS)
def test_random_general_problem(seed):
    dim, transposed, dtype, params = general_case(seed)
    print(f"seed {seed}: {dtype} dim {dim} transposed {transposed} {params}", flush=True)
    check(make_case(dim, transposed, **params), dtype)


@pytest.mark.parametrize("images", [1, 3])
@pytest.mark.parametrize("transposed,dtype", [(False, torch.float32), (True, torch.float32), (False, torch.float16),
                                              (True, torch.bfloat16)])
def test_general_kernels_in_batch_blocks_of_unaligned_images(transposed, dtype, images):
    """9 channels of 7 x 7 pixels, 5 x 5 taps: no batch-sized tensor's bytes per image are a multiple of 16, so blocks of
    1 or 3 images leave the later ones' pointers 2- or 4-byte aligned."""
    case = make_case(2, transposed, batch=7, cin=9, cout=9, kernel=[5, 5], stride=[1, 1], padding=[2, 2], dilation=[1, 1],
                     in_size=[7, 7], out_pad=[0, 0], seed=1240 + images)
    lib = _lib()
    assert lib.tvdcn_set_max_block_elements(images * _per_image(case)) == 0
    try:
        check(case, dtype)
    finally:
        assert lib.tvdcn_set_max_block_elements(2 ** 31 - 1) == 0


def test_general_kernels_channels_last():
    """A channels-last input of 9 channels: sampled in place, its gradient channels-last."""
    case = make_case(2, batch=2, cin=9, cout=20, kernel=[5, 5], stride=[1, 1], padding=[2, 2], dilation=[1, 1],
                     in_size=[9, 8], out_pad=[0, 0], seed=1250)
    names = ("input", "weight", "offset", "mask", "bias")
    ts = [case[n].to("cuda", torch.float32) for n in names]
    ts[0] = ts[0].contiguous(memory_format=torch.channels_last)
    ts = [t.requires_grad_(True) for t in ts]
    y = tvdcn.deform_conv2d(*ts, padding=2)
    gout = torch.rand(y.shape, generator=torch.Generator().manual_seed(7), dtype=torch.float64)
    y.backward(gout.to("cuda", torch.float32))
    assert ts[0].grad.is_contiguous(memory_format=torch.channels_last)
    ref_out, ref_grads = run_oracle(case, gout, torch.float32)
    assert rel_err(y, ref_out) < 1e-5
    for n, t, r in zip(names, ts, ref_grads):
        assert rel_err(t.grad, r) < 1e-4, n
