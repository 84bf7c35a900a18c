"""The launches of a call, recorded on the host (tests/cpp/launch_recorder.cpp in the place of the HIP runtime): which
kernels a problem takes, and that HIP accepts every grid: not empty, fewer than 2^32 threads along x. No kernel
runs, so the problems may be as large as the entry points take."""
import json
import os
import subprocess
import sys

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
RECORDER = os.path.join(TESTS, "cpp", "launch_recorder.cpp")
F32, F64, F16, BF16 = range(4)
SUCCESS, INVALID_ARGUMENT = 0, 1

# (a process without torch, whose libraries bring the HIP runtime's own symbols)
CHILD = """
import json, sys
sys.path.insert(0, sys.argv[1])
from launch_child import record
print(json.dumps(record(sys.argv[2], sys.argv[3], json.load(sys.stdin))))
"""


def problem(dim, batch, cin, cout, size, kernel, **kw):
    p = dict(dim=dim, batch=batch, cin=cin, cout=cout, size=size, kernel=kernel, transposed=False, dtype=F32, groups=1,
             og=1, mg=1, flags=0, stride=1, padding=0, dilation=1, out_pad=0, bias=True)
    p.update(kw)
    return p


@pytest.fixture(scope="module")
def record(tmp_path_factory):
    """record(problem) -> {"forward" / "backward": {"status", "error", "launches": [(kernel, grid, block)]}}"""
    import tvdcn
    lib = str(tmp_path_factory.mktemp("recorder") / "launch_recorder.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", RECORDER, "-o", lib], check=True)

    def go(p):
        child = subprocess.run([sys.executable, "-c", CHILD, TESTS, lib, tvdcn.extension.HIP_LIB_PATH],
                               input=json.dumps([p]), stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                               timeout=120)
        assert child.returncode == 0, (child.returncode, child.stderr[-2000:])
        return json.loads(child.stdout)[0]

    return go


@pytest.mark.parametrize("batch", [0, 2])
@pytest.mark.parametrize("cin,dtype", [(8, F32), (8, F16), (64, F32), (64, F64)])
def test_transposed_layer_of_an_empty_input_is_refused(record, cin, dtype, batch):
    """A 4 x 4 kernel gives an empty input an output of 1 x 5 pixels but no column to compute it from: an error, before
    any launch, forward and backward."""
    r = record(problem(2, batch, cin, 4, [0, 4], [4, 4], transposed=True, padding=1, dtype=dtype))
    for call in r.values():
        assert call["status"] == INVALID_ARGUMENT and "positive" in call["error"] and not call["launches"]


@pytest.mark.parametrize("cin", [3, 32])
def test_layer_of_an_empty_input_is_refused(record, cin):
    """Padding gives an empty input an output of 2 x 4 pixels: an error, few channels or many."""
    r = record(problem(2, 2, cin, 32, [0, 4], [3, 3], padding=2))
    for call in r.values():
        assert call["status"] == INVALID_ARGUMENT and "positive" in call["error"] and not call["launches"]
    assert record(problem(2, 0, cin, 32, [0, 4], [3, 3], padding=2))["forward"]["status"] == SUCCESS   # empty batch


def blocks(call, kernel):
    return [grid[0] for name, grid, _ in call["launches"] if kernel in name]


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("dim,batch,size,kernel,groups,tiles,threads", [
    # 46M input values: 4.32M data gradient workgroups of 1024 threads, more than one launch takes
    (3, 60000, [2, 2, 2], [3, 3, 3], 24, 60000 * 24 * 3, 1024),
    (2, 2200000, [2, 1], [4, 4], 1, 2200000 * 6 * 2, 512)])
def test_tiles_of_many_small_images(record, dim, batch, size, kernel, groups, tiles, threads, dtype):
    """A tile per (image, 16-channel slice or group, pass of taps), however few its pixels, in one launch or two (the
    scatter and the offset gradients)."""
    r = record(problem(dim, batch, 96, 96, size, kernel, groups=groups, padding=1 if dim == 3 else 2, dtype=dtype, mg=0))
    assert r["backward"]["status"] == SUCCESS, r["backward"]["error"]
    runs = blocks(r["backward"], "bwd_data_win_kernel")
    assert sum(runs) in (tiles, 2 * tiles) and max(runs) * threads < 2 ** 32


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("dtype", [F16, BF16])
def test_layouts_of_many_small_images(record, dtype, transposed):
    """8388600 images of one pixel: a layout block of 256 threads for each of two operands, and others'."""
    r = record(problem(1, 8388600, 16, 16, [1], [1], dtype=dtype, transposed=transposed))
    for call in r.values():
        assert call["status"] == SUCCESS, call["error"]
    assert sum(blocks(r["backward"], "prep16_kernel")) > 2 ** 24


@pytest.mark.parametrize("pixels", [2 ** 28 - 16, 2 ** 28, 2 ** 29 - 32])
def test_few_channels_of_many_pixels(record, pixels):
    """One channel of up to 2^31 - 128 positions: four threads per position below 2^30, the general kernels above."""
    r = record(problem(1, 4, 1, 1, [pixels], [1], og=0, mg=0))
    for call in r.values():
        assert call["status"] == SUCCESS, call["error"]
        assert bool(blocks(call, "few_")) == (4 * pixels < 2 ** 30)


@pytest.mark.parametrize("dim,size,kernel,channels,few", [
    (1, [5000], [13], 9, True), (1, [5041], [13], 9, True), (1, [5042], [13], 9, False), (1, [90000], [13], 5, True),
    (2, [64, 64], [4, 4], 3, True), (2, [64, 65], [4, 4], 3, False), (2, [8, 8], [4, 4], 5, False),
    (2, [300, 300], [4, 4], 2, True), (3, [3, 4, 4], [3, 3, 3], 2, False), (3, [40, 40, 40], [4, 4, 4], 1, True)])
def test_transposed_forward_of_few_channels(record, dim, size, kernel, channels, few):
    """The scatter of the few-channel kernels costs a cache line per (pixel, channel): the general kernels' for more
    channels, on larger grids and in higher rank. The backward, whose weight gradient counts too, stays few."""
    r = record(problem(dim, 1, 16, channels, size, kernel, transposed=True, stride=2, padding=1))
    assert bool(blocks(r["forward"], "few_")) == few and bool(blocks(r["forward"], "bwd_data_kernel")) == (not few)
    assert bool(blocks(r["backward"], "few_data_kernel"))


@pytest.mark.parametrize("dim,batch,channels,size,kernel,launches", [
    (1, 1, 16, [100], 3, 1), (1, 16, 512, [4096], 5, 1), (2, 1, 16, [8, 8], 1, 1), (2, 2, 256, [64, 64], 3, 1),
    (2, 8, 256, [64, 64], 3, 2), (3, 1, 16, [4, 4, 4], 1, 1), (3, 2, 64, [16, 56, 56], 3, 2)])
def test_float32_forward_loops(record, dim, batch, channels, size, kernel, launches):
    """The float32 forward's two loops, of which a flag on the device selects one: two kernels where that is faster
    than one kernel of both, whose launch that is not selected costs 4 us."""
    r = record(problem(dim, batch, channels, channels, size, [kernel] * dim, padding=kernel // 2))
    assert len(blocks(r["forward"], "fwd_win_kernel")) == launches


@pytest.mark.parametrize("dim,batch,cout,size,kernel,in_turn", [
    (2, 255, 16, [3, 4], 4, True), (2, 128, 32, [3, 4], 4, True), (2, 128, 16, [3, 4], 4, False),   # rounds 2 / 2, 2 / 2, 2 / 1
    (2, 300, 16, [3, 4], 4, False), (2, 512, 16, [3, 4], 4, True), (2, 512, 16, [3, 4], 3, False),   # 4 / 3, 4 / 4, one pass
    (1, 256, 16, [20], 16, True), (3, 256, 16, [2, 2, 2], 3, False)])
def test_passes_of_the_scatter(record, dim, batch, cout, size, kernel, in_turn):
    """The transposed forward's passes of up to nine taps: in turn in one workgroup where that takes no more rounds of
    the chip's 256 compute units, a workgroup each otherwise, in 3D and beside the offset gradients."""
    r = record(problem(dim, batch, 32, cout, size, [kernel] * dim, transposed=True, padding=1))
    slices, passes = batch * (cout // 16), (kernel ** dim + 8) // 9
    assert blocks(r["forward"], "bwd_data_win_kernel") == [slices if in_turn else slices * passes]


@pytest.mark.parametrize("kw,launches", [
    (dict(batch=128, size=[5, 4], og=0, mg=0), [256]), (dict(batch=128, size=[10, 25], stride=3), [256, 512]),
    (dict(batch=32, size=[20, 20]), [512])])
def test_passes_of_a_backward(record, kw, launches):
    """The input gradient without offset / mask gradients, with theirs in a launch of their own, in one with theirs."""
    r = record(problem(2, cin=20, cout=24, kernel=[4, 4], padding=1, **kw))
    assert blocks(r["backward"], "bwd_data_win_kernel") == launches


def test_random_general_problems_take_the_general_kernels(record):
    import torch
    from test_gpu_general import SEEDS, general_case
    codes = {torch.float32: F32, torch.float64: F64, torch.float16: F16, torch.bfloat16: BF16}
    for seed in SEEDS:
        dim, transposed, dtype, p = general_case(seed)
        r = record(problem(dim, p["batch"], p["cin"], p["cout"], p["in_size"], p["kernel"], transposed=transposed,
                           dtype=codes[dtype], groups=p["groups"], og=p["og"] * p["deformable"], mg=p["mg"] * p["modulated"],
                           stride=p["stride"], padding=1, bias=p["bias"]))
        assert r["forward"]["status"] == SUCCESS and r["backward"]["status"] == SUCCESS, (seed, r["backward"]["error"])
        names = "".join(n for c in r.values() for n, _, _ in c["launches"])
        for kernel in ("bwd_data_kernel", "bwd_weight_kernel", "fwd_gather_gemm_kernel"):
            assert kernel in names, (seed, kernel)
        assert "few_" not in names and "_win_kernel" not in names, seed


@pytest.mark.parametrize("batch", [65532, 65533])
def test_layout_copy_of_many_images(record, batch):
    """The float32 backward's layout copy has a grid slice per image and one for each job beside it, at most 65535."""
    r = record(problem(1, batch, 16, 16, [512], [3], padding=1))
    assert r["backward"]["status"] == SUCCESS
    (copy,) = [grid for name, grid, _ in r["backward"]["launches"] if "to_cl" in name]
    assert copy[2] == 65535   # the mask's check, the weight's magnitude, and the bias gradient or one image more
    assert bool(blocks(r["backward"], "bias_grad_kernel")) == (batch == 65533)
