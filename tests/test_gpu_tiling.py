"""Which workgroup shape a kernel takes follows from the grid, the type and the tap count: sizes on both
sides of each of those lines, against the float64 oracle at the parity tests' bounds."""
import ctypes

import pytest
import torch

import tvdcn
from helpers import make_case, rel_err
from test_gpu_parity import TOL, check, run_gpu, run_oracle
from test_zz_no_alloc import SCRATCH_BYTES, _desc, _lib, _run

pytestmark = pytest.mark.gpu


# data gradient: workgroups (tiles x 16-channel slices x passes of up to nine taps) up to 512 take sixteen
# waves, more take eight (3D: always sixteen; the scatter alone with passes in turn: eight float32, sixteen
# 16-bit); sixteen waves on 16-bit operands hold a step's fragments of
# every tap, unless the step's weight is staged in LDS (1D / 2D passes of nine taps)
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


# the scatter alone with several passes on grids that fill the chip: the passes in turn in one workgroup, which
# rescales its window to a pass of larger terms and sends it out before one that is not finite
PASSES_IN_TURN = [
    # dim, batch, cin, cout, size, kernel: slices x passes
    (1, 64, 36, 52, [7], [16]),      # 256 x 2
    (2, 128, 20, 24, [3, 4], [4, 4]),   # 256 x 2
    (2, 130, 36, 20, [2, 3], [5, 5]),   # 260 x 3: nine taps, staged weights
]


def passes_case(dim, batch, cin, cout, size, kernel, seed):
    return make_case(dim, True, batch=batch, cin=cin, cout=cout, kernel=kernel, stride=[1] * dim, padding=[1] * dim,
                     dilation=[1] * dim, out_pad=[0] * dim, in_size=size, seed=seed)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", PASSES_IN_TURN, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_passes_in_turn(case, dtype):
    check(passes_case(*case, seed=70 + case[0]), dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("kw", [dict(deformable=False, modulated=False, stride=[1, 1], in_size=[5, 4]),
                                dict(stride=[3, 3], in_size=[10, 25])], ids=["offset_free", "scatter_apart"])
def test_passes_in_turn_of_a_backward(kw, dtype):
    """The input gradient of a convolution by itself: nothing but it to compute from the columns, or a window too small
    beside the one of the offset gradients. 128 images of two slices, two passes."""
    check(make_case(2, False, batch=128, cin=20, cout=24, kernel=[4, 4], padding=[1, 1], dilation=[1, 1],
                    out_pad=[0, 0], seed=77, **kw), dtype)


@pytest.mark.parametrize("kind", ["growing", "shrinking", "one_large", "inf_first", "inf_later", "nan_last"])
@pytest.mark.parametrize("case", PASSES_IN_TURN, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_passes_in_turn_of_unlike_magnitudes(case, kind):
    """The mask of each pass on a scale of its own (2^40: nothing of the earlier passes is left in a window on that
    scale, and nothing of them in the sum's 24 bits), or with a value that is not finite in one of them."""
    c = passes_case(*case, seed=80 + case[0])
    kn, dim = c["weight"][0, 0].numel(), case[0]
    passes = (kn + 8) // 9
    per = (kn + passes - 1) // passes
    mask = c["mask"].clone()
    taps = mask.view(mask.shape[0], kn, -1)
    for t in range(kn):
        p = t // per
        taps[:, t] *= {"growing": 2.0 ** (6 * p), "shrinking": 2.0 ** (-7 * p),
                       "one_large": 2.0 ** 40 if p == 1 else 1.0}.get(kind, 1.0)
        if (kind, p) in (("inf_first", 0), ("inf_later", 1)):
            taps[:, t, 3] = float("inf")
        if kind == "nan_last" and p == passes - 1:
            taps[:, t, 3] = float("nan")
    c["mask"] = mask
    out, _, _ = run_gpu(c, torch.float32)
    ref, _ = run_oracle(c, torch.zeros(c["out_shape"], dtype=torch.float64), torch.float32)
    out = out.detach().double().cpu()
    assert torch.equal(torch.isnan(out), torch.isnan(ref)) and torch.equal(torch.isinf(out), torch.isinf(ref))
    assert torch.isfinite(ref).any() and torch.isfinite(ref).all() == (kind in ("growing", "shrinking", "one_large"))
    fin = torch.isfinite(ref)
    e = rel_err(out[fin], ref[fin])
    assert e < TOL[torch.float32][0], f"forward rel err {e}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("case", PASSES_IN_TURN, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_passes_in_turn_past_the_range_of_a_cell(case, dtype):
    """Every (pixel, tap) on the same position with the same term: 2^27 units at most each, of which a cell holds
    16, so the window wraps in each pass."""
    c = passes_case(*case, seed=90 + case[0])
    dim, size, cin = case[0], case[4], case[2]
    kn, kernel = c["weight"][0, 0].numel(), list(c["weight"].shape[2:])
    term = 1.9375
    c["input"], c["mask"] = torch.ones_like(c["input"]), torch.ones_like(c["mask"])
    c["weight"] = torch.full_like(c["weight"], term / cin)
    taps = torch.cartesian_prod(*[torch.arange(k) for k in kernel]).view(kn, dim)
    pixels = torch.cartesian_prod(*[torch.arange(n) for n in size]).view(-1, dim)
    pos = taps[:, :, None] + pixels.T[None] - 1     # (tap, axis, pixel) at stride 1, padding 1
    c["offset"] = (2 - pos).to(c["offset"].dtype).expand(c["offset"].shape[0], -1, -1, -1).reshape(c["offset"].shape)
    out, _, _ = run_gpu(c, dtype)
    ref, _ = run_oracle(c, torch.zeros(c["out_shape"], dtype=torch.float64), dtype)
    assert ref.max() > 48 * term
    e = rel_err(out, ref)
    assert e < TOL[dtype][0], f"forward rel err {e}"


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
    # four pixels per store: rows of the grid in whole quads, boxes four wide, rows past the GEMM side
    (2, 1, 32, 70, [18, 20], [3, 3], False),
    (2, 2, 16, 19, [33, 4], [1, 1], False),
    (1, 40, 16, 260, [300], [1], False),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", FORWARD, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_forward_shares(case, dtype):
    dim, batch, cin, cout, size, kernel, transposed = case
    stride = 2 if transposed else 1
    check(make_case(dim, transposed, batch=batch, cin=cin, cout=cout, kernel=kernel, stride=[stride] * dim,
                    padding=[k // 2 for k in kernel], dilation=[1] * dim, out_pad=[0] * dim, in_size=size,
                    seed=40 + dim + batch), dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("case", [FORWARD[3] + (1,), PASSES_IN_TURN[1] + (True, 1), PASSES_IN_TURN[2] + (True, 1)],
                         ids=["shares", "two_passes", "three_passes"])
def test_captured_graph(case, dtype):
    """A forward and backward of several shares, and of passes in turn, captured on a stream of its own and replayed on
    rewritten inputs with eager calls on the default stream in between: each replay gives the eager result. Float
    atomics add the same terms in another order; bfloat16 outputs then round to neighbours (2^-8) now and then."""
    dim, batch, cin, cout, size, kernel, transposed, padding = case
    c = make_case(dim, transposed, batch=batch, cin=cin, cout=cout, kernel=kernel, stride=[1] * dim,
                  padding=[padding] * dim, dilation=[1] * dim, out_pad=[0] * dim, in_size=size, seed=95)
    op = tvdcn.deform_conv_transpose2d if transposed else tvdcn.deform_conv2d
    names = ("input", "weight", "offset", "mask", "bias")
    ts = [c[n].to("cuda:0", dtype).requires_grad_(True) for n in names]
    gy = torch.rand(c["out_shape"], device="cuda:0").to(dtype)

    def run():
        y = op(*ts, stride=1, padding=padding)
        return (y,) + torch.autograd.grad(y, ts, gy)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            run()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        outs = run()
    g = torch.Generator(device="cuda:0").manual_seed(96)
    for rep in range(3):
        with torch.no_grad():
            for t in ts:
                t.copy_(torch.randn(t.shape, device="cuda:0", generator=g))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, a, r in zip(("output",) + names, outs, run()):
            e = rel_err(a.detach(), r.detach())
            assert e < (1e-5 if dtype == torch.float32 else 2.0 ** -8), f"replay {rep}: {name} {e}"


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


# the 16-bit types' layouts: rows in eights, in fours and odd, channels past a 64-wide copy tile, rows and
# positions past their tiles, batches, both directions
HALF_LAYOUTS = [(1, [64], False), (1, [68], False), (1, [67], False), (2, [9, 24], False), (2, [7, 12], True),
                (3, [3, 4, 8], False), (1, [130], True)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", HALF_LAYOUTS, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_half_layouts(case, dtype):
    dim, size, transposed = case
    check(make_case(dim, transposed, batch=3, cin=68, cout=72, kernel=[3] * dim, stride=[1 + transposed] * dim,
                    padding=[1] * dim, dilation=[1] * dim, out_pad=[0] * dim, in_size=size, seed=90 + dim), dtype)


# float32: the bias gradient beside the channels-last copy where that has a block for every other channel
# (rows in whole quads and not, channels past the blocks, both directions), else a launch of its own
BIAS = [(1, 144, 24, [304], False), (1, 144, 29, [301], False), (1, 144, 32, [301], False), (2, 68, 20, [16, 24], False),
        (1, 32, 16, [300], True), (1, 32, 24, [300], True), (1, 16, 20, [4097], False), (1, 16, 20, [8191], False)]


@pytest.mark.parametrize("case", BIAS, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_bias_gradient_launch(case):
    dim, cin, cout, size, transposed = case
    check(make_case(dim, transposed, batch=3, cin=cin, cout=cout, kernel=[3] * dim, stride=[1 + transposed] * dim,
                    padding=[1] * dim, dilation=[1] * dim, out_pad=[0] * dim, in_size=size, seed=95 + dim), torch.float32)


# few sampled-side channels: column lengths (channels x taps) around the 16 and 64 blocks and at the rule's
# ends, GEMM sides around 16 and 64, pixels around the 64 of a tile, more tiles than workgroups, offset and
# mask groups that do not nest, conv groups, no offset / mask / bias
FEW = [
    # dim, transposed, make_case arguments
    (1, False, dict(batch=1, cin=1, cout=1, kernel=[1], in_size=[1])),
    (1, False, dict(batch=3, cin=2, cout=17, kernel=[8], in_size=[26])),                       # 16 values, 63 pixels
    (2, False, dict(batch=2, cin=3, cout=65, kernel=[3, 3], in_size=[4, 8])),                  # 27, 64 pixels
    (2, False, dict(batch=5, cin=13, cout=16, kernel=[5, 1], in_size=[3, 9])),                # 65, 55 pixels
    (2, False, dict(batch=1, cin=6, cout=10, kernel=[3, 3], in_size=[9, 9], og=2, mg=3, groups=2)),
    (2, False, dict(batch=2, cin=6, cout=6, kernel=[2, 2], in_size=[5, 13], og=3, mg=1, groups=6, bias=False)),
    (2, False, dict(batch=9, cin=14, cout=5, kernel=[3, 3], in_size=[45, 44])),                # 126, two tiles a workgroup
    (3, False, dict(batch=1, cin=5, cout=9, kernel=[3, 3, 4], in_size=[5, 6, 7])),             # 180
    (2, False, dict(batch=2, cin=3, cout=4, kernel=[3, 3], in_size=[7, 7], deformable=False)),
    (2, False, dict(batch=2, cin=3, cout=4, kernel=[3, 3], in_size=[7, 7], modulated=False)),
    (1, False, dict(batch=2, cin=3, cout=4, kernel=[3], in_size=[7], deformable=False, modulated=False)),
    (2, True, dict(batch=2, cin=66, cout=3, kernel=[4, 4], in_size=[5, 7])),
    (3, True, dict(batch=1, cin=6, cout=2, kernel=[2, 3, 2], in_size=[3, 4, 5], groups=2, og=2, bias=False)),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16],
                         ids=["f32", "f64", "f16", "bf16"])
@pytest.mark.parametrize("i", range(len(FEW)))
def test_few_channels(i, dtype):
    dim, transposed, kw = FEW[i]
    stride = 2 if transposed else 1
    check(make_case(dim, transposed, stride=[stride] * dim, padding=[1] * dim, dilation=[1] * dim, out_pad=[0] * dim,
                    seed=60 + i, **kw), dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_few_channels_last(dtype):
    """A channels-last input gives the contiguous input's results (the same operations: only the order of the
    scatter's float atomics differs) and a channels-last gradient."""
    case = make_case(2, batch=2, cin=5, cout=7, kernel=[3, 3], stride=[1, 1], padding=[1, 1], dilation=[1, 1],
                     in_size=[9, 11], seed=80)
    outs = []
    for fmt in (torch.contiguous_format, torch.channels_last):
        ts = [case[n].to("cuda", dtype) for n in ("input", "weight", "offset", "mask", "bias")]
        ts[0] = ts[0].contiguous(memory_format=fmt)
        ts = [t.requires_grad_(True) for t in ts]
        y = tvdcn.deform_conv2d(*ts, padding=1)
        outs.append((y,) + torch.autograd.grad(y.float().square().sum(), ts))
    assert outs[1][1].is_contiguous(memory_format=torch.channels_last)
    for a, b in zip(*outs):
        assert rel_err(a, b) < (1e-6 if dtype == torch.float32 else 1e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_data_gradient_in_several_launches(dtype):
    """60000 images of 2 x 2 x 2 pixels in 24 groups, three passes of taps each: 4.32M workgroups of 1024 threads, more
    than one launch takes. An image's gradients are those of a call on it alone: the first and the last ones, and
    those on both sides of the second launch's first workgroup (72 an image)."""
    batch, c, groups = 60000, 96, 24
    g = torch.Generator(device="cuda").manual_seed(101)
    rand = lambda *shape: torch.rand(*shape, generator=g, device="cuda").to(dtype)
    x, w = rand(batch, c, 2, 2, 2), rand(c, c // groups, 3, 3, 3)
    off, msk, gy = rand(batch, 81, 2, 2, 2), rand(batch, 27, 2, 2, 2), rand(batch, c, 2, 2, 2)
    off = off * 4 - 2
    backward = lambda s: torch.ops.tvdcn._deform_conv3d_backward(gy[s], x[s], w, off[s], msk[s], rand(c), [1] * 3, [1] * 3,
                                                                 [1] * 3, groups)
    full = backward(slice(None))
    at = ((2 ** 32 - 1) // 1024 // 8 * 8) // 72
    for lo in (0, at - 2, batch - 4):
        part = backward(slice(lo, lo + 4))
        for name, a, b in zip(("input", "offset", "mask"), (full[0], full[2], full[3]), (part[0], part[2], part[3])):
            # (sums of at most 27 x 4 terms per value, in another order where atomics add them)
            assert rel_err(a[lo:lo + 4], b) < (1e-5 if dtype == torch.float32 else 1e-2), (lo, name)


def test_few_channels_bias_gradient_of_equal_values():
    """The bias gradient of few channels over 100352 equal values a channel, which leave the roundings of a chain of
    additions on one side: 6 levels of a tree over 64 lanes, 7 tiles' sums a workgroup, 7 + 2 + 3 additions of 224
    workgroups' sums. At most 25 roundings of 2^-24 of the sum so far."""
    values = torch.linspace(0.1, 1.3, 24, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(102)
    rand = lambda *shape: torch.rand(*shape, generator=g, device="cuda")
    gy = values.reshape(1, 24, 1, 1).expand(8, 24, 112, 112).contiguous()
    gb = torch.ops.tvdcn._deform_conv2d_backward(gy, rand(8, 3, 112, 112), rand(24, 3, 1, 1), rand(8, 2, 112, 112),
                                                 rand(8, 1, 112, 112), rand(24), [1, 1], [0, 0], [1, 1], 1)[4]
    exact = values.double() * 8 * 112 * 112
    assert float(((gb.double() - exact) / exact).abs().max()) < 25 * 2.0 ** -24


@pytest.mark.parametrize("dim,batch,cin,size,kernel", [
    (1, 3, 48, [300], 3), (2, 3, 32, [20, 24], 3), (2, 17, 160, [64, 64], 3), (3, 2, 16, [4, 5, 6], 1),
    (3, 3, 32, [8, 16, 16], 3)], ids=lambda v: str(v).replace(" ", ""))
def test_forward_loops(dim, batch, cin, size, kernel):
    """One sampled value of the first image too large for the scaled 16-bit pieces sends the launch to the float32 loop,
    in the same kernel or one of its own: the other images' results are those of the 16-bit loop, both within the
    parity tests' float32 bound of the exact ones."""
    case = make_case(dim, batch=batch, cin=cin, cout=20, kernel=[kernel] * dim, stride=[1] * dim,
                     padding=[kernel // 2] * dim, dilation=[1] * dim, in_size=size, seed=110 + dim + batch)
    x, w, off, msk, b = (case[n].to("cuda", torch.float32) for n in ("input", "weight", "offset", "mask", "bias"))
    op = getattr(tvdcn, f"deform_conv{dim}d")
    y = op(x, w, off, msk, b, padding=kernel // 2)
    x[0].view(-1)[0] = 2.0 ** 127
    assert rel_err(op(x, w, off, msk, b, padding=kernel // 2)[1:], y[1:]) < 2e-5
