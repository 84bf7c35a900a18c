"""The calls that the performance of this package is judged by.

Every case is one deformable convolution layer, called through the functional API as a program
calls it: the forward under ``no_grad`` for inference, the forward and all gradients for training.
Sizes of the named workloads are those of ``bench.py`` and the tests; the others are generic.
"""
import math

import torch

import tvdcn

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _case(name, dim, batch, cin, cout, size, kernel, **kw):
    """A layer: `size` (input) is written as in "64x64"; kernel, stride, padding and dilation hold for every axis."""
    case = dict(name=name, dim=dim, transposed=False, train=True, dtype="f32", batch=batch, cin=cin, cout=cout,
                size=size, kernel=kernel, stride=1, padding=(kernel - 1) // 2, dilation=1, groups=1, og=1, mg=1,
                softmax=False, channels_last=False, sigma=2.0)
    case.update(kw)
    return case


def listed():
    return [
        # the smallest call of the tests: three image channels, a 10 x 10 grid. Launches and host time.
        _case("conv2d_tiny_infer", 2, 4, 3, 5, "10x10", 3, train=False, padding=0, sigma=1.0),
        # the same layer trained: what a unit test, a toy model or a gradient check does all day
        _case("conv2d_tiny_train", 2, 4, 3, 5, "10x10", 3, padding=0, sigma=1.0),
        # one image through a layer at a coarse level of a feature pyramid: latency of a served model
        _case("conv2d_image_infer_f16", 2, 1, 256, 256, "25x38", 3, train=False, dtype="f16"),
        # a fine level of the same: two images, few channels, many pixels
        _case("conv2d_level_infer_bf16", 2, 2, 128, 128, "100x152", 3, train=False, dtype="bf16"),
        # the backbone layer of bench.py's metric line
        _case("conv2d_layer_train", 2, 8, 256, 256, "64x64", 3),
        # the same layer in a channels-last bfloat16 model
        _case("conv2d_layer_train_bf16", 2, 8, 256, 256, "64x64", 3, dtype="bf16", channels_last=True),
        # a grouped, strided layer whose channels and grid divide by nothing useful
        _case("conv2d_ragged_train", 2, 3, 72, 100, "61x47", 3, stride=2, groups=2, og=2, mg=2),
        # a short half-precision sequence layer
        _case("conv1d_short_train_f16", 1, 8, 128, 128, "1000", 7, dtype="f16", sigma=3.0),
        # the long sequence layer of bench.py's suite, its mask a softmax over the taps: the largest
        _case("conv1d_layer_train", 1, 16, 512, 512, "4096", 5, og=4, mg=4, softmax=True, sigma=3.0),
        # one small volume, served
        _case("conv3d_volume_infer_f16", 3, 1, 32, 32, "9x28x30", 3, train=False, dtype="f16", sigma=1.5),
        # the video layer of bench.py's suite
        _case("conv3d_layer_train", 3, 2, 64, 64, "16x56x56", 3, sigma=1.5),
        # the upsampling layer of bench.py's suite, in half precision, its mask a softmax over the taps
        _case("conv_transpose2d_train_f16", 2, 8, 256, 128, "32x32", 4, transposed=True, stride=2, padding=1, og=2,
              mg=2, softmax=True, dtype="f16", sigma=1.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A layer of the same kinds: any rank and direction, inference or training, every dtype, 1 to 512
    channels, 1 to 16 images and grids from a few pixels to the listed ones, odd sizes included."""
    while True:
        dim = rng.choice((1, 2, 2, 2, 3))
        transposed = rng.random() < 0.2
        if rng.random() < 0.15:
            # a first or last layer: channel counts of images and labels
            groups, og = 1, 1
            cin, cout = rng.randint(1, 9), rng.randint(1, 24)
        else:
            # channel counts in multiples of 4, the offset / mask groups in whole quads
            groups = rng.choice((1, 1, 1, 2))
            og = rng.choice((1, 1, 2, 4))
            unit = 4 * max(groups, og)
            cin = unit * _log_int(rng, max(1, 16 // unit), {1: 512, 2: 320, 3: 96}[dim] // unit)
            cout = unit * _log_int(rng, max(1, 16 // unit), {1: 512, 2: 320, 3: 96}[dim] // unit)
        kernel = rng.choice({1: (3, 5, 7), 2: (1, 3, 3, 3, 5), 3: (1, 3, 3)}[dim])
        if transposed:
            kernel = rng.choice((2, 3, 4))
        lo, hi = {1: (16, 4096), 2: (5, 120), 3: (3, 32)}[dim]
        if transposed and dim > 1:
            hi //= 2
        size = [_log_int(rng, lo, hi) for _ in range(dim)]
        case = _case("", dim, _log_int(rng, 1, 16), cin, cout, "x".join(str(s) for s in size), kernel,
                     transposed=transposed, train=rng.random() < 0.6, dtype=rng.choice(("f32", "f32", "f16", "bf16")),
                     stride=2 if transposed else rng.choice((1, 1, 1, 2)), groups=groups, og=og, mg=og,
                     softmax=rng.random() < 0.3, channels_last=not transposed and dim > 1 and rng.random() < 0.2,
                     sigma=rng.choice((0.5, 1.0, 2.0, 3.0)))
        del case["name"]
        if transposed:
            case["padding"] = 1 if kernel > 2 else 0
        # no more than the largest listed layer: by its contraction, and by its sampled values (the cost of
        # layers of few output channels), eight corners each in three dimensions
        col, k = _column_pixels(case), kernel ** dim
        flops = 2.0 * case["batch"] * col * cin * cout // groups * k
        samples = float(case["batch"]) * col * (cout if transposed else cin) * k * 2 ** dim
        quads = cin % 4 == 0 and cout % 4 == 0
        if flops <= 5e10 and samples <= (1e9 if quads else 5e7) and min(_out_size(case)) > 0:
            return case


def _in_size(case):
    return [int(s) for s in case["size"].split("x")]


def _out_size(case):
    k, s, p, d = case["kernel"], case["stride"], case["padding"], case["dilation"]
    if case["transposed"]:
        return [(n - 1) * s - 2 * p + d * (k - 1) + 1 for n in _in_size(case)]
    return [(n + 2 * p - d * (k - 1) - 1) // s + 1 for n in _in_size(case)]


def _grid(case):
    """the grid of the offsets and masks"""
    return _in_size(case) if case["transposed"] else _out_size(case)


def _column_pixels(case):
    return math.prod(_grid(case))


def _op(case):
    return getattr(tvdcn, f"deform_conv{'_transpose' if case['transposed'] else ''}{case['dim']}d")


def _draw_inputs(case, seed):
    """input, weight, offset, mask (or its logits), bias and the upstream gradient"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    dim, k, groups = case["dim"], case["kernel"], case["groups"]
    taps, grid = k ** dim, _grid(case)

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * scale

    x = normal(case["batch"], case["cin"], *_in_size(case))
    if case["transposed"]:
        wshape = (case["cin"], case["cout"] // groups) + (k,) * dim
    else:
        wshape = (case["cout"], case["cin"] // groups) + (k,) * dim
    fan = case["cin"] // groups * taps
    w = normal(*wshape, scale=(2.0 / fan) ** 0.5)
    o = normal(case["batch"], case["og"] * taps * dim, *grid, scale=case["sigma"])
    m = normal(case["batch"], case["mg"] * taps, *grid)
    if not case["softmax"]:
        m = torch.sigmoid(m)
    b = normal(case["cout"], scale=0.1)
    gout = normal(case["batch"], case["cout"], *_out_size(case))
    x, w, o, m, b, gout = (t.to(dtype) for t in (x, w, o, m, b, gout))
    if case["channels_last"]:
        x = x.contiguous(memory_format=torch.channels_last if dim == 2 else torch.channels_last_3d)
    return x, w, o, m, b, gout


def prepare(case, seed):
    x, w, o, m, b, gout = _draw_inputs(case, seed)
    params = [x, w, o, m, b]
    if case["train"]:
        params = [p.requires_grad_(True) for p in params]
    kwargs = dict(stride=case["stride"], padding=case["padding"], dilation=case["dilation"], groups=case["groups"])
    softmax = getattr(tvdcn, f"mask_softmax{case['dim']}d") if case["softmax"] else None
    return dict(op=_op(case), softmax=softmax, kernel_size=(case["kernel"],) * case["dim"], params=params,
                kwargs=kwargs, gout=gout, train=case["train"])


def _layer(state):
    x, w, o, m, b = state["params"]
    if state["softmax"] is not None:
        m = state["softmax"](m, state["kernel_size"])
    return state["op"](x, w, o, m, b, **state["kwargs"])


def run(state):
    if not state["train"]:
        with torch.no_grad():
            return _layer(state)
    out = _layer(state)
    return (out,) + torch.autograd.grad(out, state["params"], state["gout"])


def work(case):
    taps, col = case["kernel"] ** case["dim"], _column_pixels(case)
    x = case["batch"] * case["cin"] * math.prod(_in_size(case))
    y = case["batch"] * case["cout"] * math.prod(_out_size(case))
    w = case["cin"] * case["cout"] // case["groups"] * taps
    om = case["batch"] * (case["og"] * case["dim"] + case["mg"]) * taps * col
    flops = 2.0 * case["batch"] * col * w
    inputs = x + w + om + case["cout"]
    if case["train"]:
        # forward, then the gradients of its five operands from the upstream gradient
        elems, flops = 2 * inputs + 2 * y, 3 * flops
    else:
        elems = inputs + y
    return {"bytes": elems * torch.finfo(_DTYPES[case["dtype"]]).bits // 8, "flops": flops}


def tolerance(case):
    # about four times the largest error against `exact` over the listed and some drawn layers: float32
    # forwards 7e-7 (their sums); float32 training 3.3e-6 in one and two dimensions and 1.6e-5 in three
    # (the input's gradient, summed in fixed point); float16 3.6e-4 and bfloat16 2.9e-3 (the rounding of
    # the sampled columns and of the results)
    if case["dtype"] == "f32":
        return {"rel": 4e-6 if not case["train"] else 6.5e-5 if case["dim"] == 3 else 1.3e-5}
    return {"rel": 1.5e-3 if case["dtype"] == "f16" else 1.2e-2}


def _image(case, x, w, pos, m, b, in_size, out_size):
    """One image in float64: x (Cin, *in), pos (og, taps, dim, col), m (mg, taps, col) -> (Cout, out)."""
    dim, tr, groups = case["dim"], case["transposed"], case["groups"]
    taps, col = case["kernel"] ** dim, pos.shape[-1]
    og, mg = case["og"], case["mg"]
    side = out_size if tr else in_size   # the sampled grid
    C = case["cout"] if tr else case["cin"]
    low = torch.floor(pos.detach())
    frac = pos - low
    corners = []
    for corner in range(2 ** dim):
        idx, weight, ok = 0, 1.0, True
        for a in range(dim):
            bit = corner >> a & 1
            at = low[:, :, a] + bit
            weight = weight * (frac[:, :, a] if bit else 1.0 - frac[:, :, a])
            ok = ok & (at >= 0) & (at < side[a])
            idx = idx * side[a] + at.clamp(0, side[a] - 1)
        corners.append((idx.long().reshape(og, 1, -1).expand(og, C // og, taps * col),
                        (weight * ok).reshape(og, 1, -1)))
    m = m.reshape(mg, 1, taps * col)
    if not tr:
        src = x.reshape(og, C // og, -1)
        cols = sum(src.gather(2, idx) * weight for idx, weight in corners)
        cols = (cols.reshape(mg, C // mg, -1) * m).reshape(groups, C // groups * taps, col)
        y = torch.matmul(w.reshape(groups, case["cout"] // groups, -1), cols).reshape(case["cout"], -1)
    else:
        wt = w.reshape(groups, case["cin"] // groups, -1).transpose(1, 2).contiguous()
        cols = torch.matmul(wt, x.reshape(groups, case["cin"] // groups, col))
        cols = (cols.reshape(mg, C // mg, -1) * m).reshape(og, C // og, -1)
        y = cols.new_zeros(og, C // og, math.prod(out_size))
        for idx, weight in corners:
            y = y.scatter_add(2, idx, cols * weight)
        y = y.reshape(case["cout"], -1)
    return y + b.reshape(-1, 1)


def exact(case, seed):
    """The layer in float64 torch operations. The sampling positions are those of the layer's own type
    (float32 for bfloat16): base + offset, rounded once, which decides the cell a sample falls in."""
    x, w, o, m, b, gout = _draw_inputs(case, seed)
    dim, taps = case["dim"], case["kernel"] ** case["dim"]
    grid, in_size, out_size = _grid(case), _in_size(case), _out_size(case)
    col, B = math.prod(grid), case["batch"]
    # base positions (taps, dim, col)
    tap = torch.cartesian_prod(*[torch.arange(case["kernel"], device="cuda")] * dim).reshape(taps, dim, 1)
    pix = torch.cartesian_prod(*[torch.arange(n, device="cuda") for n in grid]).reshape(col, dim).t().reshape(1, dim, col)
    base = (pix * case["stride"] - case["padding"] + tap * case["dilation"]).double()
    ptype = torch.float16 if case["dtype"] == "f16" else torch.float32
    pos = (base + o.double().reshape(B, case["og"], taps, dim, col)).to(ptype).double()
    logits = m.double().reshape(B, case["mg"], taps, col)
    w, b, x = w.double(), b.double(), x.double().contiguous()
    gout = gout.double().reshape(B, case["cout"], -1)
    y = torch.empty(B, case["cout"], math.prod(out_size), device="cuda", dtype=torch.float64)
    grads = [torch.empty_like(x), torch.zeros_like(w), torch.empty_like(pos), torch.empty_like(logits),
             torch.zeros_like(b)]
    for i in range(B):
        leaves = [x[i], w, pos[i], logits[i], b]
        with torch.set_grad_enabled(case["train"]):
            if case["train"]:
                leaves = [t.detach().clone().requires_grad_(True) for t in leaves]
            xi, wi, pi, mi, bi = leaves
            yi = _image(case, xi, wi, pi, mi.softmax(1) if case["softmax"] else mi, bi, in_size, out_size)
        y[i] = yi.detach()
        if case["train"]:
            gx, gw, gp, gm, gb = torch.autograd.grad(yi, leaves, gout[i])
            grads[0][i], grads[2][i], grads[3][i] = gx, gp, gm
            grads[1] += gw
            grads[4] += gb
    y = y.reshape(B, case["cout"], *out_size)
    if not case["train"]:
        return y
    grads[2], grads[3] = grads[2].reshape(o.shape), grads[3].reshape(m.shape)
    return (y, *grads)
