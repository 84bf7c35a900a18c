"""The few-channel kernels (few_channels.hip) on what other layers' tests reach only with many channels: values that are
not finite, mask activations applied in the mask load, a captured graph and a stream of its own."""
import pytest
import torch

import tvdcn
from tvdcn.ops.deform_conv import _deform_conv_mask_activation
from helpers import make_case, rel_err
from test_gpu_mask_fusion import _oracle_activated
from test_gpu_parity import TOL, run_gpu, run_oracle

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
NAMES = ("input", "weight", "offset", "mask", "bias")


def few_case(dim, transposed, seed, **kw):
    channels = dict(cin=12, cout=2) if transposed else dict(cin=3, cout=20)
    return make_case(dim, transposed, batch=2, kernel=[3] * dim, stride=[1 + transposed] * dim, padding=[1] * dim,
                     dilation=[1] * dim, out_pad=[0] * dim, in_size={1: [70], 2: [9, 11], 3: [4, 5, 6]}[dim], seed=seed,
                     **{**channels, **kw})


@pytest.mark.parametrize("where", ["input", "weight", "mask"])
@pytest.mark.parametrize("dim,transposed", [(1, False), (2, False), (3, False), (1, True), (2, True)])
def test_nonfinite_values(dim, transposed, where):
    """An inf in one operand: inf and nan where the oracle has them, everywhere else the parity tests' bounds."""
    case = few_case(dim, transposed, 1300 + dim)
    t = case[where].clone()
    t.view(-1)[t.numel() // 2] = float("inf")
    case[where] = t
    gout = torch.rand(case["out_shape"], generator=torch.Generator().manual_seed(1), dtype=torch.float64)
    out, grads, _ = run_gpu(case, torch.float32, grad_out=gout)
    ref_out, ref_grads = run_oracle(case, gout, torch.float32)
    for name, a, r in zip(("output",) + NAMES, [out] + list(grads), [ref_out] + list(ref_grads)):
        a = a.detach().double().cpu()
        assert torch.equal(torch.isnan(a), torch.isnan(r)), f"{name}: nan pattern differs"
        assert torch.equal(torch.isinf(a), torch.isinf(r)), f"{name}: inf pattern differs"
        fin = torch.isfinite(r)
        if fin.any():
            assert rel_err(a[fin], r[fin]) < TOL[torch.float32][1], name


@pytest.mark.parametrize("activation", [1, 2], ids=["sigmoid", "softmax"])
@pytest.mark.parametrize("dim,transposed,dtype", [
    (1, False, torch.float32), (2, False, torch.float32), (3, False, torch.float32), (2, True, torch.float32),
    (2, False, torch.float64), (2, False, torch.float16), (2, True, torch.bfloat16)])
def test_fused_mask_activation(dim, transposed, dtype, activation):
    """The mask given as logits (fp16 / bf16, whose logit gradient is finished in float32: the general kernels)."""
    case = few_case(dim, transposed, 1310 + dim)
    g = torch.Generator().manual_seed(1311)
    logits = torch.randn(case["mask"].shape, generator=g, dtype=torch.float64) * 2.0
    vals = [(case[n] if n != "mask" else logits).to(dtype) for n in NAMES]
    ts = [v.to(DEV).requires_grad_(True) for v in vals]
    y = _deform_conv_mask_activation(*ts, case["stride"], case["padding"], [0] * dim, case["dilation"], 1, transposed,
                                     activation, 2.0)
    gout = torch.randn(y.shape, generator=g, dtype=torch.float64).to(dtype)
    y.backward(gout.to(DEV))
    y_ref, leaves = _oracle_activated(case, dim, transposed, vals, activation, 2.0)
    y_ref.backward(gout.double())
    tf, tb = TOL[dtype]
    assert rel_err(y, y_ref) < tf
    for n, a, r in zip(NAMES, ts, leaves):
        assert rel_err(a.grad, r.grad) < tb, n


@pytest.mark.parametrize("transposed", [False, True])
def test_captured_graph_and_stream(transposed):
    """A forward and backward captured on a stream of its own, replayed on rewritten inputs with eager calls on the
    default stream in between: each replay gives the eager result."""
    case = few_case(2, transposed, 1320)
    op = tvdcn.deform_conv_transpose2d if transposed else tvdcn.deform_conv2d
    ts = [case[n].to(DEV, torch.float32).requires_grad_(True) for n in NAMES]
    gy = torch.rand(case["out_shape"], device=DEV)

    def run():
        y = op(*ts, stride=1 + transposed, padding=1)
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
    g = torch.Generator(device=DEV).manual_seed(1321)
    for rep in range(3):
        with torch.no_grad():
            for t in ts:
                t.copy_(torch.randn(t.shape, device=DEV, generator=g))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, a, r in zip(("output",) + NAMES, outs, run()):
            # (sums of the same terms, in another order where atomics add them)
            assert rel_err(a, r) < 1e-5, f"replay {rep}: {name}"
