"""The matrix kernel of small projections (mi_gemm through ops.linear / ops.projections): forward products, input, weight and
bias gradients against float64 products of the same rounded operands."""

import os
import subprocess
import sys

import pytest
import torch

from scaling_amd import _lib, ops
from scaling_amd.nn import ParallelSwiGLUMLP
from tests.kernels import launched

pytestmark = pytest.mark.gpu
DEV = "cuda"
# unit roundoff: half an ulp over the smallest value of a binade, 2^-p for a significand of p bits (8, 11 and 24)
HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _close(name, got, ref, magnitude, k, dtype):
    """One rounding of the result (half an ulp of its value, or of the smallest normal number) and k fp32 additions, each off
    by at most 2^-24 of the running sum of magnitudes."""
    tiny = 2.0 ** -25 if dtype == torch.float16 else 2.0 ** -133
    bound = HALF_ULP[dtype] * ref.abs() + (k + 1) * 2.0 ** -24 * magnitude + tiny
    err = (got.double().cpu() - ref).abs()
    assert bool((err <= bound * 1.001).all()), f"{name}: {float((err / bound).max()):.2f} x the bound"


def _case(rows, ins, outs, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, ins, generator=g).to(dtype)
    ws = [(torch.randn(o, ins, generator=g) * 0.1).to(dtype) for o in outs]
    bs = [torch.randn(o, generator=g).to(dtype) if i != 1 else None for i, o in enumerate(outs)]
    dys = [torch.randn(rows, o, generator=g).to(dtype) for o in outs]
    return x, ws, bs, dys


# rows around the 32- and 64-row blocks, contractions of less than a step, of several prefetch rounds and with a remainder; the
# wide ones have a 64 x 64 block per compute unit (256) and take that tiling
@pytest.mark.parametrize("rows,ins,outs", [
    (1, 8, (8,)), (3, 264, (40, 8, 16)), (33, 72, (64, 24)), (65, 520, (136,)), (127, 256, (264, 64, 64)),
    (1030, 136, (1048,)), (520, 1032, (1096, 1032)),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_projections_and_their_gradients(rows, ins, outs, dtype):
    print(f"case gemm rows={rows} in={ins} out={outs} dtype={dtype}", flush=True)
    x, ws, bs, dys = _case(rows, ins, outs, dtype, rows + ins)
    xg = x.to(DEV).requires_grad_()
    wg = [w.to(DEV).requires_grad_() for w in ws]
    bg = [b.to(DEV).requires_grad_() if b is not None else None for b in bs]
    ys = ops.projections(xg, wg, bg)
    torch.autograd.backward(ys, [d.to(DEV) for d in dys])
    torch.cuda.synchronize()
    xd, wd, dyd = x.double(), [w.double() for w in ws], [d.double() for d in dys]
    for i in range(len(outs)):
        b = bs[i].double() if bs[i] is not None else torch.zeros(outs[i], dtype=torch.float64)
        _close(f"y{i}", ys[i].detach(), xd @ wd[i].t() + b, xd.abs() @ wd[i].abs().t() + b.abs(), ins, dtype)
        _close(f"dw{i}", wg[i].grad, dyd[i].t() @ xd, dyd[i].abs().t() @ xd.abs(), rows, dtype)
        if bs[i] is not None:
            _close(f"db{i}", bg[i].grad, dyd[i].sum(0), dyd[i].abs().sum(0), rows, dtype)
    _close("dx", xg.grad, sum(d @ w for d, w in zip(dyd, wd)), sum(d.abs() @ w.abs() for d, w in zip(dyd, wd)), sum(outs), dtype)


# 16 and 17 rows (the kernel of few rows, the matrix kernel or the library), contractions on both sides of 3072
@pytest.mark.parametrize("rows,ins,outs", [(16, 4096, (256,)), (9, 3068, (64, 128)), (9, 3072, (64, 128)), (17, 2552, (64, 128)), (17, 2560, (64, 128)), (17, 3064, (64, 128)), (17, 3072, (64, 128)), (40, 4096, (1024,)), (64, 8192, (512, 256, 256))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_outputs_are_the_same_with_and_without_gradients(rows, ins, outs, dtype):
    """A forward pass under no_grad that is recomputed with gradients (reentrant checkpointing) has the same bits."""
    x, ws, bs, dys = _case(rows, ins, outs, dtype, ins)
    xg, wg, bg = x.to(DEV).requires_grad_(), [w.to(DEV).requires_grad_() for w in ws], [None if b is None else b.to(DEV) for b in bs]
    res = dys[0].to(DEV)
    calls = (lambda i: ops.projections(xg, wg, bg, *i), lambda i: [ops.linear(xg, wg[0], bg[0], None, *i)], lambda i: [ops.linear(xg, wg[0], None, res, *i)])
    for inference in ((), (True,)):
        for call in calls:
            with torch.no_grad():
                want = call(inference)
            assert all(torch.equal(a, b) for a, b in zip(want, call(inference)))


@pytest.mark.parametrize("rows,ins,outs", [(16, 2048, (512,)), (17, 2552, (64, 128)), (17, 2560, (64, 128)), (32, 2816, (1024,)), (64, 2048, (2048, 512, 512)),
                                           (33, 3072, (256,))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_captured_products(rows, ins, outs, dtype):
    """Products of inference in a captured graph, on both sides of the line to the library: every replay on new inputs against float64, with
    eager work between the replays."""
    x, ws, bs, dys = _case(rows, ins, outs, dtype, ins)
    wg, bg = [w.to(DEV) for w in ws], [None if b is None else b.to(DEV) for b in bs]
    inputs = [x, x.flip(0), 2 * x.roll(1, 1)]
    xs, res = inputs[0].to(DEV), dys[0].to(DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(side):
        ops.projections(xs, wg, bg, True), ops.linear(xs, wg[0], None, res, True)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        ys = [*ops.projections(xs, wg, bg, True), ops.linear(xs, wg[0], None, res, True)]
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for new in inputs:
        xs.copy_(new.to(DEV))
        graph.replay()
        (xs.float() @ wg[0].float().t()).sum().item()
        for i, y in enumerate(ys):
            last = i == len(ws)
            w, b = (ws[0], None) if last else (ws[i], bs[i])
            want = new.double() @ w.double().t() + (0 if b is None else b.double())
            add = dys[0].double() if last else torch.zeros(())
            # the product is rounded, and with the residual the sum again
            err = (y.double().cpu() - want - add).norm()
            assert err <= 1.01 * eps * (want.norm() + (want + add).norm() * last) + 1e-6


def test_capture_after_one_call():
    """A first call outside the capture makes whatever the captured one needs, in a process that has used no library product."""
    code = """
import torch
from scaling_amd import ops
for k in (2048, 2816, 3064, 3072):
    x, w = torch.ones(17, k, device="cuda", dtype=torch.bfloat16), torch.full((64, k), 0.5, device="cuda", dtype=torch.bfloat16)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(side):
        ops.linear(x, w, None, None, True)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        y = ops.linear(x, w, None, None, True)
    for scale in (1.0, 2.0, 4.0):
        x.fill_(scale)
        graph.replay()
        assert bool((y == scale * k / 2).all()), (k, scale)
print("captured")
"""
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert run.returncode == 0 and "captured" in run.stdout, run.stderr[-2000:]


def test_reentrant_checkpoint_over_a_long_contraction():
    """The MLP of a layer whose second product contracts over 4096 features, 24 rows: loss and gradients of a plain step."""
    from torch.utils.checkpoint import checkpoint
    torch.manual_seed(3)
    mlp = ParallelSwiGLUMLP(io_features=1024, intermediate_feature_factor=4.0, bias=False, device=torch.device(DEV), dtype=torch.bfloat16)
    x = torch.randn(24, 1024, device=DEV).bfloat16()

    def step(forward):
        mlp.zero_grad(set_to_none=True)
        a = x.clone().requires_grad_()
        y = forward(a)
        y.float().pow(2).sum().backward()
        return [y.detach(), a.grad] + [p.grad for p in mlp.parameters()]
    assert all(torch.equal(a, b) for a, b in zip(step(mlp), step(lambda t: checkpoint(mlp, t, use_reentrant=True))))


def test_projection_that_does_not_reach_the_loss():
    """Only the used outputs contribute; frozen weights get no gradient; an odd width runs on the library product."""
    x, ws, bs, dys = _case(40, 64, (32, 48, 16), torch.float32, 5)
    xg, wg = x.to(DEV).requires_grad_(), [w.to(DEV) for w in ws]
    wg[2].requires_grad_()
    ys = ops.projections(xg, wg, [None, None, None])
    ys[2].backward(dys[2].to(DEV))
    assert wg[0].grad is None and wg[1].grad is None
    _close("dx", xg.grad, dys[2].double() @ ws[2].double(), dys[2].double().abs() @ ws[2].double().abs(), 16, torch.float32)
    _close("dw", wg[2].grad, dys[2].double().t() @ x.double(), dys[2].double().abs().t() @ x.double().abs(), 40, torch.float32)
    odd = torch.randn(7, 64)
    _close("odd", ops.linear(xg.detach(), odd.to(DEV)), x.double() @ odd.double().t(), x.double().abs() @ odd.double().abs().t(), 64, torch.float32)
    assert ops.linear(torch.empty(0, 64, device=DEV), wg[0]).shape == (0, 32)


@pytest.mark.parametrize("rows,ins,outs", [(24, 64, (32, 16)), (2048, 512, (2048, 256)), (2048, 516, (2044, 252))])   # small and large blocks, library products
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_what_no_gradient_reads_may_change_before_the_backward_pass(rows, ins, outs, dtype):
    """As with torch.nn.functional.linear: the input where no weight is trained, the weights where the input takes no gradient."""
    print(f"case gemm frozen rows={rows} dtype={dtype}", flush=True)
    x, ws, bs, dys = _case(rows, ins, outs, dtype, 17)
    own = any("gemm_kernel" in k or "wide_kernel" in k for k in launched(lambda: ops.linear(x.to(DEV), ws[0].to(DEV))))
    assert own == (rows < 2048 or dtype != torch.float32 and ins % 8 == 0)
    xd, wd, dyd = x.double(), [w.double() for w in ws], [d.double() for d in dys]
    for n in (1, 2):
        def forward(xg, wg, bg):
            return [ops.linear(xg, wg[0], bg)] if n == 1 else ops.projections(xg, wg[:n], [bg, None])

        def backward(ys):
            torch.autograd.backward(ys, [d.to(DEV) for d in dys[:n]])
        # frozen weights, a trained bias: the input is a temporary that is overwritten
        leaf, wg, bg = x.to(DEV).requires_grad_(), [w.to(DEV) for w in ws], bs[0].to(DEV).requires_grad_()
        xg = leaf * 1
        ys = forward(xg, wg, bg)
        xg.detach().zero_()
        backward(ys)
        # a library product per projection is rounded before the next is added
        slack = HALF_ULP[dtype] * (dyd[0] @ wd[0]).abs() if n == 2 else 0.0
        ref, mag = sum(d @ w for d, w in zip(dyd[:n], wd)), sum(d.abs() @ w.abs() for d, w in zip(dyd[:n], wd))
        err = (leaf.grad.double().cpu() - ref).abs()
        assert bool((err <= (HALF_ULP[dtype] * ref.abs() + slack + (sum(outs) + 1) * 2.0 ** -24 * mag + 2.0 ** -133) * 1.001).all()), float(err.max())
        _close("db", bg.grad, dyd[0].sum(0), dyd[0].abs().sum(0), rows, dtype)
        # an input without gradients: the weights are stepped between forward and backward
        wg = [w.to(DEV).requires_grad_() for w in ws]
        ys = forward(x.to(DEV), wg, None)
        with torch.no_grad():
            for w in wg:
                w.add_(1.0)
        backward(ys)
        for i in range(n):
            _close(f"dw{i}", wg[i].grad, dyd[i].t() @ xd, dyd[i].abs().t() @ xd.abs(), rows, dtype)


def test_operands_that_do_not_fit_are_the_librarys():
    """What torch.nn.functional.linear refuses is refused, what it broadcasts is broadcast: no kernel sees such an operand."""
    x, w, b = torch.randn(4, 64, device=DEV), torch.randn(32, 64, device=DEV), torch.randn(32, device=DEV)
    for args in ((x, w, b[:16]), (x, w, b.half()), (x, w, b.cpu()), (x, w.cpu(), b), (x, w[:, :32], b), (x, w.half(), b)):
        with pytest.raises(RuntimeError):
            ops.linear(*args)
    _close("broadcast bias", ops.linear(x, w, b[:1]), x.double().cpu() @ w.double().cpu().t() + b[0].double().cpu(),
           x.double().cpu().abs() @ w.double().cpu().abs().t() + b[0].abs().double().cpu(), 65, torch.float32)
    # strided bias, residual off the 16-byte boundary, residual of another shape
    ref = torch.nn.functional.linear(x.double(), w.double(), b[::2].double().repeat(2)).cpu()
    mag = x.double().cpu().abs() @ w.double().cpu().abs().t() + b.abs().max().double().cpu()
    _close("strided", ops.linear(x, w, torch.stack([b[::2].repeat(2), b], 1)[:, 0]), ref, mag, 65, torch.float32)
    res = torch.randn(4 * 32 + 1, device=DEV)[1:].view(4, 32)
    _close("residual", ops.linear(x, w, None, res), (x.double() @ w.double().t() + res.double()).cpu(), mag + res.abs().double().cpu(), 65, torch.float32)
    assert ops.linear(x, w, None, res[:1]).shape == (4, 32)


# a weight that the library takes and mi_gemm does not: strided rows, a transposed matrix, rows off the 16-byte boundary
WEIGHT_VIEWS = {
    "every second column": lambda w: torch.stack([w, torch.zeros_like(w)], 2)[..., 0],
    "transposed": lambda w: w.t().contiguous().t(),
    "off the boundary": lambda w: torch.cat([w.new_zeros(1), w.flatten()])[1:].view_as(w),
    "rows of an odd stride": lambda w: torch.cat([w, w.new_zeros(w.shape[0], 3)], 1)[:, :-3],
}


@pytest.mark.parametrize("view", list(WEIGHT_VIEWS))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gradients_with_weights_in_other_layouts(view, dtype):
    """Input, weight and bias gradients of one projection and of two that share their input (one of them in the other layout)."""
    print(f"case gemm weight view={view} dtype={dtype}", flush=True)
    x, ws, bs, dys = _case(24, 64, (32, 16), dtype, 11)
    wg = [WEIGHT_VIEWS[view](ws[0].to(DEV)).detach().requires_grad_(), ws[1].to(DEV).requires_grad_()]
    assert torch.equal(wg[0].detach().cpu(), ws[0])
    for n in (1, 2):
        xg, bg = x.to(DEV).requires_grad_(), bs[0].to(DEV).requires_grad_()
        for w in wg:
            w.grad = None
        ys = [ops.linear(xg, wg[0], bg)] if n == 1 else ops.projections(xg, wg, [bg, None])
        torch.autograd.backward(ys, [d.to(DEV) for d in dys[:n]])
        xd, wd, dyd = x.double(), [w.double() for w in ws[:n]], [d.double() for d in dys[:n]]
        dx, mag = sum(d @ w for d, w in zip(dyd, wd)), sum(d.abs() @ w.abs() for d, w in zip(dyd, wd))
        # a library product per projection: the first is rounded before the second is added
        slack = HALF_ULP[dtype] * (dyd[0] @ wd[0]).abs() if n == 2 else torch.zeros_like(dx)
        err = (xg.grad.double().cpu() - dx).abs()
        assert bool((err <= (HALF_ULP[dtype] * dx.abs() + slack + 49 * 2.0 ** -24 * mag + 2.0 ** -133) * 1.001).all()), (n, float(err.max()))
        for i in range(n):
            _close(f"dw{i}", wg[i].grad, dyd[i].t() @ xd, dyd[i].abs().t() @ xd.abs(), 24, dtype)
        _close("db", bg.grad, dyd[0].sum(0), dyd[0].abs().sum(0), 24, dtype)


@pytest.mark.parametrize("rows,ins,outs", [(6, 16, 8), (2048, 512, 2048)])      # matrix kernel, library product
def test_gradients_that_lie_on_top_of_each_other(rows, ins, outs):
    """An output summed over its rows (or altogether) sends back one row for all of them."""
    x, w, b = (torch.randn(*s, device=DEV, requires_grad=True) for s in ((rows, ins), (outs, ins), (outs,)))
    v = torch.randn(outs, device=DEV)
    for loss in (lambda y: (y.sum(0) * v).sum(), lambda y: y.sum()):
        got = torch.autograd.grad(loss(ops.linear(x, w, b)), (x, w, b))
        xd, wd, bd = (t.detach().double().requires_grad_() for t in (x, w, b))
        ref = torch.autograd.grad(loss(torch.nn.functional.linear(xd, wd, bd)), (xd, wd, bd))
        for name, g, r, mag in zip(("dx", "dw", "db"), got, ref, (v.abs().double() @ wd.abs() + wd.abs().sum(0), (v.abs().double()[:, None] + 1) * xd.abs().sum(0),
                                                                  rows * (v.abs().double() + 1))):
            _close(name, g, r.detach().cpu(), mag.detach().expand(r.shape).cpu(), max(rows, outs), torch.float32)


@pytest.mark.parametrize("rows,ins,outs", [(6, 16, 8), (2048, 512, 2048), (40, 20, 12)])   # matrix kernel, library products
@pytest.mark.parametrize("bias", [False, True])
def test_outputs_can_be_changed_in_place(rows, ins, outs, bias):
    x, w = torch.randn(2, rows // 2, ins, device=DEV, requires_grad=True), torch.randn(outs, ins, device=DEV, requires_grad=True)
    b = torch.randn(outs, device=DEV) if bias else None
    for call in (lambda: ops.linear(x, w, b), lambda: ops.projections(x, [w, w.detach()], [b, None])[0]):
        y, z = call(), call()
        y.mul_(2.0).relu_()
        for got, want in zip(torch.autograd.grad(y.sum(), (x, w)), torch.autograd.grad((2.0 * z).relu().sum(), (x, w))):
            assert torch.equal(got, want)


def test_transforms_see_a_library_product():
    """Second derivatives, torch.func and forward-mode AD go through a projection as they do through torch.nn.functional.linear."""
    x, w = torch.randn(5, 24, device=DEV, requires_grad=True), torch.randn(16, 24, device=DEV, requires_grad=True)
    f, ref = (lambda a, b: ops.linear(a, b).pow(3).sum()), (lambda a, b: torch.nn.functional.linear(a, b).pow(3).sum())

    def second(fn, a, b):
        ga, gb = torch.autograd.grad(fn(a, b), (a, b), create_graph=True)
        return torch.autograd.grad(ga.pow(2).sum() + gb.pow(2).sum(), (a, b))
    exact = second(ref, x.detach().double().requires_grad_(), w.detach().double().requires_grad_())
    for got, r in zip(second(f, x, w), exact):             # float32 sums of at most 24 terms in four nested products
        assert float((got.double() - r).norm() / r.norm()) < 4 * 24 * 2.0 ** -24
    t = torch.randn_like(x)
    for a, b in ((torch.func.jvp(lambda q: ops.linear(q, w), (x,), (t,))[1], t @ w.t()),
                 (torch.func.vmap(lambda q: ops.linear(q, w))(x), x @ w.t()),
                 (torch.func.grad(lambda q: f(q, w))(x), torch.func.grad(lambda q: ref(q, w))(x))):
        assert float((a - b).norm() / b.norm()) < 24 * 2.0 ** -23


@pytest.mark.parametrize("rows,ins,outs", [(5, 24, (16,)), (5, 24, (16, 8)), (600, 1024, (1536, 1024))])
def test_batched_gradients(rows, ins, outs):
    """torch.autograd.grad with is_grads_batched, and a dispatch mode around the backward pass, see library products."""
    from torch.utils.flop_counter import FlopCounterMode
    x, ws, bs, dys = _case(rows, ins, outs, torch.float32, 4)
    xg, wg, bg = x.to(DEV).requires_grad_(), [w.to(DEV).requires_grad_() for w in ws], bs[0].to(DEV).requires_grad_()
    inputs = (xg, *wg, bg)
    gs = [torch.stack([d, d.flip(0), 2 * d]).to(DEV) for d in dys]
    ys = ops.projections(xg, wg, [bg] + [None] * (len(ws) - 1))
    got = torch.autograd.grad(ys, inputs, gs, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        one = torch.autograd.grad(ys, inputs, [g[i] for g in gs], retain_graph=True)
        for a, b in zip(got, one):                         # float32 sums of at most `rows` or sum(outs) terms in another order
            assert a.shape == (3, *b.shape)
            assert float((a[i] - b).norm()) <= 2 * max(rows, sum(outs)) ** 0.5 * 2.0 ** -24 * float(b.norm()) * 8
    with FlopCounterMode(display=False) as counter:
        torch.autograd.grad(ys, inputs, [g[0] for g in gs])
    assert counter.get_total_flops() == sum(4 * rows * ins * o for o in outs)


# products over 3 GFLOP take blocks of 128 or 256: remainders in every direction, one segment and several problems, contractions that
# are split over the chip (512 x 8200 -> 520, 264 x 16392 -> 520) and that end inside a step, launches of whole rounds with the rest behind
# them, by rows (4097 x 520 -> 4104; weight gradient of 600 x 1040 -> 13320) and by columns (2047 x 520 -> 16904)
@pytest.mark.parametrize("rows,ins,outs", [
    (1031, 1032, (1544,)), (2049, 1096, (1048, 264)), (513, 8200, (520,)), (264, 16392, (520,)), (129, 3080, (4104, 1032, 1032)),
    (2050, 2056, (5640,)), (4097, 520, (4104,)), (2047, 520, (16904,)), (600, 1040, (13320,)),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_large_products_and_their_gradients(rows, ins, outs, dtype):
    print(f"case wide rows={rows} in={ins} out={outs} dtype={dtype}", flush=True)
    x, ws, bs, dys = (t.to(DEV) if torch.is_tensor(t) else [u if u is None else u.to(DEV) for u in t] for t in _case(rows, ins, outs, dtype, rows + ins))
    for t in [x, *ws, *(b for b in bs if b is not None)]:
        t.requires_grad_()
    ys = ops.projections(x, ws, bs)
    torch.autograd.backward(ys, dys)
    xd, wd, dyd = x.detach().double(), [w.detach().double() for w in ws], [d.double() for d in dys]
    close = lambda name, got, ref, magnitude, k: _close(name, got, ref.cpu(), magnitude.cpu(), k, dtype)
    for i in range(len(outs)):
        b = bs[i].detach().double() if bs[i] is not None else torch.zeros(outs[i], dtype=torch.float64, device=DEV)
        close(f"y{i}", ys[i].detach(), xd @ wd[i].t() + b, xd.abs() @ wd[i].abs().t() + b.abs(), ins)
        close(f"dw{i}", ws[i].grad, dyd[i].t() @ xd, dyd[i].abs().t() @ xd.abs(), rows)
        if bs[i] is not None:
            close(f"db{i}", bs[i].grad, dyd[i].sum(0), dyd[i].abs().sum(0), rows)
    close("dx", x.grad, sum(d @ w for d, w in zip(dyd, wd)), sum(d.abs() @ w.abs() for d, w in zip(dyd, wd)), sum(outs))


def test_large_product_with_residual_and_in_a_graph():
    """The residual is added to the rounded product; replays with eager work between them give the eager bits."""
    g = torch.Generator().manual_seed(3)
    x, w, res = (torch.randn(*s, generator=g).bfloat16().to(DEV) for s in ((1200, 2056), (1032, 2056), (1200, 1032)))
    with torch.no_grad():
        want = ops.linear(x, w, None, res)
        assert torch.equal(want, ops.linear(x, w) + res)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = ops.linear(x, w, None, res)
        for _ in range(3):
            y.zero_()
            graph.replay()
            (x.float() @ w.float().t()).sum().item()
            assert torch.equal(y, want)


@pytest.mark.parametrize("rows,ins,outs", [(2047, 520, 16904), (4097, 520, 4104)])
def test_bias_and_residual_of_a_product_in_two_launches(rows, ins, outs):
    g = torch.Generator().manual_seed(outs)
    x, w, b, res = (torch.randn(*s, generator=g).bfloat16().to(DEV) for s in ((rows, ins), (outs, ins), (outs,), (rows, outs)))
    with torch.no_grad():
        y = ops.linear(x, w, b)
        ref, magnitude = x.double() @ w.double().t() + b.double(), x.double().abs() @ w.double().abs().t() + b.double().abs()
        _close("y", y, ref.cpu(), magnitude.cpu(), ins, torch.bfloat16)
        assert torch.equal(ops.linear(x, w, b, res), y + res)


@pytest.mark.parametrize("rows,hidden,vocab", [(2047, 1024, 50257), (300, 520, 20003), (1025, 2048, 1000), (1025, 2048, 128)])   # the last: library
def test_lm_head_products(rows, hidden, vocab):
    """Loss and gradients of the chunked LM head over ragged vocabularies against float64."""
    g = torch.Generator(device=DEV).manual_seed(rows)
    h = torch.randn(rows, hidden, generator=g, device=DEV).bfloat16().requires_grad_()
    w = (torch.randn(vocab, hidden, generator=g, device=DEV) * 2 / hidden ** 0.5).bfloat16().requires_grad_()
    t = torch.randint(0, vocab, (rows,), generator=g, device=DEV)
    weights = torch.ones(rows, device=DEV)
    loss = ops.linear_cross_entropy(h, w, t, weights)[0]
    loss.backward()
    hd, wd = h.detach().double().requires_grad_(), w.detach().double().requires_grad_()
    ref = torch.nn.functional.cross_entropy(hd @ wd.t(), t)
    ref.backward()
    assert abs(loss.item() - ref.item()) <= 1e-3 * ref.item()
    # logits and their gradient are rounded to bfloat16 (2^-9 on average a half of 2^-8 each, over sums with independent errors)
    for name, a, b in (("dh", h.grad, hd.grad), ("dw", w.grad, wd.grad)):
        err = ((a.double() - b).norm() / b.norm()).item()
        assert err <= 2.0 ** -7, f"{name}: {err}"


@pytest.mark.parametrize("rows,ins,outs", [(512, 1024, 4101), (512, 4100, 1024)])
def test_ragged_extents_need_the_entry_with_a_workspace(rows, ins, outs):
    """mi_gemm takes whole vectors whatever the size of the product; the other entry takes any n of a large one, and no ragged contraction
    between operands that are both contiguous along it."""
    lib = _lib.load()
    g = torch.Generator(device=DEV).manual_seed(ins)
    x, w = (torch.randn(n, 4104, generator=g, device=DEV).bfloat16() for n in (rows, outs))
    c = torch.full((rows, 4104), 7.0, dtype=torch.bfloat16, device=DEV)
    p = _lib.MiGemmProblem(c=c.data_ptr(), ldc=4104, n_segments=1, m=rows, n=outs)
    p.segments[0] = _lib.MiGemmSegment(x.data_ptr(), w.data_ptr(), 4104, 4104, ins)
    assert lib.mi_gemm(p, 1, 0, ops.stream_ptr()) != 0
    assert (lib.mi_gemm_with_workspace(p, 1, 0, None, 0, ops.stream_ptr()) == 0) == (ins % 8 == 0)
    torch.cuda.synchronize()
    if ins % 8 == 0:
        xd, wd = x[:, :ins].double(), w[:, :ins].double()
        _close("c", c[:, :outs], (xd @ wd.t()).cpu(), (xd.abs() @ wd.abs().t()).cpu(), ins, torch.bfloat16)
    assert bool((c[:, outs if ins % 8 == 0 else 0:] == 7).all())


# results of whole and ragged rows: blocks of 128 and 256, one launch, two launches by rows and by columns, and contractions that are split;
# with bias and residual (a wider matrix, or the result itself), whatever lies behind a row of the result left as it is
@pytest.mark.parametrize("rows,ins,outs", [(513, 8200, 520), (264, 16392, 517), (512, 1032, 4101), (2050, 2056, 5633), (2047, 520, 16903), (4097, 520, 4101), (130, 4104, 4099)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_results_bias_and_residual_of_ragged_rows(rows, ins, outs, dtype):
    print(f"case wide epilogue rows={rows} in={ins} out={outs} dtype={dtype}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(outs)
    lib, code, ld = _lib.load(), ops.dtype_code(dtype), (outs + 15) // 8 * 8
    x, w, b, res = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((rows, ins), (outs, ins), (outs,), (rows, ld)))
    xd, wd = x.double(), w.double()
    ref, magnitude = xd @ wd.t() + b.double(), xd.abs() @ wd.abs().t() + b.double().abs()

    def run(c, add):
        p = _lib.MiGemmProblem(c=c.data_ptr(), ldc=ld, n_segments=1, m=rows, n=outs, bias=b.data_ptr(), add=None if add is None else add.data_ptr(), ldadd=ld)
        p.segments[0] = _lib.MiGemmSegment(x.data_ptr(), w.data_ptr(), ins, ins, ins)
        bytes_ = lib.mi_gemm_workspace_bytes(p, 1, code)
        ws = torch.full((max(bytes_, 16) // 4,), float("nan"), device=DEV)
        _lib.check(lib.mi_gemm_with_workspace(p, 1, code, ws.data_ptr(), bytes_, ops.stream_ptr()), "mi_gemm_with_workspace")
        return bytes_ > 0

    c, d, e = torch.full((rows, ld), 7.0, dtype=dtype, device=DEV), torch.full((rows, ld), 7.0, dtype=dtype, device=DEV), res.clone()
    split = [run(c, None), run(d, res), run(e, e)]
    assert split == [(rows, ins, outs) in ((513, 8200, 520), (264, 16392, 517), (130, 4104, 4099))] * 3
    _close("product", c[:, :outs], ref.cpu(), magnitude.cpu(), ins, dtype)
    assert torch.equal(d[:, :outs], c[:, :outs] + res[:, :outs]) and torch.equal(e[:, :outs], d[:, :outs])   # the rounded product, then the sum
    assert bool((c[:, outs:] == 7).all() and (d[:, outs:] == 7).all()) and torch.equal(e[:, outs:], res[:, outs:])



# contractions that end inside a 32-bit word and at either end of a vector, of an operand contiguous along them; rows at the end of a block
# (127, 255, 383 and the last), where nothing lies behind the row that may be read, take nearly all of their result from the last index
@pytest.mark.parametrize("k", [16385, 16387, 16391, 16390, 65, 16384 + 63])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_last_index_of_a_ragged_contraction(k, dtype):
    print(f"case ragged contraction k={k} dtype={dtype}", flush=True)
    rows, n = (389, 520) if k > 1000 else (12293, 2056)
    ld = (k + 7) // 8 * 8
    g = torch.Generator(device=DEV).manual_seed(k)
    p = torch.zeros(rows, ld, dtype=dtype, device=DEV)
    p[:, :k] = (torch.randn(rows, k, generator=g, device=DEV) * 2.0 ** -6).to(dtype)
    q = torch.randn(k, n, generator=g, device=DEV).to(dtype)
    ends = sorted({*range(127, rows, 128), rows - 1})
    p[ends, k - 1] = 8.0
    q[k - 1] = 4.0
    c = torch.full((rows, n), float("nan"), dtype=dtype, device=DEV)
    pr = _lib.MiGemmProblem(c=c.data_ptr(), ldc=n, n_segments=1, m=rows, n=n, q_kmajor=1)
    pr.segments[0] = _lib.MiGemmSegment(p.data_ptr(), q.data_ptr(), ld, n, k)
    lib, code = _lib.load(), ops.dtype_code(dtype)
    bytes_ = lib.mi_gemm_workspace_bytes(pr, 1, code)
    ws = torch.empty(max(bytes_, 16) // 4, device=DEV)
    _lib.check(lib.mi_gemm_with_workspace(pr, 1, code, ws.data_ptr(), bytes_, ops.stream_ptr()), "mi_gemm_with_workspace")
    pd, qd = p[:, :k].double(), q.double()
    _close("c", c, (pd @ qd).cpu(), (pd.abs() @ qd.abs()).cpu(), k, dtype)


def test_lm_head_rows_whose_target_is_the_last_entry():
    """dh over an odd vocabulary, row by row: where the target is the last entry, the last index of the contraction is half of the row."""
    rows, hidden, vocab = 519, 256, 20003
    g = torch.Generator(device=DEV).manual_seed(1)
    h = torch.randn(rows, hidden, generator=g, device=DEV).bfloat16().requires_grad_()
    w = (torch.randn(vocab, hidden, generator=g, device=DEV) * 2 / hidden ** 0.5).bfloat16().requires_grad_()
    t = torch.full((rows,), vocab - 1, device=DEV)
    ops.linear_cross_entropy(h, w, t, torch.ones(rows, device=DEV))[0].backward()
    hd, wd = h.detach().double().requires_grad_(), w.detach().double()
    torch.nn.functional.cross_entropy(hd @ wd.t(), t).backward()
    err = (h.grad.double() - hd.grad).norm(dim=1) / hd.grad.norm(dim=1)
    assert float(err.max()) <= 2.0 ** -6, (int(err.argmax()), float(err.max()))   # logits, their gradient and dh rounded to bfloat16


# both gradients of a projection where one of them is a long chain of few blocks: many tokens of a narrow layer (weight gradient; with the
# bias gradient beside a split), few tokens before a wide output (input gradient).  Each gets the plan that it has alone, splits included.
@pytest.mark.parametrize("rows,ins,outs,bias", [(32768, 256, 256, True), (20000, 264, 520, False), (257, 1024, 16384, True), (130, 776, 40960, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gradients_of_which_one_is_a_long_chain(rows, ins, outs, bias, dtype):
    print(f"case chain rows={rows} in={ins} out={outs} dtype={dtype}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(rows)
    x, w, dy = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((rows, ins), (outs, ins), (rows, outs)))
    lib, code = _lib.load(), ops.dtype_code(dtype)

    def problems(dx, dw, db):
        a = _lib.MiGemmProblem(c=dx.data_ptr(), ldc=ins, n_segments=1, m=rows, n=ins, q_kmajor=1)
        a.segments[0] = _lib.MiGemmSegment(dy.data_ptr(), w.data_ptr(), outs, ins, outs)
        b = _lib.MiGemmProblem(c=dw.data_ptr(), ldc=ins, n_segments=1, m=outs, n=ins, p_kmajor=1, q_kmajor=1, p_sum=db.data_ptr() if bias else None)
        b.segments[0] = _lib.MiGemmSegment(dy.data_ptr(), x.data_ptr(), outs, ins, rows)
        return (_lib.MiGemmProblem * 2)(a, b)

    def run(p, count):
        bytes_ = lib.mi_gemm_workspace_bytes(p, count, code)
        ws = torch.full((max(bytes_, 16) // 4,), float("nan"), device=DEV)
        _lib.check(lib.mi_gemm_with_workspace(p, count, code, ws.data_ptr(), bytes_, ops.stream_ptr()), "mi_gemm_with_workspace")
        torch.cuda.synchronize()
        return bytes_

    new = lambda: (torch.empty_like(x), torch.empty_like(w), torch.empty(outs, dtype=dtype, device=DEV))
    both, each = new(), new()
    need = run(problems(*both), 2)
    single = problems(*each)
    assert need == max(run(_lib.MiGemmProblem.from_buffer_copy(bytes(single[i])), 1) for i in range(2)) > 0
    xd, wd, dyd = x.double(), w.double(), dy.double()
    _close("dx", both[0], (dyd @ wd).cpu(), (dyd.abs() @ wd.abs()).cpu(), outs, dtype)
    _close("dw", both[1], (dyd.t() @ xd).cpu(), (dyd.abs().t() @ xd.abs()).cpu(), rows, dtype)
    assert torch.equal(both[0], each[0]) and torch.equal(both[1], each[1])
    if bias:
        _close("db", both[2], dyd.sum(0).cpu(), dyd.abs().sum(0).cpu(), rows, dtype)
        assert torch.equal(both[2], each[2])
    xg, wg = x.clone().requires_grad_(), w.clone().requires_grad_()
    bg = torch.zeros(outs, dtype=dtype, device=DEV, requires_grad=True) if bias else None
    ops.linear(xg, wg, bg).backward(dy)
    assert torch.equal(xg.grad, both[0]) and torch.equal(wg.grad, both[1]) and (not bias or torch.equal(bg.grad, both[2]))


def test_chain_alone_and_the_rest_in_one_launch():
    """1024 rows of two wide projections: the input gradient (one sum over both) in a launch of its own, both weight gradients in another."""
    rows, ins, outs = 1024, 4096, 14336
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(rows, ins, generator=g, device=DEV).bfloat16().requires_grad_()
    ws = [torch.randn(outs, ins, generator=g, device=DEV).bfloat16().requires_grad_() for _ in range(2)]
    dys = [torch.randn(rows, outs, generator=g, device=DEV).bfloat16() for _ in range(2)]
    ys = ops.projections(x, ws, [None, None])
    names = launched(lambda: torch.autograd.backward(ys, dys))
    assert sum("wide_kernel" in k for k in names) == 2, names
    rows_ = torch.tensor([0, 127, 128, 700, rows - 1], device=DEV)
    dyd, wd, xd = [d.double() for d in dys], [w.detach().double() for w in ws], x.detach().double()
    _close("dx", x.grad[rows_], sum(d[rows_] @ w for d, w in zip(dyd, wd)).cpu(), sum(d[rows_].abs() @ w.abs() for d, w in zip(dyd, wd)).cpu(), 2 * outs, torch.bfloat16)
    cols = torch.tensor([0, 255, 256, 9000, outs - 1], device=DEV)
    for w, d in zip(ws, dyd):
        a = d[:, cols].t().contiguous()
        _close("dw", w.grad[cols], (a @ xd).cpu(), (a.abs() @ xd.abs()).cpu(), rows, torch.bfloat16)


# short contractions into large outputs are the library's, each product by itself: forward (k = ins), input gradient (k = outs) and weight
# gradient (k = rows); one step more, a step that is not whole or a column block that is not, and the package's kernel takes it.  Of fewer than
# 32 features everything is the library's.
@pytest.mark.parametrize("rows,ins,outs,library", [
    (8192, 64, 8192, "y"), (8192, 8192, 64, "dx"), (320, 8192, 4096, "dw"), (8192, 96, 8192, "y"), (8192, 448, 4096, "y"), (8192, 512, 4096, ""),
    (8192, 72, 8192, ""), (8192, 64, 8200, ""), (8192, 24, 8192, "y dx dw"),
])
def test_short_contractions_into_large_outputs(rows, ins, outs, library):
    print(f"case thin rows={rows} in={ins} out={outs}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(ins)
    x, w, dy = (torch.randn(*s, generator=g, device=DEV).bfloat16() for s in ((rows, ins), (outs, ins), (rows, outs)))
    b = torch.randn(outs, generator=g, device=DEV).bfloat16().requires_grad_()
    xg, wg = x.clone().requires_grad_(), w.clone().requires_grad_()
    y = ops.linear(xg, wg)
    calls = {"y": lambda: ops.linear(xg, wg), **{n: lambda t=t: torch.autograd.grad(y, t, dy, retain_graph=True)[0] for n, t in (("dx", xg), ("dw", wg))}}
    ref = {"y": torch.mm(x, w.t()), "dx": torch.mm(dy, w), "dw": torch.mm(dy.t(), x)}
    eps = 2.0 ** -7                                        # two roundings of one sum
    for name, call in calls.items():
        got = call()
        assert float((got.float() - ref[name].float()).norm() / ref[name].float().norm()) < eps
        assert any("wide_kernel" in k for k in launched(call)) == (name not in library.split()), name
    ops.linear(xg, wg, b).backward(dy)                     # together, and with a bias, whose gradient goes with the weight's or by itself
    for name, t in (("dx", xg), ("dw", wg)):
        assert float((t.grad.float() - ref[name].float()).norm() / ref[name].float().norm()) < eps
    _close("db", b.grad, dy.double().sum(0).cpu(), dy.double().abs().sum(0).cpu(), rows, torch.bfloat16)


# inference: one round of 128 x 128 blocks, or short contractions, on the package's kernel; a second round beyond 512 contraction indices is the
# library's, by the average of projections that share their input
@pytest.mark.parametrize("rows,ins,outs,own", [
    (1078, 1024, (3072,), True), (1024, 1024, (4096,), True), (1025, 1024, (4096,), False), (1450, 520, (3072,), False), (1450, 512, (3072,), True),
    (1163, 1024, (4096, 256), True), (1163, 1024, (4096, 4096), False), (1000, 1544, (1024,), False),
])
def test_route_of_inference_products(rows, ins, outs, own):
    g = torch.Generator(device=DEV).manual_seed(rows)
    x = torch.randn(rows, ins, generator=g, device=DEV).bfloat16()
    ws = [torch.randn(o, ins, generator=g, device=DEV).bfloat16() for o in outs]
    with torch.no_grad():
        call = lambda: ops.projections(x, ws, [None] * len(ws), True)
        for y, w in zip(call(), ws):
            ref = x.double() @ w.double().t()
            assert float((y.double() - ref).norm() / ref.norm()) < 2.0 ** -8
        names = launched(call)
    assert any("wide_kernel" in k for k in names) == own and any("wide_kernel" not in k for k in names) != own, names


@pytest.mark.parametrize("rows,ins,outs,large", [(64, 14336, 4096, False), (96, 4096, 4096, False), (32, 8192, 8192, False), (16, 12288, 8192, False), (96, 8192, 8192, True),
                                                 (16, 4096, 32000, True), (64, 4096, 14336, True)])
def test_few_blocks_without_a_workspace(rows, ins, outs, large):
    """mi_gemm has nothing to split a long contraction with: few large blocks are left to the small ones; with a workspace they are split."""
    g = torch.Generator(device=DEV).manual_seed(rows)
    x, w = (torch.randn(n, ins, generator=g, device=DEV).bfloat16() for n in (rows, outs))
    c = torch.empty(rows, outs, dtype=torch.bfloat16, device=DEV)
    p = _lib.MiGemmProblem(c=c.data_ptr(), ldc=outs, n_segments=1, m=rows, n=outs)
    p.segments[0] = _lib.MiGemmSegment(x.data_ptr(), w.data_ptr(), ins, ins, ins)
    lib, ws = _lib.load(), torch.empty(1 << 26, device=DEV)
    ref, magnitude = (x.double() @ w.double().t()).cpu(), (x.double().abs() @ w.double().abs().t()).cpu()
    for call, wide in ((lambda: lib.mi_gemm(p, 1, 0, ops.stream_ptr()), large),
                       (lambda: lib.mi_gemm_with_workspace(p, 1, 0, ws.data_ptr(), 1 << 28, ops.stream_ptr()), True)):
        c.fill_(float("nan"))
        names = launched(lambda: _lib.check(call(), "mi_gemm"))
        assert any("wide_kernel" in k for k in names) == wide, names
        _close("c", c, ref, magnitude, ins, torch.bfloat16)


def test_lm_head_over_more_entries_than_large_blocks_reach():
    """2^22 + 1 entries (a row of logits is longer than the blocks address): the library's products, as for any operand they do not take."""
    rows, hidden, vocab = 128, 64, (1 << 22) + 1
    g = torch.Generator(device=DEV).manual_seed(1)
    h = torch.randn(rows, hidden, generator=g, device=DEV).bfloat16().requires_grad_()
    w = (torch.randn(vocab, hidden, generator=g, device=DEV) * 0.25).bfloat16().requires_grad_()
    t = torch.randint(0, vocab, (rows,), generator=g, device=DEV)
    loss = ops.linear_cross_entropy(h, w, t, torch.ones(rows, device=DEV))[0]
    loss.backward()
    hd, wd = h.detach().double().requires_grad_(), w.detach().double().requires_grad_()
    ref = torch.nn.functional.cross_entropy(hd @ wd.t(), t)
    ref.backward()
    assert abs(loss.item() - ref.item()) <= 1e-3 * ref.item()
    for name, a, b in (("dh", h.grad, hd.grad), ("dw", w.grad, wd.grad)):
        err = ((a.double() - b).norm() / b.norm()).item()
        assert err <= 2.0 ** -7, f"{name}: {err}"          # logits and their gradient are rounded to bfloat16


def test_projection_of_rows_that_lie_far_apart():
    """Rows 2^22 elements apart go to the library, forward and backward, at any size of the product that is not a small one."""
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.zeros(128, 1 << 22, dtype=torch.bfloat16, device=DEV)[:, :4096].copy_(torch.randn(128, 4096, generator=g, device=DEV))
    w = torch.randn(4096, 4096, generator=g, device=DEV).bfloat16().requires_grad_()
    dy = torch.randn(128, 4096, generator=g, device=DEV).bfloat16()
    out = []
    names = launched(lambda: out.append(ops.linear(x, w)) or out[0].backward(dy))
    assert not any("wide_kernel" in k or "gemm_kernel" in k for k in names), names
    xd, wd, dyd = x.double(), w.detach().double(), dy.double()
    _close("y", out[0].detach(), (xd @ wd.t()).cpu(), (xd.abs() @ wd.abs().t()).cpu(), 4096, torch.bfloat16)
    _close("dw", w.grad, (dyd.t() @ xd).cpu(), (dyd.abs().t() @ xd.abs()).cpu(), 128, torch.bfloat16)


def test_lm_head_with_a_weight_that_is_stored_transposed():
    """The library's products; the weight gradient of 107 GFLOP with the activations transposed first."""
    rows, hidden, vocab = 2048, 2048, 12800
    g = torch.Generator(device=DEV).manual_seed(1)
    h = torch.randn(rows, hidden, generator=g, device=DEV).bfloat16().requires_grad_()
    w = (torch.randn(hidden, vocab, generator=g, device=DEV) * 2 / hidden ** 0.5).bfloat16().t().requires_grad_()
    t = torch.randint(0, vocab, (rows,), generator=g, device=DEV)
    grads = []
    names = launched(lambda: grads.extend(torch.autograd.grad(ops.linear_cross_entropy(h, w, t, torch.ones(rows, device=DEV))[0], (h, w))))
    assert any("transpose_kernel" in k for k in names) and not any("wide_kernel" in k for k in names), names
    hd, wd = h.detach().double().requires_grad_(), w.detach().double().requires_grad_()
    ref = torch.autograd.grad(torch.nn.functional.cross_entropy(hd @ wd.t(), t), (hd, wd))
    for name, a, b in zip(("dh", "dw"), grads, ref):
        err = ((a.double() - b).norm() / b.norm()).item()
        assert err <= 2.0 ** -7, f"{name}: {err}"          # logits and their gradient are rounded to bfloat16


def test_gradients_with_workspaces_in_a_graph():
    """A split product of one projection and a chain with a launch of its own, captured: every replay, with eager work that reuses the allocator
    between them, gives the eager bits."""
    g = torch.Generator(device=DEV).manual_seed(1)
    x, w, dy = (torch.randn(*s, generator=g, device=DEV).bfloat16() for s in ((257, 1024), (16384, 1024), (257, 16384)))
    x.requires_grad_(), w.requires_grad_()
    step = lambda: torch.autograd.grad(ops.linear(x, w), (x, w), dy)
    want = step()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step()
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        assert all(torch.equal(a, b) for a, b in zip(step(), want))
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("rows,ins,outs", [(4097, 520, 4104), (2050, 2056, 5632), (512, 1032, 4104), (513, 8200, 520), (1030, 1544, 1028)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bias_off_the_boundaries_of_vectors(rows, ins, outs, dtype):
    """Blocks of 256 and 128 and split contractions: a bias that starts between words of eight bytes gives the bits of one that does not."""
    g = torch.Generator(device=DEV).manual_seed(rows)
    lib, code = _lib.load(), ops.dtype_code(dtype)
    ld = (outs + 7) // 8 * 8
    x, w, b = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((rows, ins), (outs, ins), (outs,)))
    results = []
    for shift in range(4):
        bias = torch.empty(outs + 4, dtype=dtype, device=DEV)[shift:shift + outs].copy_(b)
        c = torch.full((rows, ld), 7.0, dtype=dtype, device=DEV)
        p = _lib.MiGemmProblem(c=c.data_ptr(), ldc=ld, n_segments=1, m=rows, n=outs, bias=bias.data_ptr())
        p.segments[0] = _lib.MiGemmSegment(x.data_ptr(), w.data_ptr(), ins, ins, ins)
        bytes_ = lib.mi_gemm_workspace_bytes(p, 1, code)
        ws = torch.empty(max(bytes_, 16) // 4, device=DEV)
        names = launched(lambda: _lib.check(lib.mi_gemm_with_workspace(p, 1, code, ws.data_ptr(), bytes_, ops.stream_ptr()), "mi_gemm_with_workspace"))
        assert any("wide_kernel" in n for n in names), names
        results.append(c)
    xd, wd, bd = x.double(), w.double(), b.double()
    _close("c", results[0][:, :outs], (xd @ wd.t() + bd).cpu(), (xd.abs() @ wd.abs().t() + bd.abs()).cpu(), ins, dtype)
    assert all(torch.equal(c, results[0]) for c in results[1:]) and bool((results[0][:, outs:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_chains_shorter_than_the_stages_of_a_block(dtype):
    """Contractions of 1, 2, 3, 4 and 5 steps, in every layout, beside a long one in a launch of blocks of 128."""
    lib, code, g = _lib.load(), ops.dtype_code(dtype), torch.Generator(device=DEV).manual_seed(3)
    normal = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    for layout in range(3):                                # rows and rows; rows and contraction-major; contraction-major both
        ks, problems, results = (2048, 8, 72, 136, 200, 264), (_lib.MiGemmProblem * 6)(), []
        for i, k in enumerate(ks):
            m, n = (2048, 2048) if i == 0 else (136, 264)
            p, q = normal(m, k), normal(n, k)
            c = torch.full((m, n), float("nan"), dtype=dtype, device=DEV)
            pm, qm = p.t().contiguous() if layout == 2 else p, q.t().contiguous() if layout > 0 else q
            problems[i] = _lib.MiGemmProblem(c=c.data_ptr(), ldc=n, n_segments=1, m=m, n=n, p_kmajor=int(layout == 2), q_kmajor=int(layout > 0))
            problems[i].segments[0] = _lib.MiGemmSegment(pm.data_ptr(), qm.data_ptr(), pm.stride(0), qm.stride(0), k)
            results.append((p, q, c, pm, qm))
        names = launched(lambda: _lib.check(lib.mi_gemm_with_workspace(problems, 6, code, None, 0, ops.stream_ptr()), "mi_gemm_with_workspace"))
        assert sum("wide_kernel" in n and "128" in n for n in names) == len(names) == 1, names
        for k, (p, q, c, _, _) in zip(ks, results):
            pd, qd = p.double(), q.double()
            _close(f"layout {layout} k {k}", c, (pd @ qd.t()).cpu(), (pd.abs() @ qd.abs().t()).cpu(), k, dtype)


# both sides of the lines between the two kernels below 3 GFLOP: blocks of gradients, work and blocks of a forward product, a contraction that is split,
# rows that end inside a block
@pytest.mark.parametrize("rows,ins,outs,forward,backward", [
    (2048, 256, 512, "gemm", "gemm"), (2048, 512, 256, "gemm", "wide"), (1000, 768, 1032, "gemm", "wide"), (1028, 1024, 768, "wide", "wide"), (256, 2048, 256, "gemm", "gemm"),
    (300, 4096, 520, "wide", "wide"), (300, 4088, 520, "gemm", "wide"), (120, 4096, 520, "gemm", "gemm"), (1021, 520, 1048, "gemm", "wide"),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_large_blocks_below_three_gflop(rows, ins, outs, forward, backward, dtype):
    print(f"case large blocks rows={rows} in={ins} out={outs} {dtype}", flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are per compute unit; these sizes are for 256")
    g = torch.Generator(device=DEV).manual_seed(rows)
    x, w, dy = (torch.randn(s, generator=g, device=DEV).to(dtype).requires_grad_() for s in ((rows, ins), (outs, ins), (rows, outs)))
    b = torch.randn(outs, generator=g, device=DEV).to(dtype).requires_grad_()
    y = ops.linear(x, w, b)
    got = [y, *torch.autograd.grad(y, (x, w, b), dy.detach(), retain_graph=True)]
    for kind, call in ((forward, lambda: ops.linear(x, w, b)), (backward, lambda: torch.autograd.grad(y, (x, w, b), dy.detach(), retain_graph=True))):
        names = launched(call)
        assert any(f"{kind}_kernel" in n for n in names) and not any(("gemm" if kind == "wide" else "wide") + "_kernel" in n for n in names), names
    xd, wd, dyd = (t.detach().double() for t in (x, w, dy))
    half_ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for name, a, p, q, k, add in (("y", got[0], xd, wd.t(), ins, b.detach().double()), ("dx", got[1], dyd, wd, outs, 0.0), ("dw", got[2], dyd.t(), xd, rows, 0.0),
                                  ("db", got[3], dyd.t(), torch.ones(rows, 1, dtype=torch.float64, device=DEV), rows, 0.0)):
        ref, mag = (p @ q).reshape(a.shape) + add, (p.abs() @ q.abs()).reshape(a.shape)
        # one rounding of the result, k + 1 of float32 sums, the smallest step of float16
        assert bool(((a.detach().double() - ref).abs() <= half_ulp * ref.abs() + (k + 1) * 2.0 ** -24 * (mag + abs(add)) + 2.0 ** -25).all()), name
