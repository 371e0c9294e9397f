"""GPU: the linear maps around a layer's attention (csrc/linear.hpp) against float64, and the calls that stay with nn.Linear."""

import pytest
import torch
from torch import nn

import natten_amd
from natten_amd import _lib, linear
from natten_amd.fna import _open_call_plan

pytestmark = pytest.mark.gpu

# (rows, input columns, columns per output tensor, output tensors): rows around a tile and a step of the weight
# gradient, columns that take tiles of 128 and of 64, result tiles of either width, more slices than one
SIZES = [(1, 64, 64, 3), (63, 128, 128, 1), (65, 192, 64, 2), (129, 64, 192, 3), (300, 512, 512, 3), (1000, 256, 256, 3),
         (12544, 256, 256, 3), (25000, 128, 512, 1)]


def _bound(ref, magnitude, length, dtype):
    """One rounding to `dtype` and float32 sums of `length` products whose absolute values add up to `magnitude`."""
    unit = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[dtype]
    return unit * ref.abs() + (length + 64) * 2.0**-24 * magnitude + 2.0**-24


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,k,part,parts", SIZES)
def test_maps_against_float64(rows, k, part, parts, dtype):
    gen = torch.Generator().manual_seed(rows + k)
    n = part * parts
    x, w, b, dy = ((torch.randn(s, generator=gen) * f).to(dtype).cuda() for s, f in
                   (((rows, k), 1), ((n, k), k**-0.5), ((n,), 1), ((rows, n), 1)))
    ys = _lib.linear_forward(x, w, b, parts, (rows, part))
    dys = [d.contiguous() for d in dy.split(part, dim=1)]
    dx, dw, db = grads = _lib.linear_backward(dys, x, w, True, True, True)
    assert all(torch.equal(a, b) for a, b in zip(grads, _lib.linear_backward(dys, x, w, True, True, True)))
    # parts of them, in launches of their own
    for need in ((True, False, False), (False, True, False), (False, False, True), (True, False, True)):
        for flag, got, ref in zip(need, _lib.linear_backward(dys, x, w, *need), grads):
            assert torch.equal(got, ref) if flag else got is None
    X, W, B, DY = (t.double() for t in (x, w, b, dy))
    for got, ref, size, length in (
            (torch.cat(ys, dim=1), X @ W.t() + B, X.abs() @ W.abs().t() + B.abs(), k + 1),
            (dx, DY @ W, DY.abs() @ W.abs(), n),
            (dw, DY.t() @ X, DY.abs().t() @ X.abs(), rows),
            (db, DY.sum(0), DY.abs().sum(0), rows)):
        assert got.shape == ref.shape
        assert ((got.double() - ref).abs() <= _bound(ref, size, length, dtype)).all()
    assert torch.equal(_lib.linear_forward(x, w, None, parts, (rows, part))[0].float(),
                       _lib.linear_forward(x, w, torch.zeros_like(b), parts, (rows, part))[0].float())


def test_the_copies_behind_the_last_token_count_nowhere():
    # infinities in the last row reach the gradients once, through the products that hold them
    x, dy = torch.ones((70, 64), dtype=torch.float16, device="cuda"), torch.ones((70, 64), dtype=torch.float16, device="cuda")
    x[-1, 3] = float("inf")
    _, dw, db = _lib.linear_backward([dy], x, torch.zeros((64, 64), dtype=torch.float16, device="cuda"), False, True, True)
    assert torch.isinf(dw[:, 3]).all() and (dw[:, :3] == 70).all() and (dw[:, 4:] == 70).all() and (db == 70).all()


def test_sizes_that_the_kernels_do_not_take_are_refused():
    x, w = torch.zeros((8, 64), dtype=torch.bfloat16, device="cuda"), torch.zeros((96, 64), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="multiples of 64"):
        _lib.linear_forward(x, w, None, 1, (8, 96))
    with pytest.raises(RuntimeError, match="workspace"):
        _lib._check(_lib.lib().natten_amd_linear_backward(
            x.data_ptr(), None, None, x.data_ptr(), None, None, w.data_ptr(), None, w.data_ptr(), 16, 1, 8, 64, 64, 64, None))


def _layer(**kwargs):
    torch.manual_seed(0)
    return natten_amd.NeighborhoodAttention2D(128, 4, (5, 5), **kwargs).to("cuda", torch.bfloat16)


def _step(layer, x, d):
    x = x.detach().requires_grad_(True)
    out = layer(x)
    params = [p for p in layer.parameters() if p.requires_grad]
    return [out.detach(), *torch.autograd.grad(out, [x, *params], d)]


def _close(a, b):
    # two roundings to bf16 of the same sums, carried through the attention and the second map
    return all(float((p.double() - q.double()).norm()) <= 2.0**-6 * float(q.double().norm()) for p, q in zip(a, b))


@pytest.mark.parametrize("qkv_bias", [True, False])
def test_layer_steps_of_both_routes_agree(qkv_bias, monkeypatch):
    layer, gen = _layer(qkv_bias=qkv_bias), torch.Generator(device="cuda").manual_seed(1)
    x, d = (torch.randn((2, 12, 13, 128), generator=gen, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    assert linear.takes_linear(layer.qkv, x, 3) and linear.takes_linear(layer.proj, x, 1)
    own = _step(layer, x, d)
    with torch.no_grad():
        assert torch.equal(layer(x), own[0])
    # a strided input and a strided gradient
    strided = _step(layer, x.transpose(1, 2).contiguous().transpose(1, 2), d.transpose(1, 2).contiguous().transpose(1, 2))
    assert all(torch.equal(a, b) for a, b in zip(own, strided))
    # the three nodes that stand for the one where its plan has no place
    with monkeypatch.context() as m:
        m.setattr(linear, "_layer_backward_plan", lambda *a: None)
        assert all(torch.equal(a, b) for a, b in zip(own, _step(layer, x, d)))
    with monkeypatch.context() as m:
        m.setattr(linear, "takes_linear", lambda *a: False)
        general = _step(layer, x, d)
    assert _close(own, general)
    # the gradient of a gradient

    def twice(layer):
        y = x.detach().requires_grad_(True)
        dx, = torch.autograd.grad(layer(y), y, d, create_graph=True)
        return torch.autograd.grad(dx.float().square().sum(), layer.qkv.weight, allow_unused=True)

    second = twice(layer)
    monkeypatch.setattr(linear, "takes_linear", lambda *a: False)
    assert _close(second, twice(layer))


def test_a_step_whose_forward_runs_in_pairs_agrees_with_the_other_routes(monkeypatch):
    # the one node's forward leaves the launch open (two groups of waves a Q tile here), those of three nodes and of the
    # general route do not: other orders of summation
    torch.manual_seed(0)
    layer = natten_amd.NeighborhoodAttention2D(128, 2, (13, 13)).to("cuda", torch.bfloat16)
    plan = _open_call_plan(torch.bfloat16, (1, 128, 128, 2, 64), 2, *((n, n) for n in (13, 1, 1)), (False, False), None)
    assert plan[2] == "paired"
    x, d = (torch.randn((1, 128, 128, 128), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    own = _step(layer, x, d)
    with torch.no_grad():
        assert torch.equal(layer(x), own[0])
    for name, stand_in in (("_layer_backward_plan", lambda *a: None), ("takes_linear", lambda *a: False)):
        with monkeypatch.context() as m:
            m.setattr(linear, name, stand_in)
            assert _close(own, _step(layer, x, d))


def test_what_is_attached_to_a_map_is_kept():
    layer, x = _layer(), torch.randn((1, 8, 8, 128), device="cuda", dtype=torch.bfloat16)
    seen = []
    handle = layer.qkv.register_forward_hook(lambda m, a, out: seen.append(tuple(out.shape)))
    layer(x)
    assert seen == [(1, 8, 8, 384)] and not linear.takes_linear(layer.qkv, x, 3)
    handle.remove()

    class Adapted(nn.Linear):
        def forward(self, x):
            return super().forward(x) * 0

    assert linear.takes_linear(layer.qkv, x, 3)
    for attempt in (lambda: linear.takes_linear(Adapted(128, 384).to("cuda", torch.bfloat16), x, 3),
                    lambda: linear.takes_linear(layer.qkv.float(), x, 3), lambda: linear.takes_linear(layer.qkv, x.float(), 3)):
        assert not attempt()
    layer.qkv.to(torch.bfloat16)
    with torch.autocast("cuda", dtype=torch.float16):
        assert not linear.takes_linear(layer.qkv, x, 3) and layer(x).dtype == torch.float16
    nn.utils.parametrizations.weight_norm(layer.proj)
    assert not linear.takes_linear(layer.proj, x, 1)
    layer(x)


@pytest.mark.parametrize("columns", [64, 192])
def test_an_output_map_to_another_width_is_that_of_its_module(columns, monkeypatch):
    layer, x = _layer(), torch.randn((2, 12, 13, 128), device="cuda", dtype=torch.bfloat16)
    layer.proj = nn.Linear(128, columns).to("cuda", torch.bfloat16)
    d = torch.randn((2, 12, 13, columns), device="cuda", dtype=torch.bfloat16)
    got = _step(layer, x, d)
    with torch.no_grad():
        assert torch.equal(layer(x), got[0])
    monkeypatch.setattr(linear, "takes_linear", lambda *a: False)
    assert got[0].shape == d.shape and all(torch.equal(a, b) for a, b in zip(got, _step(layer, x, d)))


@pytest.mark.parametrize("name,sizes", [("proj", (64, 64)), ("proj", (256, 128)), ("qkv", (64, 192)), ("qkv", (64, 384)),
                                        ("qkv", (128, 192))])
@pytest.mark.parametrize("grad", [False, True])
def test_maps_that_do_not_fit_the_layer_are_refused(name, sizes, grad):
    layer, x = _layer(), torch.randn((2, 12, 14, 128), device="cuda", dtype=torch.bfloat16)
    setattr(layer, name, nn.Linear(*sizes).to("cuda", torch.bfloat16))
    assert not linear.takes_linear(getattr(layer, name), x, 3 if name == "qkv" else 1)
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="shapes cannot be multiplied|is invalid for input of size"):
        layer(x)


def test_a_bias_of_one_element_is_left_to_its_module():
    layer, x = _layer(), torch.randn((2, 12, 13, 128), device="cuda", dtype=torch.bfloat16)
    layer.proj.bias = nn.Parameter(torch.ones((1,), device="cuda", dtype=torch.bfloat16))
    assert not linear.takes_linear(layer.proj, x, 1)
    with torch.no_grad():
        assert layer(x).shape == x.shape


def test_tensors_that_do_not_fit_a_map_are_refused():
    x, w = torch.zeros((8, 128), dtype=torch.bfloat16, device="cuda"), torch.zeros((64, 64), dtype=torch.bfloat16, device="cuda")
    for operand, shape in ((x, (8, 128)), (x, (16, 64)), (x.view(16, 64), (8, 64)), (x.view(16, 64), (8, 128))):
        with pytest.raises(ValueError, match="columns"):
            _lib.linear_forward(operand, w, None, 1, shape)
    with pytest.raises(ValueError, match="rows"):
        _lib.linear_backward([x.view(16, 64)[:8]], x.view(16, 64), w, True, True, False)


def test_frozen_weights_and_saved_tensor_hooks():
    layer, x = _layer(), torch.randn((1, 8, 8, 128), device="cuda", dtype=torch.bfloat16)
    d = torch.randn_like(x)
    ref = _step(layer, x, d)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu(), lambda t: t.cuda()):
        assert all(torch.equal(a, b) for a, b in zip(ref, _step(layer, x, d)))
    assert packed
    for p in layer.parameters():
        p.requires_grad_(False)
    assert all(torch.equal(a, b) for a, b in zip(ref[:2], _step(layer, x, d)))
    layer.qkv.bias.requires_grad_(True)
    names = [name for name, _ in layer.named_parameters()]
    assert torch.equal(_step(layer, x, d)[2], ref[2 + names.index("qkv.bias")])
    # a weight changed between the passes is noticed
    out = layer(x.requires_grad_(True))
    with torch.no_grad():
        layer.proj.weight.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(d)
