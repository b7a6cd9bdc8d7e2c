"""The native autograd functions behind the layer operators (csrc/host_ops.cpp) as autograd sees them: what they keep, what
they refuse, which inputs get gradients, and inputs in other types and layouts.  Their values are compared with the oracle
in the operators' own tests."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _ops():
    from difflut_amd import ops
    return ops


def _calls():
    """name -> (function of the differentiable inputs, those inputs), one small call of every native operator."""
    ops = _ops()
    g = torch.Generator(DEV).manual_seed(5)
    B, I, N, k = 70, 40, 65, 4

    def rand(*shape):
        return torch.rand(*shape, device=DEV, generator=g)

    plan = ops.MappingPlan(torch.randint(0, I, (N, k), device=DEV, generator=g, dtype=torch.int32), I)
    plan2 = ops.MappingPlan(torch.randint(0, N, (64, k), device=DEV, generator=g, dtype=torch.int32), N)
    x, luts, luts2 = rand(B, I), rand(N, 1, 1 << k) * 2 - 1, rand(64, 1, 1 << k) * 2 - 1
    alpha, beta, scale = rand(N), rand(N) * 0.4, rand(N) + 0.5
    both = [(alpha, beta, 0.4), (alpha[:64].clone(), beta[:64].clone(), 0.4)]
    labels = torch.randint(0, 5, (B,), device=DEV, generator=g)
    return {
        "dwn": (lambda a, t: ops.DWNLayerFunction.apply(a, t, plan, 0.3, 0.25), [x, luts]),
        "dwn_per_node": (lambda a, t: ops.DWNLayerFunction.apply(a, t, plan, alpha, beta, 0.4), [x, luts]),
        "dwn_stable": (lambda a, t: ops.DWNStableLayerFunction.apply(a, t, scale, plan), [x, luts]),
        "hybrid": (lambda a, t: ops.HybridLayerFunction.apply(a, t, plan), [x, luts]),
        "hybrid_no_tiles": (lambda a, t: ops.HybridLayerFunction.apply(a, t, plan, False), [x, luts]),
        "sigmoid": (ops.TableSigmoidFunction.apply, [luts]),
        "prob": (lambda a, t: ops.ProbLayerFunction.apply(a, t, plan, 0.7), [x, rand(N, 1 << k, 1)]),
        "prob_per_node": (lambda a, t: ops.ProbLayerFunction.apply(a, t, plan, alpha + 0.5), [x, rand(N, 1 << k, 1)]),
        "soft_map": (lambda a, w: ops.SoftMapFunction.apply(a, w, 0.8, 0), [x, rand(N, I)]),
        "stack": (lambda a, s, t: ops.DWNStackFunction.apply(a, None, [plan, plan2], both, None, s, t), [x, luts, luts2]),
        "stack_numbers": (lambda a, s, t: ops.DWNStackFunction.apply(a, None, [plan, plan2], [(0.3, 0.25), (0.2, 0.3)], None, s, t),
                          [x, luts, luts2]),
        "cross_entropy": (lambda a: ops.CrossEntropyFunction.apply(a, labels), [rand(B, 5)]),
    }


NAMES = ["dwn", "dwn_per_node", "dwn_stable", "hybrid", "hybrid_no_tiles", "sigmoid", "prob", "prob_per_node", "soft_map", "stack",
         "stack_numbers", "cross_entropy"]


def _run(call, inputs, gy=None, wanted=None, **options):
    leaves = [t.detach().requires_grad_(wanted is None or i in wanted) for i, t in enumerate(inputs)]
    y = call(*leaves)
    y.backward(torch.ones_like(y) if gy is None else gy, **options)
    return y, [t.grad for t in leaves]


@pytest.mark.parametrize("name", NAMES)
def test_gradients_go_where_they_are_asked_for(name):
    call, inputs = _calls()[name]
    y, grads = _run(call, inputs)
    assert y.requires_grad and all(g.shape == t.shape for g, t in zip(grads, inputs))
    for i in range(len(inputs)):
        _, only = _run(call, inputs, wanted={i})
        assert [g is None for g in only] == [j != i for j in range(len(inputs))]
        torch.testing.assert_close(only[i], grads[i], rtol=1e-5, atol=1e-6)
    assert not call(*inputs).requires_grad
    with torch.no_grad():
        assert torch.equal(call(*[t.detach().requires_grad_() for t in inputs]), y)


@pytest.mark.parametrize("name", NAMES)
def test_a_second_backward(name):
    call, inputs = _calls()[name]
    leaves = [t.detach().requires_grad_() for t in inputs]
    y = call(*leaves)
    gy = torch.ones_like(y)
    y.backward(gy, retain_graph=True)
    first = [t.grad.clone() for t in leaves]
    y.backward(gy)  # adds the same gradients once more
    for t, g in zip(leaves, first):
        assert torch.equal(t.grad, 2 * g)
    with pytest.raises(RuntimeError, match="second time"):
        y.backward(gy)


@pytest.mark.parametrize("name", NAMES)
def test_saved_tensor_hooks_and_versions(name):
    call, inputs = _calls()[name]
    y, grads = _run(call, inputs)
    packed = []

    def pack(t):
        packed.append(t)
        return t.cpu()  # as an offloading hook does

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
        leaves = [t.detach().requires_grad_() for t in inputs]
        y = call(*leaves)
    y.backward(torch.ones_like(y))
    assert packed and all(torch.equal(t.grad, g) for t, g in zip(leaves, grads))
    if name not in ("sigmoid", "cross_entropy"):  # those keep nothing but their own results
        leaves = [t.detach().clone().requires_grad_() for t in inputs]
        y = call(*leaves)
        with torch.no_grad():
            leaves[-1].mul_(2.0)  # the tables, which every backward reads
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.backward(torch.ones_like(y))


@pytest.mark.parametrize("name", NAMES)
def test_transforms_that_would_pass_the_kernels_by_are_refused(name):
    call, inputs = _calls()[name]
    with pytest.raises(RuntimeError):
        torch.func.vmap(call)(*[t.unsqueeze(0) for t in inputs])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda *a: call(*a).sum())(*inputs)
    with pytest.raises(RuntimeError):
        with torch.autograd.forward_ad.dual_level():
            call(torch.autograd.forward_ad.make_dual(inputs[0], torch.ones_like(inputs[0])), *inputs[1:])


@pytest.mark.parametrize("name", NAMES)
def test_other_types_and_layouts(name):
    call, inputs = _calls()[name]
    y, grads = _run(call, inputs)
    # strided inputs, and an expanded upstream gradient
    strided = [torch.empty(*t.shape[:-1], 2 * t.shape[-1], device=DEV)[..., ::2].copy_(t) for t in inputs]
    leaves = [t.requires_grad_() for t in strided]
    out = call(*leaves)
    assert not any(t.is_contiguous() for t in leaves) and torch.equal(out, y)
    out.backward(torch.ones((), device=DEV).expand_as(out))
    assert all(torch.equal(t.grad, g) for t, g in zip(leaves, grads))
    # double inputs: fp32 inside, double gradients
    leaves = [t.double().requires_grad_() for t in inputs]
    out = call(*leaves)
    assert out.dtype == torch.float32 and torch.equal(out, y)
    out.backward(torch.ones_like(out))
    assert all(t.grad.dtype == torch.float64 and torch.equal(t.grad.float(), g) for t, g in zip(leaves, grads))


@pytest.mark.parametrize("name", NAMES)
def test_the_current_stream_and_tensors_on_the_cpu(name):
    call, inputs = _calls()[name]
    y, grads = _run(call, inputs)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        out, side_grads = _run(call, inputs)
    side.synchronize()
    assert torch.equal(out, y) and all(torch.equal(a, b) for a, b in zip(side_grads, grads))
    with pytest.raises(RuntimeError, match="ROCm devices only"):
        call(*[t.cpu() for t in inputs])


@pytest.mark.parametrize("shape", [(8,), (4, 8, 2), (4, 8, 1), ()])
def test_soft_map_refuses_inputs_that_are_no_matrix(shape):
    with pytest.raises((ValueError, IndexError, RuntimeError)):
        _ops().SoftMapFunction.apply(torch.rand(shape, device=DEV), torch.rand(6, 8, device=DEV), 1.0, 0)


@pytest.mark.parametrize("alpha,beta", [(0.3, "tensor"), ("tensor", 0.25), (0.3, 0.25), ([0.3], "tensor")])
def test_stack_takes_a_number_beside_per_node_values(alpha, beta):
    ops = _ops()
    _, (x, luts, luts2) = _calls()["stack"]
    plan = ops.MappingPlan(torch.arange(65 * 4, device=DEV, dtype=torch.int32).reshape(65, 4) % 40, 40)
    plan2 = ops.MappingPlan(torch.arange(64 * 4, device=DEV, dtype=torch.int32).reshape(64, 4) % 65, 65)

    def scalars(n, as_given):
        return tuple(torch.full((n,), fill, device=DEV) if v == "tensor" or not as_given else v for v, fill in ((alpha, 0.3), (beta, 0.25)))

    def run(as_given):
        both = [scalars(n, as_given) + (0.25,) for n in (65, 64)]
        return _run(lambda a, s, t: ops.DWNStackFunction.apply(a, None, [plan, plan2], both, None, s, t), [x, luts, luts2])

    (y, grads), (want, want_grads) = run(True), run(False)
    assert torch.equal(y, want) and all(torch.equal(a, b) for a, b in zip(grads, want_grads))
