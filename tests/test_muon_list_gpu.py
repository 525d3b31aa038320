"""Muon updates of tensors that lie apart (marked ``gpu``): the same bits as the update of
their stack, whose arithmetic and launch plan they share, at the edges of what one launch
takes (128 matrices) and of the element paths (vector, 8 at a time, one at a time)."""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
KW = dict(lr=0.03, momentum=0.9, weight_decay=0.05)


@pytest.fixture(scope="module", autouse=True)
def _native():
    assert torch.cuda.is_available(), "GPU tests need a ROCm GPU"
    import muon_fusion_ascend950_amd  # noqa: F401  (fails loudly without the HIP library)

    yield


def tensors(count, shape, gen, dtype=torch.float32, offset=0):
    """`count` tensors of one shape, each `offset` elements into an allocation of its own."""
    numel = torch.Size(shape).numel()
    out = []
    for _ in range(count):
        base = torch.randn(numel + offset, generator=gen, device=DEV) * 0.02
        out.append(base.to(dtype)[offset:].view(shape))
    return out


@pytest.mark.parametrize("count,shape,dtype,offset", [
    (2, (256, 512), torch.float32, 0),
    (3, (96, 80), torch.bfloat16, 0),  # right-Gram form
    (5, (33, 130), torch.bfloat16, 0),  # m·n % 8 != 0: one element at a time
    (5, (33, 130), torch.float32, 0),
    (4, (40, 72), torch.float32, 1),  # 8 elements at a time, unaligned
    (4, (40, 72), torch.bfloat16, 3),
    (2, (3, 64, 128), torch.float32, 0),  # several matrices in each tensor
    (43, (3, 16, 24), torch.bfloat16, 0),  # 129 matrices: a second launch of one matrix
    (128, (16, 24), torch.float32, 0),
    (129, (16, 24), torch.float32, 0),
    (2, (768, 3072), torch.float32, 0),
    (1, (2, 512, 1024), torch.bfloat16, 0),
])
@pytest.mark.parametrize("nesterov", [True, False])
def test_apart_equals_stacked(count, shape, dtype, offset, nesterov):
    import muon_fusion_ascend950_amd.optim as optim

    gen = torch.Generator(device=DEV).manual_seed(count * 1000 + shape[-1] + offset)
    p = tensors(count, shape, gen, offset=offset)
    g = tensors(count, shape, gen, dtype, offset)
    b = tensors(count, shape, gen, offset=offset)
    sp, sb = torch.stack(p), torch.stack(b)
    optim.muon_update(sp, torch.stack(g).float(), sb, nesterov=nesterov, **KW)
    assert optim._updatable_in_place(p, g, b)
    optim.muon_update(optim._Matrices(p), optim._Matrices(g), optim._Matrices(b),
                      nesterov=nesterov, **KW)
    assert torch.isfinite(sp).all() and torch.isfinite(sb).all()
    assert torch.equal(torch.stack(p), sp) and torch.equal(torch.stack(b), sb)


def test_what_cannot_be_updated_where_it_lies_is_stacked():
    import muon_fusion_ascend950_amd.optim as optim

    gen = torch.Generator(device=DEV).manual_seed(5)
    p, g, b = (tensors(2, (32, 48), gen) for _ in range(3))
    ok = optim._updatable_in_place
    assert ok(p, g, b) and ok(p, [g[0], g[0]], b)
    over = torch.zeros(33 * 48, device=DEV)
    halves = [over[: 32 * 48].view(32, 48), over[48:].view(32, 48)]
    assert not ok(halves, g, b) and not ok(p, g, halves) and not ok(p, p, b)
    assert not ok([p[0], p[1].T.contiguous().T], g, b)
    assert not ok(p, [g[0], g[1].bfloat16()], b) and not ok(p, [t.half() for t in g], b)
    assert not ok(p, g, [t.bfloat16() for t in b])
    tall = [tensors(2, (48, 36), gen) for _ in range(3)]
    assert not ok(*tall)
    with pytest.raises(RuntimeError, match="overlap"):
        torch.ops.muon_ascend950.muon_update_list(halves, g, b, 0.9, True, [1.0, 0.0, 0.0], 0.1,
                                                  0.0, 1.0)
    # one buffer column-major: the optimizer's step takes it through the stack
    params = [torch.nn.Parameter(t.clone()) for t in p]
    opt = optim.Muon(params, **KW)
    for i, (q, t) in enumerate(zip(params, b)):
        opt.state[q]["momentum_buffer"] = t.clone() if i else t.T.contiguous().T
        q.grad = g[i].clone()
    stack = [torch.stack(t) for t in (p, g, b)]
    optim.muon_update(*stack, **KW)
    versions = [q._version for q in params]
    opt.step()
    for i, q in enumerate(params):
        assert q._version > versions[i]
        assert torch.equal(q.detach(), stack[0][i])
        assert torch.equal(opt.state[q]["momentum_buffer"], stack[2][i])


def test_step_of_apart_parameters_is_seen_by_autograd():
    from muon_fusion_ascend950_amd import Muon

    params = [torch.nn.Parameter(torch.randn(32, 48, device=DEV)) for _ in range(3)]
    for q in params:
        q.grad = torch.randn_like(q)
    y = sum((q * q).sum() for q in params)
    Muon(params, lr=0.1).step()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()


@pytest.mark.parametrize("transform", ["grad", "jvp"])
def test_a_bfloat16_gradient_inside_a_function_transform(transform):
    """The transforms wrap what is computed from their input in tensors without an
    address; the update takes those too, through the operations on tensors."""
    import muon_fusion_ascend950_amd.optim as optim

    gen = torch.Generator(device=DEV).manual_seed(7)
    (p,), (x,), (b,) = (tensors(1, (2, 32, 48), gen) for _ in range(3))
    want_p, want_b = p.clone(), b.clone()
    optim.muon_update(want_p, (2 * x).bfloat16(), want_b, **KW)

    def f(x):
        q, buf = p + 0 * x.detach(), b + 0 * x.detach()
        optim.muon_update(q, (2 * x.detach()).bfloat16(), buf, **KW)
        return (x * x).sum(), (q, buf)

    if transform == "grad":
        d, (q, buf) = torch.func.grad(f, has_aux=True)(x)
        assert torch.equal(d, 2 * x)
    else:
        _, d, (q, buf) = torch.func.jvp(f, (x,), (torch.ones_like(x),), has_aux=True)
        assert torch.allclose(d, 2 * x.sum(), rtol=1e-4)
    assert torch.equal(q, want_p) and torch.equal(buf, want_b)


def graph_nodes(f):
    """Nodes (launches) of `f` captured in a graph."""
    f()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        f()
    with open("/proc/self/maps") as maps:
        path = next(line.split()[-1] for line in maps if "libamdhip64.so" in line)
    nodes = ctypes.c_size_t(0)
    assert ctypes.CDLL(path).hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None,
                                              ctypes.byref(nodes)) == 0
    return nodes.value


@pytest.mark.parametrize("count,shape,launches", [
    (4, (300, 16, 24), 1),  # several matrices in each tensor: one pointer per tensor
    (129, (3, 16, 24), 2),
])
def test_launches_of_a_pass_follow_the_tensors_not_their_matrices(monkeypatch, count, shape,
                                                                  launches):
    import muon_fusion_ascend950_amd.optim as optim

    monkeypatch.delenv("MUON_POLAR_RESIDENT", raising=False)
    gen = torch.Generator(device=DEV).manual_seed(count)
    p, g, b = (tensors(count, shape, gen) for _ in range(3))
    sp, sg, sb = torch.stack(p), torch.stack(g), torch.stack(b)
    apart = [optim._Matrices(t) for t in (p, g, b)]
    update = lambda: optim.muon_update(*apart, **KW)
    # the iteration, and the momentum and the parameter pass
    assert graph_nodes(update) == 1 + 2 * launches
    for t, s in ((p, sp), (b, sb)):
        for i, u in enumerate(t):
            u.copy_(s[i])
    update()
    optim.muon_update(sp, sg, sb, **KW)
    assert torch.equal(torch.stack(p), sp) and torch.equal(torch.stack(b), sb)
