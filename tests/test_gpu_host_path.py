"""The operators' native host path: what it refuses, what it returns, and how its autograd nodes behave under the tools that
reach into a backward pass.  (What the operators compute is tested by the other GPU tests, which all go through it.)"""
import pytest
import torch

from tests.gpu_util import dev, make_inputs

pytestmark = pytest.mark.gpu

S, M, E = 96, 32, 4


def _inputs(dtype=torch.float32):
    data, logits = make_inputs(5, S, M, E)
    return dev(data).to(dtype), dev(logits)


@pytest.mark.parametrize("case", ["cpu", "strided", "rank", "rows", "dtype", "top_k", "noise", "used", "capacity", "mask", "partition",
                                  "top_k_zero", "not_a_tensor", "status"])
def test_refused_arguments(pkg, case):
    ops = pkg.ops
    data, gate = _inputs()
    il = torch.zeros((2, S), dtype=torch.int32, device="cuda")
    buf, g = torch.zeros((E, 8, M), device="cuda"), torch.ones(S, device="cuda")
    calls = {
        "cpu": (ValueError, lambda: ops.moe_encode(data.cpu(), gate, None)),
        "strided": (ValueError, lambda: ops.moe_encode(data.t(), gate, None)),
        "rank": (ValueError, lambda: ops.moe_encode(data[None], gate, None)),
        "rows": (ValueError, lambda: ops.moe_encode(data[:-1], gate, None)),
        "dtype": (TypeError, lambda: ops.moe_encode(data.double(), gate, None)),
        "top_k": (ValueError, lambda: ops.moe_encode(data, gate, None, top_k=3)),
        "noise": (ValueError, lambda: ops.moe_encode(data, gate, None, gate2_noise=gate)),
        "used": (ValueError, lambda: ops.moe_encode(data, gate, torch.zeros(E, dtype=torch.int64, device="cuda"))),
        "capacity": (ValueError, lambda: ops.moe_encode(data, gate, None, capacity=-1)),
        "mask": (ValueError, lambda: ops.moe_decode(buf, g, il[:, :-1].contiguous())),
        "partition": (ValueError, lambda: ops.moe_encode_batch_prioritized(data, gate, 2, 2)),
        "top_k_zero": (ValueError, lambda: ops.moe_decode(buf, g, il, top_k=0)),
        "not_a_tensor": (TypeError, lambda: ops.moe_decode([1.0], g, il)),
        "status": (pkg.capi.LancetError, lambda: ops.moe_encode(data, gate[:, :1].contiguous(), None, top_k=2)),
    }
    error, call = calls[case]
    with pytest.raises(error) as info:
        call()
    if case == "status":
        assert info.value.status == pkg.capi.ERR_TOPK


def test_given_outputs_are_returned(pkg):
    ops = pkg.ops
    data, gate = _inputs()
    first = ops.moe_encode(data, gate, None, 1.0, gate_is_logits=True)
    assert first[3].dtype == torch.uint64
    outs = [torch.empty_like(t) for t in first[:3]] + [torch.empty(E, dtype=torch.int64, device="cuda"), torch.empty_like(first[4])]
    second = ops.moe_encode(data, gate, None, 1.0, gate_is_logits=True, out=outs)
    assert all(second[i] is outs[i] for i in (0, 1, 2, 4)) and second[3].dtype == torch.uint64
    assert second[3].data_ptr() == outs[3].data_ptr()
    for a, b in zip(first, second):
        assert torch.equal(a.view(torch.int64) if a.dtype == torch.uint64 else a, b.view(torch.int64) if b.dtype == torch.uint64 else b)
    y = torch.empty((S, M), device="cuda")
    assert ops.moe_decode(first[4], first[0], first[1], out=y) is y


def _layer(grad, data, gate):
    gates_s, il, _, _, disp = grad.moe_encode(data, gate, None, 1.0, top_k=2, gate_is_logits=True)
    return grad.moe_decode(disp, gates_s, il, top_k=2)


def test_autograd_nodes_under_tools(pkg):
    """Hooks on saved tensors and on gradients, checkpointing, gradients of one input alone, a second backward, and what
    functions with a backward rule alone refuse."""
    grad = pkg.grad
    data, gate = (t.requires_grad_(True) for t in _inputs())
    y = _layer(grad, data, gate)
    dy = torch.randn_like(y)
    want = torch.autograd.grad(y, (data, gate), dy, retain_graph=True)
    again = torch.autograd.grad(y, (data, gate), dy)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, (data, gate), dy)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t) or t, lambda t: t):
        z = _layer(grad, data, gate)
    assert len(seen) >= 5                                  # mask and gate of the encode; rows, weights and mask of the decode
    scaled = []
    z.register_hook(lambda g: scaled.append(g) or g)
    hooked = torch.autograd.grad(z, (data, gate), dy)
    assert len(scaled) == 1
    kept = torch.utils.checkpoint.checkpoint(lambda d, g: _layer(grad, d, g), data, gate, use_reentrant=False)
    checkpointed = torch.autograd.grad(kept, (data, gate), dy)
    alone = (torch.autograd.grad(_layer(grad, data, gate.detach()), data, dy)[0],
             torch.autograd.grad(_layer(grad, data.detach(), gate), gate, dy)[0])
    for got in (again, hooked, checkpointed, alone):
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    # the weights alone depend on the loss: the dispatched rows' gradient is zero, and so is the tokens'
    gates_s, il, used, elems, disp = grad.moe_encode(data, gate, None, 1.0, top_k=2, gate_is_logits=True)
    assert not (il.requires_grad or used.requires_grad or elems.requires_grad) and gates_s.requires_grad and disp.requires_grad
    assert not torch.autograd.grad(gates_s.sum(), data)[0].any()
    # what one version of the saved rows was computed from must still be there
    buf = disp.detach().clone().requires_grad_(True)
    out = grad.moe_decode(buf, gates_s.detach(), il, top_k=2)
    with torch.no_grad():
        buf += 1
    with pytest.raises(RuntimeError, match="inplace"):
        out.sum().backward()
    # no forward-mode rule, no batching rule
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(data.detach(), torch.ones_like(data))
        with pytest.raises(RuntimeError):
            _layer(grad, dual, gate.detach())
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda d: _layer(grad, d, gate.detach()))(data.detach()[None])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda d: _layer(grad, d, gate.detach()).sum())(data.detach())


def test_bpr_gradient_covers_the_partition_alone(pkg):
    grad = pkg.grad
    data, gate = (t.requires_grad_(True) for t in _inputs())
    out = grad.moe_encode_batch_prioritized(data, gate, 2, 1, 1.0, gate_is_logits=True)
    dx, dg = torch.autograd.grad((out[0].sum() + out[4].sum()), (data, gate))
    assert dx.shape == data.shape and dg.shape == gate.shape
    assert not dx[:S // 2].any() and not dg[:S // 2].any() and dx[S // 2:].any() and dg[S // 2:].any()


@pytest.mark.parametrize("case", ["route", "route_workspace", "scatter", "decode", "ranges", "ranges_workspace"])
def test_named_streams_take_given_arrays_alone(pkg, case):
    """What a native call would allocate belongs to the current stream, not to the one that is named."""
    ops, host = pkg.ops, pkg.capi.host()
    data, gate = _inputs()
    il, g = torch.zeros((2, S), dtype=torch.int32, device="cuda"), torch.ones(S, device="cuda")
    used, buf = torch.zeros(E, dtype=torch.int32, device="cuda"), torch.zeros((E, 8, M), device="cuda")
    outs = (g, il, used, torch.zeros(E, dtype=torch.int64, device="cuda"))
    pair = (torch.zeros((2, E), dtype=torch.int64, device="cuda"),) * 2
    side = torch.cuda.Stream().cuda_stream
    calls = {
        "route": lambda: host.moe_route(gate, None, None, M, 1.0, 8, 1, 0, ops.ScanWorkspace(1 << 16), None, side),
        "route_workspace": lambda: host.moe_route(gate, None, None, M, 1.0, 8, 1, 0, None, outs, side),
        "scatter": lambda: host.moe_scatter_tokens(data, il, None, used, 0, E, 8, 1, 0, None, side),
        "decode": lambda: host.moe_decode_tokens(buf, g, il, 0, S, 1, None, side),
        "ranges": lambda: host.moe_partition_ranges(il, 2, E, M, 1, torch.zeros(4096, dtype=torch.uint8, device="cuda"), None, side),
        "ranges_workspace": lambda: host.moe_partition_ranges(il, 2, E, M, 1, None, pair, side),
    }
    with pytest.raises(ValueError, match="named stream"):
        calls[case]()
