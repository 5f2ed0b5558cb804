"""Gradients where their kernels take another path: rows of a gate that end inside a 16-byte granule or start off one, and the
map from buffer rows to slots in memory that holds anything."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as mo
from tests.gpu_util import TORCH_DT, dev, make_inputs, to_np

pytestmark = pytest.mark.gpu


def _off(t, n):
    """t's values n elements into an allocation."""
    buf = torch.empty(t.numel() + n, dtype=t.dtype, device=t.device)
    view = buf[n:].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("S,E", [(1, 2), (63, 9), (65, 13), (130, 60), (64, 61), (257, 7), (100, 255), (33, 512)])
@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("gdt,offset", [("f32", 0), ("f32", 1), ("bf16", 0), ("f16", 3)])
def test_gate_gradient_of_rows_of_any_length(pkg, S, E, k, gdt, offset):
    """The bars of the gate gradient's own tests: 1e-5 relative, with 1e-6 of the row's largest entry where terms cancel;
    16-bit gates one unit in the last place or that floor."""
    tdt = TORCH_DT[gdt]
    data, logits = make_inputs(S + E, S, 4, E)
    gate = dev(logits).to(tdt)
    rounded = gate.float().cpu().numpy()
    enc = mo.moe_encode_top2 if k == 2 else mo.moe_encode
    il = enc(data, rounded, np.zeros(E, np.int32), 0.8, gate_is_logits=True, fast_scatter=True)[1]
    dy = dev(np.random.default_rng(S).standard_normal(k * S).astype(np.float32)).to(tdt)
    want = mo.moe_encode_dgate(dy.float().cpu().numpy(), rounded, il, k, True)
    out = _off(torch.full((S, E), 7.0, dtype=tdt, device="cuda"), offset)
    got = to_np(pkg.ops.moe_encode_dgate(dy, _off(gate, offset), dev(il), top_k=k, gate_is_logits=True, out=out)).astype(np.float64)
    scale = np.abs(want).max(axis=1, keepdims=True)
    eps = {"f32": 1e-5, "bf16": 2.0 ** -7, "f16": 2.0 ** -10}[gdt]          # one unit in the last place of a 16-bit value
    tiny = {"f32": 1e-30, "bf16": 1e-30, "f16": 2.0 ** -24}[gdt]
    assert (np.abs(got - want) <= eps * np.abs(want) + 1e-6 * scale + tiny).all()


# one, two and four values per lane; one granule per lane, and the first rows with two; blocks written by value and in granules
@pytest.mark.parametrize("S,E", [(64, 3), (65, 4), (129, 5), (64, 8), (70, 12), (63, 14), (64, 16), (66, 17), (257, 24), (65, 32), (64, 33)])
@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("gdt,offset", [("f32", 0), ("bf16", 0), ("f16", 3)])
def test_gate_gradient_of_short_rows(pkg, S, E, k, gdt, offset):
    test_gate_gradient_of_rows_of_any_length(pkg, S, E, k, gdt, offset)
    # on probabilities, and on logits of which some are masked out: those get no gradient, the others what the oracle says
    tdt = TORCH_DT[gdt]
    logits = make_inputs(E, S, 4, E)[1]
    masked = logits.copy()
    masked[::3, ::2] = -np.inf
    for gate, is_logits in ((np.exp(logits) / np.exp(logits).sum(axis=1, keepdims=True), False), (masked, True)):
        gate = dev(gate.astype(np.float32)).to(tdt)
        rounded = gate.float().cpu().numpy()
        il = np.zeros((2, k * S), np.int32)
        il[0] = np.argsort(-rounded, axis=1, kind="stable")[:, :k].T.reshape(-1)
        il[0][::7] = -1
        if is_logits:                              # a masked expert is nobody's choice
            chosen = rounded[np.tile(np.arange(S), k), il[0]]
            il[0][np.isinf(chosen)] = -1
        dy = dev(np.random.default_rng(S).standard_normal(k * S).astype(np.float32)).to(tdt)
        want = mo.moe_encode_dgate(dy.float().cpu().numpy(), rounded, il, k, is_logits)
        out = _off(torch.full((S, E), 7.0, dtype=tdt, device="cuda"), offset)
        got = to_np(pkg.ops.moe_encode_dgate(dy, _off(gate, offset), dev(il), top_k=k, gate_is_logits=is_logits, out=out)).astype(np.float64)
        scale = np.abs(want).max(axis=1, keepdims=True)
        eps = {"f32": 1e-5, "bf16": 2.0 ** -7, "f16": 2.0 ** -10}[gdt]
        tiny = {"f32": 1e-30, "bf16": 1e-30, "f16": 2.0 ** -24}[gdt]
        assert np.isfinite(got).all() and (np.abs(got - want) <= eps * np.abs(want) + 1e-6 * scale + tiny).all()


@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("fill", ["zeros", "ones", "last", "others", "large"])
def test_row_map_in_memory_that_holds_anything(pkg, k, fill):
    """decode_dx and decode_grad on a workspace full of numbers that look like slots: rows nobody owns are zero all the same."""
    ops, lib = pkg.ops, pkg.capi.load()
    S, M, E = 9000, 16, 5                         # more slots than are walked without a map
    data, logits = make_inputs(21, S, M, E, zipf_bias=True)
    enc = mo.moe_encode_top2 if k == 2 else mo.moe_encode
    g, il, used, _, disp = enc(data, logits, np.zeros(E, np.int32), 0.9, gate_is_logits=True, fast_scatter=True)
    C = disp.shape[1]
    assert (used < C).any() and (il[0] < 0).any()
    n = int(lib.lancet_moe_decode_dx_workspace_bytes(E, C)) // 4
    ws = {"zeros": lambda: torch.zeros(n, dtype=torch.int32), "ones": lambda: torch.ones(n, dtype=torch.int32),
          "last": lambda: torch.full((n,), k * S - 1, dtype=torch.int32), "large": lambda: torch.full((n,), 0x7fffffff, dtype=torch.int32),
          "others": lambda: torch.arange(n, dtype=torch.int32) % (k * S)}[fill]().cuda().view(torch.uint8)
    tok = np.random.default_rng(1).standard_normal((S, M)).astype(np.float32)
    want = mo.moe_decode_dx(tok, g, il, E, C, k)
    got = ops.moe_decode_dx(dev(tok), dev(g), dev(il), E, C, top_k=k, workspace=ws.clone())
    np.testing.assert_array_equal(to_np(got), want)
    d_rows, d_g = ops.moe_decode_grad(dev(tok), dev(disp), dev(g), dev(il), top_k=k, workspace=ws.clone())
    np.testing.assert_array_equal(to_np(d_rows), want)


# a wave with one row to look up and with several, ends inside them; up to 262144 rows the map is checked, beyond it is cleared
@pytest.mark.parametrize("S,M,E,cf", [(9000, 512, 5, 0.9), (9000, 520, 33, 1.3), (5000, 2050, 7, 1.1), (60000, 8, 3, 3.0), (70000, 264, 64, 2.0)])
@pytest.mark.parametrize("k", [1, 2])
def test_row_map_of_rows_looked_up_together(pkg, S, M, E, cf, k):
    """Gradients of the expert rows, bit for bit: a copy of dy where the weight is a power of two, zero where nobody owns the row."""
    ops, lib = pkg.ops, pkg.capi.load()
    logits = torch.randn((S, E), device="cuda", generator=torch.Generator(device="cuda").manual_seed(S)) + torch.arange(E, device="cuda") % 3
    C = ops.moe_capacity(S, E, cf)
    dy = torch.randn((S, M), device="cuda", generator=torch.Generator(device="cuda").manual_seed(M)).bfloat16()
    _, il, _, _ = ops.moe_route(logits, None, M, top_k=k, gate_is_logits=True, capacity=C)
    g = torch.exp2(-(torch.arange(k * S, device="cuda") % 4).float())
    want = torch.zeros((E, C, M), dtype=torch.bfloat16, device="cuda")
    keep = il[0] >= 0
    want[il[0][keep].long(), il[1][keep].long()] = (dy.repeat(k, 1) * g[:, None].bfloat16())[keep]
    assert (~keep).any() or cf > 1.0
    ws = (torch.arange(int(lib.lancet_moe_decode_dx_workspace_bytes(E, C)) // 4, dtype=torch.int32, device="cuda") % (k * S)).view(torch.uint8)
    got = ops.moe_decode_dx(dy, g, il, E, C, top_k=k, workspace=ws.clone())
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    rows = torch.randn((E, C, M), device="cuda").bfloat16()
    d_rows, _ = ops.moe_decode_grad(dy, rows, g, il, top_k=k, workspace=ws.clone())
    assert torch.equal(d_rows.view(torch.int16), want.view(torch.int16))
