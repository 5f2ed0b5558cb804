"""Row movers where their launches are laid out in another way: tails cleared among the tokens' workgroups, and wide rows in the
gradient of decode."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as mo
from tests.gpu_util import TORCH_DT, dev, make_inputs, rows_as_oracle, rows_to_torch, to_np, ulp_distance

pytestmark = pytest.mark.gpu


# tails among the tokens: one eight in two to in many, tails that are no multiple of eight, the most tails there may be workgroups (64 x
# 256, 512 x 19: one per expert has several turns), long passes of shorter rows; behind them: more workgroups of tails than of tokens, rows and passes just
# short of that, top-1 rows just longer, short rows
@pytest.mark.parametrize("S,M,E,C", [(8200, 768, 5, 8000), (8193, 776, 2, 15001), (20000, 768, 64, 4096), (40000, 768, 512, 300), (8200, 2048, 7, 1500), (30000, 1600, 3, 100),
                                     (150000, 384, 11, 20000), (8200, 768, 5, 30000), (8200, 760, 7, 4900), (8200, 768, 7, 4700), (8200, 2056, 7, 1300),
                                     (8200, 8, 64, 4096), (70001, 16, 3, 100)])
@pytest.mark.parametrize("k", [1, 2])
def test_every_row_of_the_buffer_is_written_once(pkg, S, M, E, C, k):
    """Rows of tokens are copies, all others zero; with rows_at_used the rows below used_capacity stay as they were."""
    ops = pkg.ops
    data, logits = make_inputs(S + E, S, M, E, zipf_bias=True)
    d_data, d_gate = rows_to_torch(data, "bf16"), dev(logits)
    used0 = torch.arange(E, dtype=torch.int32, device="cuda") % 40
    for used, at_used in ((None, False), (used0, False), (used0, True)):
        first = ops.moe_encode(d_data, d_gate, used, top_k=k, gate_is_logits=True, capacity=C, rows_at_used=at_used)
        outs = [torch.full_like(t, 7) if t.dtype != torch.uint64 else torch.full((E,), 7, dtype=torch.int64, device="cuda") for t in first]
        got = ops.moe_encode(d_data, d_gate, used, top_k=k, gate_is_logits=True, capacity=C, rows_at_used=at_used, out=outs)
        idx, loc = (got[1][i].long() for i in (0, 1))
        want = torch.zeros_like(got[4])
        if at_used:
            want[torch.arange(C, device="cuda")[None, :] < used[:, None].clamp(max=C)] = 7
            loc = loc + used[idx.clamp(min=0)]
        keep = (idx >= 0) & (loc < C)
        if used is not None and not at_used:
            keep &= loc < C - used[idx.clamp(min=0)]
        tok = torch.arange(k * S, device="cuda") % S
        want[idx[keep], loc[keep]] = d_data[tok[keep]]
        assert torch.equal(got[4].view(torch.int16), want.view(torch.int16)), (used is not None, at_used)


# 383 granules, 384, 512 (every lane has two), 513; few slots (walked) and many (looked up)
@pytest.mark.parametrize("M,dt", [(3064, "bf16"), (3072, "bf16"), (4096, "f16"), (4104, "bf16"), (2048, "f32"), (4099, "bf16")])
@pytest.mark.parametrize("S,k", [(1, 1), (130, 2), (4200, 2), (8200, 1)])
@pytest.mark.parametrize("spare", [0, 3000])  # rows nobody owns: 3000 per expert put the pass beyond the cache
def test_decode_gradient_of_wide_rows(pkg, M, dt, S, k, spare):
    """Rows bit for bit, 16-bit ones to one unit in the last place (a product may be rounded once instead of to fp32 first); the
    dot products within 40 roundings of the sum of the products' sizes (chains of eight products and of up to four granules, a tree
    over 256 lanes)."""
    ops, E = pkg.ops, 5
    data, logits = make_inputs(S + M, S, 4, E, zipf_bias=True)
    enc = mo.moe_encode_top2 if k == 2 else mo.moe_encode
    g, il, used, _, disp = enc(data, logits, np.zeros(E, np.int32), 0.7, gate_is_logits=True, fast_scatter=True)
    C = disp.shape[1] + spare
    rng = np.random.default_rng(M)
    dy, rows = (rng.standard_normal(shape, dtype=np.float32) for shape in ((S, M), (E, C, M)))
    dy_o, rows_o = rows_as_oracle(dy, dt), rows_as_oracle(rows, dt)
    d_rows, d_g = ops.moe_decode_grad(rows_to_torch(dy, dt), rows_to_torch(rows, dt), dev(g), dev(il), top_k=k)
    want = rows_to_torch(mo.moe_decode_dx(dy_o, g, il, E, C, k), dt)
    assert torch.equal(d_rows, want) if dt == "f32" else ulp_distance(d_rows, want) <= 1
    got = to_np(d_g).astype(np.float64)
    for i in range(k * S):
        e, l = il[0][i], il[1][i]
        if e < 0 or l < 0:
            assert got[i] == 0
            continue
        terms = dy_o[i % S].astype(np.float64) * rows_o[e, l]
        assert abs(got[i] - terms.sum()) <= 40 * 2.0 ** -24 * np.abs(terms).sum()
