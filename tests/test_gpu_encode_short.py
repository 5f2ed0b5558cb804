"""moe_encode of few tokens (routing and row movement in one kernel up to 256 tokens, in two up to 8192) against the separate
kernels, which scan_lookback=True asks for, bit for bit, and against the oracle, at the edges of its tiles, workgroups and rules."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import moe_oracle as mo
from tests.gpu_util import TORCH_DT, dev, make_inputs, rows_as_oracle, rows_to_torch, to_np

pytestmark = pytest.mark.gpu

# (S, M, E): one token, ends of a wave and of a tile, one token more; rows of less than a granule, of one and a bit, of whole
# granules, of more than two per lane; as many tiles as there may be; the most experts a tile of tokens may have
SHAPES = [(1, 8, 2), (63, 3, 5), (64, 1024, 8), (255, 1003, 60), (256, 4200, 128), (32, 64, 512), (256, 8, 129), (257, 5, 3), (300, 4096, 7),
          (513, 24, 64), (6000, 77, 33), (8192, 512, 8), (8192, 16, 64), (8000, 2, 128)]


@pytest.mark.parametrize("S,M,E", SHAPES)
@pytest.mark.parametrize("k", [1, 2])
def test_short_encodes_are_what_the_separate_kernels_give(pkg, S, M, E, k):
    ops = pkg.ops
    for i, dt in enumerate(("f32", "bf16", "f16")):
        data, logits = make_inputs(S + M + k + i, S, M, E, zipf_bias=True, ties=i == 1)
        rows, logits_in = rows_as_oracle(data, dt), logits.astype(np.float32)
        d_data = rows_to_torch(data, dt)
        used0 = (np.arange(E) % 3).astype(np.int32)
        noise = torch.randn(S, E, device="cuda").to(TORCH_DT[dt]) if k == 2 and i == 0 else None
        for used, logit, tail, at_used, gdt in ((None, True, True, False, "f32"), (used0, False, True, False, dt), (used0, True, True, True, "f32"),
                                                (used0, True, False, False, "f32"), (None, True, False, False, dt)):
            gate = (dev(logits_in) if logit else torch.softmax(dev(logits_in), 1)).to(TORCH_DT[gdt])
            n = noise.to(gate.dtype) if noise is not None else None
            args = dict(capacity_factor=0.75, top_k=k, gate_is_logits=logit, zero_tail=tail, gate2_noise=n, rows_at_used=at_used)
            d_used = None if used is None else dev(used)
            first = ops.moe_encode(d_data, gate, d_used, **args)
            outs = [[torch.full_like(t, 7) if t.dtype != torch.uint64 else torch.full((E,), 7, dtype=torch.int64, device="cuda") for t in first]
                    for _ in range(2)]
            got = ops.moe_encode(d_data, gate, d_used, out=outs[0], **args)
            want = ops.moe_encode(d_data, gate, d_used, out=outs[1], scan_lookback=True, **args)
            for a, b in zip(got, want):
                assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), (dt, used is not None, logit, tail, at_used, gdt)
        if k == 1:
            ref = mo.moe_encode(rows, logits_in, used0, 0.75, gate_is_logits=True, fast_scatter=True)
        else:
            ref = mo.moe_encode_top2(rows, logits_in, used0, 0.75, gate_is_logits=True, fast_scatter=True)
        got = ops.moe_encode(d_data, dev(logits_in), dev(used0), 0.75, top_k=k, gate_is_logits=True)
        for j in (1, 2, 3, 4):
            np.testing.assert_array_equal(to_np(got[j]), ref[j])
        np.testing.assert_allclose(to_np(got[0]), ref[0], rtol=1e-5)


# one and two tokens more than workgroups there may be, of one and of two tokens; rows of either side of the limits of 36 MB (below 32
# experts) and 12 MB
@pytest.mark.parametrize("S,M,E", [(1701, 1500, 6), (3402, 772, 5), (2001, 1540, 3), (2305, 4096, 31), (2305, 4096, 32)])
@pytest.mark.parametrize("k", [1, 2])
def test_short_encodes_at_the_limits_of_their_rule(pkg, S, M, E, k):
    test_short_encodes_are_what_the_separate_kernels_give(pkg, S, M, E, k)


def test_used_capacity_updated_in_place(pkg):
    """used_capacity as input and output of one call (rows that feed moe_redispatch): the separate kernels take it, as before."""
    ops = pkg.ops
    S, M, E = 200, 32, 6
    data, logits = make_inputs(9, S, M, E)
    used = dev(np.full(E, 2, np.int32))
    want = ops.moe_encode(dev(data), dev(logits), used.clone(), 1.0, gate_is_logits=True, zero_tail=False)
    outs = [torch.zeros_like(want[0]), torch.zeros_like(want[1]), used, torch.zeros(E, dtype=torch.int64, device="cuda"), torch.zeros_like(want[4])]
    got = ops.moe_encode(dev(data), dev(logits), used, 1.0, gate_is_logits=True, zero_tail=False, out=outs)
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])


@pytest.mark.parametrize("S", [100, 3000])
def test_short_top1_on_memory_that_was_never_set_up(pkg, S):
    """As the look-back form does: every output marked, the buffer cleared, the error word set; whole again after the set-up."""
    lib, capi, ops = pkg.capi.load(), pkg.capi, pkg.ops
    M, E = 8, 8
    data, logits = make_inputs(3, S, M, E)
    d_data, d_gate = dev(data), dev(logits)
    Cap, nws = ops.moe_capacity(S, E, 1.0), int(lib.lancet_moe_encode_workspace_bytes(S, E, 1))
    ws = torch.full((nws,), 0xff, dtype=torch.uint8, device="cuda")
    outs = (torch.ones(S, device="cuda"), torch.zeros((2, S), dtype=torch.int32, device="cuda"), torch.zeros(E, dtype=torch.int32, device="cuda"),
            torch.ones(E, dtype=torch.int64, device="cuda"), torch.ones((E, Cap, M), device="cuda"))
    p = lambda t: t.data_ptr()
    call = lambda: lib.lancet_moe_encode(p(d_data), p(d_gate), None, None, S, M, E, Cap, 1, capi.F32, capi.F32, capi.GATE_IS_LOGITS,
                                         *[p(t) for t in outs], p(ws), nws, None)
    assert call() == 0
    torch.cuda.synchronize()
    err = C.c_int(0)
    assert (to_np(outs[1]) == -1).all() and (to_np(outs[2]) == -1).all() and not to_np(outs[0]).any()
    assert not to_np(outs[3]).any() and not to_np(outs[4]).any()
    assert lib.lancet_scan_workspace_error(p(ws), None, C.byref(err)) == 0 and err.value == 1
    assert lib.lancet_scan_workspace_init(p(ws), nws, None) == 0 and call() == 0
    want = mo.moe_encode(data, logits, np.zeros(E, np.int32), 1.0, gate_is_logits=True, fast_scatter=True)
    np.testing.assert_array_equal(to_np(outs[1]), want[1])
    np.testing.assert_array_equal(to_np(outs[4]), want[4])


# lanes that are full, five in eight, fewer (logits of more than half a tile are walked then), rows that end inside a granule
@pytest.mark.parametrize("S", [1, 15, 17, 64, 65, 128, 129, 257, 700])
@pytest.mark.parametrize("E,gdt", [(32, "f32"), (56, "f32"), (61, "f32"), (64, "f32"), (76, "f32"), (80, "f32"), (100, "f32"), (125, "f32"), (129, "f32"), (132, "f32"),
                                   (256, "f32"), (96, "bf16"), (128, "bf16"), (249, "bf16"), (101, "f16"), (272, "f16"), (512, "bf16")])
def test_selection_by_sixteen_waves(pkg, S, E, gdt):
    """Rows whose selection sixteen waves share, and those beside them: choices against the oracle's on the rounded gate (massive ties of 16-bit values
    included), rows with a NaN and rows of -inf against the same rows in a batch that sixteen waves do not take (noise of zero
    sends a top-2 call to the row-by-row walk)."""
    ops = pkg.ops
    data, logits = make_inputs(S + E, S, 4, E, ties=S % 2 == 1)
    gate = dev(logits).to(TORCH_DT[gdt])
    rounded = gate.float().cpu().numpy()
    for k in (1, 2):
        for is_logits in (True, False):
            sel = mo.select_topk(rounded, k, gate_is_logits=is_logits)[0]
            got = ops.moe_encode(dev(data), gate, None, float(E), top_k=k, gate_is_logits=is_logits)
            np.testing.assert_array_equal(to_np(got[1])[0], np.concatenate([sel[j] for j in range(k)]))
    odd = gate.clone()
    odd[::3, E // 2] = float("nan")
    odd[1::3] = float("-inf")
    for is_logits in (True, False):
        a = ops.moe_encode(dev(data), odd, None, float(E), top_k=2, gate_is_logits=is_logits)
        b = ops.moe_encode(dev(data), odd, None, float(E), top_k=2, gate_is_logits=is_logits, gate2_noise=torch.zeros_like(odd))
        np.testing.assert_array_equal(to_np(a[1]), to_np(b[1]))


# buffers far larger than the load: turns of one expert (E = 2), of all (more experts than workgroups clear), an end of a turn off
# the expert's last row, rows of less than a granule; a few tiles; more rows than one workgroup per turn could be launched for
@pytest.mark.parametrize("S,M,E,C", [(1, 8, 2, 5000), (64, 24, 128, 700), (256, 1024, 128, 33), (256, 4104, 3, 300), (20, 3, 512, 129),
                                     (256, 1, 128, (1 << 19) + 5), (300, 8, 60, 4096), (2000, 1024, 5, 2500), (8192, 2, 64, 9000)])
@pytest.mark.parametrize("k", [1, 2])
def test_tails_of_buffers_larger_than_the_load(pkg, S, M, E, C, k):
    """Every row of the buffer as the separate kernels leave it, in memory that held something else."""
    ops = pkg.ops
    data, logits = make_inputs(S + C, S, M, E, zipf_bias=True)
    d_data, gate = rows_to_torch(data, "bf16"), dev(logits)
    used0 = torch.arange(E, dtype=torch.int32, device="cuda") % 3
    for used, at_used in ((None, False), (used0, False), (used0, True)):
        got, want = (ops.moe_encode(d_data, gate, used, top_k=k, gate_is_logits=True, capacity=C, rows_at_used=at_used, scan_lookback=separate,
                                    out=[torch.empty(k * S, device="cuda"), torch.empty((2, k * S), dtype=torch.int32, device="cuda"),
                                         torch.empty(E, dtype=torch.int32, device="cuda"), torch.empty(E, dtype=torch.int64, device="cuda"),
                                         torch.full((E, C, M), 7.0, dtype=torch.bfloat16, device="cuda")]) for separate in (False, True))
        for a, b in zip(got, want):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
