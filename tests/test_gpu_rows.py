"""Row movers at the row lengths where their pieces can go wrong: rows of less than 16 bytes (moved by elements), rows
that end inside a 16-byte granule (the last one drawn back over the one before), rows of whole granules at addresses that
are not aligned to them.  Against the oracle: rows bit-exact, 16-bit products within one unit in the last place, dot
products within 1e-5 of sum|a_i * b_i| (fp32 sums of up to 1003 terms in another order)."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as mo
from tests.gpu_util import dev, make_inputs, rows_as_oracle, rows_to_torch, to_np, ulp_distance

pytestmark = pytest.mark.gpu

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _at(t, offset):
    """t's values in memory that starts `offset` elements into an allocation."""
    buf = torch.empty(t.numel() + offset, dtype=t.dtype, device=t.device)
    view = buf[offset:].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("dt,M,offset", [("f32", 3, 0), ("f32", 4, 1), ("f32", 5, 0), ("f32", 255, 0), ("f32", 258, 3), ("bf16", 7, 0),
                                         ("bf16", 8, 1), ("bf16", 9, 0), ("f16", 15, 1), ("bf16", 513, 0), ("f16", 1003, 0), ("bf16", 512, 3)])
@pytest.mark.parametrize("k", [1, 2])
def test_rows_of_any_length_and_alignment(pkg, dt, M, offset, k):
    ops = pkg.ops
    S, E, cf = 300, 6, 0.7
    data, logits = make_inputs(M + k, S, M, E, zipf_bias=True)
    x = rows_as_oracle(data, dt)
    enc = mo.moe_encode_top2 if k == 2 else mo.moe_encode
    g, il, used, _, disp = enc(x, logits, np.zeros(E, np.int32), cf, gate_is_logits=True, fast_scatter=True)
    C = disp.shape[1]
    assert (il[0] < 0).any() and (used < C).any()
    rng = np.random.default_rng(M)
    outs = [torch.empty(k * S, device="cuda"), torch.empty((2, k * S), dtype=torch.int32, device="cuda"),
            torch.empty(E, dtype=torch.int32, device="cuda"), torch.empty(E, dtype=torch.int64, device="cuda"),
            _at(torch.full((E, C, M), 7.0, dtype=_TORCH[dt], device="cuda"), offset)]
    d_g, d_il, _, _, d_disp = ops.moe_encode(_at(rows_to_torch(data, dt), offset), dev(logits), None, cf, top_k=k, gate_is_logits=True, out=outs)
    np.testing.assert_array_equal(to_np(d_il), il)
    np.testing.assert_array_equal(to_np(d_disp), disp)

    def near(got, want):                       # products and sums of two, rounded once
        if dt == "f32":
            np.testing.assert_array_equal(to_np(got), want)
        else:
            assert ulp_distance(got, torch.from_numpy(want).to(_TORCH[dt]).cuda()) <= 1

    buf = rows_as_oracle(rng.standard_normal((E, C, M), dtype=np.float32), dt)
    tok = rows_as_oracle(rng.standard_normal((S, M), dtype=np.float32), dt)
    d_buf, d_tok = _at(rows_to_torch(buf, dt), offset), _at(rows_to_torch(tok, dt), offset)
    w = to_np(d_g)                              # the GPU's own combine weights, so that products compare exactly
    out = _at(torch.full((S, M), 7.0, dtype=_TORCH[dt], device="cuda"), offset)
    rows = _at(torch.full((E, C, M), 7.0, dtype=_TORCH[dt], device="cuda"), offset)
    near(ops.moe_decode(d_buf, d_g, d_il, top_k=k, out=out), mo.moe_decode(buf, w, il, k=k))
    near(ops.moe_encode_dx(d_buf, d_il, top_k=k, out=out), mo.moe_encode_dx(buf, il, k))
    near(ops.moe_decode_dx(d_tok, d_g, d_il, E, C, top_k=k, out=rows), mo.moe_decode_dx(tok, w, il, E, C, k))
    dg = to_np(ops.moe_decode_dg(d_tok, d_buf, d_il, top_k=k))
    bound = mo.moe_decode_dg(np.abs(tok), np.abs(buf), il, k)
    assert (np.abs(dg - mo.moe_decode_dg(tok, buf, il, k)) <= 1e-5 * bound).all()
    d_rows, d_w = ops.moe_decode_grad(d_tok, d_buf, d_g, d_il, top_k=k, out=(torch.full_like(rows, 7.0), torch.full_like(d_g, 7.0)))
    near(d_rows, mo.moe_decode_dx(tok, w, il, E, C, k))
    assert (np.abs(to_np(d_w) - mo.moe_decode_dg(tok, buf, il, k)) <= 1e-5 * bound).all() and not to_np(d_w)[il[0] < 0].any()
    if k == 1:                                  # partition buffers: the same rows, the tail zero-filled again
        merged = ops.moe_redispatch([d_disp], [d_il], out=rows)
        np.testing.assert_array_equal(to_np(merged), disp)


@pytest.mark.parametrize("S,k,M,dt,gdt", [(7, 1, 64, "f32", "f32"), (4096, 2, 24, "bf16", "bf16"), (4097, 2, 24, "bf16", "f32"), (8192, 1, 8, "f16", "f16"),
                                          (5000, 1, 24, "bf16", "bf16"), (5001, 1, 24, "f32", "f16"), (3450, 2, 24, "f32", "f32"), (3451, 2, 360, "bf16", "bf16"),
                                          (4096, 1, 384, "bf16", "bf16"), (4097, 1, 192, "f32", "f16"), (2048, 2, 520, "bf16", "f32"),
                                          (8193, 1, 8, "f32", "bf16"), (700, 2, 512, "bf16", "f32"), (700, 2, 1024, "f32", "f32"), (300, 2, 4100, "bf16", "f16")])
def test_decode_gradients_in_one_pass(pkg, S, k, M, dt, gdt):
    """moe_decode_grad against the two ops it stands for: rows bit for bit (the same products and roundings), weights within
    1e-5 of sum|a_i * b_i| plus one rounding to the gate's type.  Sizes on both sides of the slots up to which the
    workgroups that clear unowned rows walk the slots themselves; rows of one wave, of several, and longer than a pass."""
    ops = pkg.ops
    E = 5
    gen = torch.Generator(device="cuda").manual_seed(S + M)
    normal = lambda *shape: torch.empty(shape, device="cuda").normal_(generator=gen).to(_TORCH[dt])  # noqa: E731
    logits = torch.empty((S, E), device="cuda").normal_(generator=gen) + torch.arange(E, device="cuda")
    g, il, _, _, disp = ops.moe_encode(normal(S, M), logits.to(_TORCH[gdt]), None, 0.8, top_k=k, gate_is_logits=True)
    C = disp.shape[1]
    data, dy = normal(E, C, M), normal(S, M)
    d_data, d_gate = ops.moe_decode_grad(dy, data, g, il, top_k=k, out=(torch.full_like(data, 7.0), torch.full_like(g, 7.0)))
    assert torch.equal(d_data, ops.moe_decode_dx(dy, g, il, E, C, top_k=k))
    want = ops.moe_decode_dg(dy, data, il, top_k=k)
    bound = ops.moe_decode_dg(dy.abs(), data.abs(), il, top_k=k)
    ulp = {"f32": 0.0, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}[gdt]
    assert d_gate.dtype == _TORCH[gdt]
    assert bool(((d_gate.float() - want).abs() <= 1e-5 * bound + ulp * want.abs()).all())


@pytest.mark.parametrize("S", [1, 1023, 8193, 16384, 16385])
@pytest.mark.parametrize("P,E", [(1, 1), (3, 70), (2, 512)])
def test_partition_counts_at_the_limits_of_one_workgroup(pkg, S, P, E):
    """moe_merge_masks on partitions that one workgroup counts alone (up to 16384 tokens) and on longer ones; exact."""
    rng = np.random.default_rng(S + E)
    masks = []
    for _ in range(P):
        e = rng.integers(-1, E, S).astype(np.int32)
        masks.append(np.stack([e, rng.integers(0, 50, S).astype(np.int32)]))
    got = to_np(pkg.ops.moe_merge_masks([dev(m) for m in masks], E))
    before = np.zeros(E, np.int64)
    for p, (e, l) in enumerate(masks):
        part = got[:, p * S:(p + 1) * S]
        np.testing.assert_array_equal(part[0], e)
        np.testing.assert_array_equal(part[1], np.where(e >= 0, l + before[np.maximum(e, 0)], -1))
        before += np.bincount(e[e >= 0], minlength=E)


@pytest.mark.parametrize("dt,M,offset", [("f32", 5, 0), ("f32", 9, 0), ("f32", 255, 0), ("f32", 12, 1), ("bf16", 9, 0), ("bf16", 15, 1), ("f16", 1003, 0),
                                         ("bf16", 64, 3)])
def test_weight_gradients_of_rows_with_an_infinity(pkg, dt, M, offset):
    """One infinity per row, at every place among the last 24 elements (two granules and more: also those that the
    drawn-back granule reads a second time), in the token row or in the expert's.  The other factor is not zero, so the
    weight gradient is that infinity with the factor's sign, from moe_decode_dg and moe_decode_grad alike."""
    ops = pkg.ops
    S = min(M, 24)
    gen = torch.Generator(device="cuda").manual_seed(M)
    rows = lambda: (torch.rand((S, M), device="cuda", generator=gen) + 0.5) * (torch.randint(0, 2, (S, M), device="cuda", generator=gen) * 2 - 1)  # noqa: E731
    il = torch.stack([torch.zeros(S, dtype=torch.int32, device="cuda"), torch.arange(S, dtype=torch.int32, device="cuda")])
    weights = torch.ones(S, device="cuda")
    at = torch.arange(M - S, M, device="cuda")
    here = torch.arange(S, device="cuda")
    for infinite in (0, 1):
        pair = [rows(), rows()]
        pair[infinite][here, at] = float("inf")
        want = pair[1 - infinite][here, at].sign() * float("inf")
        tok, buf = (_at(x.to(_TORCH[dt]), offset) for x in pair)
        assert torch.equal(ops.moe_decode_dg(tok, buf.view(1, S, M), il), want)
        assert torch.equal(ops.moe_decode_grad(tok, buf.view(1, S, M), weights, il)[1], want)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("M", [5, 8, 24, 64, 120, 256, 264, 512, 9, 60, 100, 257, 383, 500, 511])
def test_weight_gradients_are_sums_of_granules(pkg, dt, M):
    """Rows of up to 64 granules: a weight gradient is the sum over the granules' own sums, added up as a tree, however many
    granules a lane takes.  Products of 16-bit values are exact in fp32, so that the order of the additions says every bit:
    inside a granule in order where rows are whole granules, in pairs where they end inside one."""
    ops = pkg.ops
    S = 64
    gen = torch.Generator(device="cuda").manual_seed(M)
    tok, buf = (torch.empty((S, M), device="cuda").normal_(generator=gen).to(_TORCH[dt]) for _ in range(2))
    il = torch.stack([torch.zeros(S, dtype=torch.int32, device="cuda"), torch.arange(S, dtype=torch.int32, device="cuda")])
    prod = to_np(tok) * to_np(buf)
    if M < 8:
        parts = prod                                             # a lane per element
    else:
        n = (M + 7) // 8
        padded = np.zeros((S, n * 8), np.float32)
        padded[:, :M] = prod
        if M % 8:                                                # drawn back: zeros in front
            padded[:, n * 8 - 8:] = 0
            padded[:, n * 8 - (M - (n - 1) * 8):] = prod[:, (n - 1) * 8:]
        p = padded.reshape(S, n, 8)
        if M % 8 == 0:
            parts = p[:, :, 0].copy()
            for i in range(1, 8):
                parts = parts + p[:, :, i]
        else:
            q = p[:, :, 0::2] + p[:, :, 1::2]
            parts = (q[:, :, 0] + q[:, :, 1]) + (q[:, :, 2] + q[:, :, 3])
    lanes = np.zeros((S, 64), np.float32)
    lanes[:, :parts.shape[1]] = parts
    o = 32
    while o:
        lanes = lanes[:, :o] + lanes[:, o:2 * o]
        o //= 2
    want = lanes[:, 0]
    np.testing.assert_array_equal(to_np(ops.moe_decode_dg(tok, buf.view(1, S, M), il)), want)
    np.testing.assert_array_equal(to_np(ops.moe_decode_grad(tok, buf.view(1, S, M), torch.ones(S, device="cuda"), il)[1]), want)


def test_decode_gradient_outputs_are_checked(pkg):
    """moe_decode_grad writes E * C * M elements and k * S weights: outputs that do not hold them are refused on the host."""
    ops = pkg.ops
    S, E, C, M = 8, 2, 4, 16
    data, dy, gate = torch.ones((E, C, M), device="cuda"), torch.ones((S, M), device="cuda"), torch.ones(S, device="cuda")
    il = torch.stack([torch.arange(S, device="cuda") // C, torch.arange(S, device="cuda") % C]).int()
    rows, weights = torch.empty_like(data), torch.empty_like(gate)
    for out in ((rows[:, :3].contiguous(), weights), (rows.half(), weights), (rows.transpose(0, 1).contiguous().transpose(0, 1), weights),
                (rows.cpu(), weights), (rows, weights[:7]), (rows, weights.half()), (rows, torch.empty(2 * S, device="cuda")[::2]),
                (rows, weights.cpu())):
        with pytest.raises(ValueError):
            ops.moe_decode_grad(dy, data, gate, il, out=out)
    ops.moe_decode_grad(dy, data, gate, il, out=(rows, weights))
    assert bool((rows == 1).all()) and bool((weights == M).all())


@pytest.mark.parametrize("S,E", [(16384, 1), (16384, 512), (16383, 64), (40, 512)])
@pytest.mark.parametrize("kind", ["one", "two", "sorted"])
def test_partition_counts_of_few_experts(pkg, S, E, kind):
    """Tokens that meet in one counter, in two, or expert by expert in token order: every lane counts in a copy of its own
    modulo their number.  The second partition's locations are the first one's counts; exact."""
    e = {"one": np.full(S, E - 1), "two": np.arange(S) % 2 * (E - 1), "sorted": np.arange(S) * E // S}[kind].astype(np.int32)
    e[::13] = -1
    mask = dev(np.stack([e, np.zeros(S, np.int32)]))
    got = to_np(pkg.ops.moe_merge_masks([mask, mask], E))
    np.testing.assert_array_equal(got[0], np.concatenate([e, e]))
    counts = np.bincount(e[e >= 0], minlength=E)
    np.testing.assert_array_equal(got[1, S:], np.where(e >= 0, counts[np.maximum(e, 0)], -1))


@pytest.mark.parametrize("dt,M,S", [("bf16", 768, 1365), ("bf16", 768, 1366), ("f32", 520, 1100), ("bf16", 1003, 1100), ("f16", 520, 2017), ("f32", 256, 2049), ("bf16", 24, 43691)])
@pytest.mark.parametrize("k", [1, 2])
def test_gathers_of_one_and_two_granules_per_lane(pkg, dt, M, S, k):
    """Lanes take one or two granules of a row by the number of granules in all (131072) and by whether a row fills its
    lanes: sizes on both sides of the line, rows of 96 and 126 granules among them.  Bit for bit in fp32, 16-bit sums
    within one unit in the last place."""
    ops = pkg.ops
    E = 4
    data, logits = make_inputs(S + M, S, M, E)
    x = rows_as_oracle(data, dt)
    d_g, d_il, _, _, _ = ops.moe_encode(rows_to_torch(data[:, :1], dt), dev(logits), None, 0.9, top_k=k, gate_is_logits=True)
    C = ops.moe_capacity(S, E, 0.9 * k)
    il, w = to_np(d_il), to_np(d_g)
    buf = rows_as_oracle(np.random.default_rng(S).standard_normal((E, C, M), dtype=np.float32), dt)
    d_buf = rows_to_torch(buf, dt)

    def near(got, want):
        if dt == "f32":
            np.testing.assert_array_equal(to_np(got), want)
        else:
            assert ulp_distance(got, torch.from_numpy(want).to(_TORCH[dt]).cuda()) <= 1

    near(ops.moe_decode(d_buf, d_g, d_il, top_k=k), mo.moe_decode(buf, w, il, k=k))
    near(ops.moe_encode_dx(d_buf, d_il, top_k=k), mo.moe_encode_dx(buf, il, k))
    near(ops.moe_decode_dx(rows_to_torch(data, dt), d_g, d_il, E, C, top_k=k), mo.moe_decode_dx(x, w, il, E, C, k))
