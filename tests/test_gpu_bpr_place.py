"""moe_encode_batch_prioritized of up to 2048 tokens (the expert's workgroup also places its tokens) against the scan that
scan_lookback=True asks for, bit for bit, and against the oracle."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as mo
from tests.gpu_util import TORCH_DT, dev, make_inputs, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S0,E,P", [(1, 3, 1), (255, 4, 1), (256, 16, 2), (257, 5, 3), (1000, 64, 4), (2000, 3, 2), (1999, 300, 1), (2048, 2, 1),
                                    (2048, 64, 8), (2049, 7, 1), (5000, 3, 2)])
@pytest.mark.parametrize("cf", [0.0, 0.5, 1.25, 400.0])
@pytest.mark.parametrize("gdt", ["f32", "bf16"])
def test_places_by_expert_are_the_scans(pkg, S0, E, P, cf, gdt):
    ops = pkg.ops
    M = 8
    data, logits = make_inputs(S0 + E, S0, M, E, zipf_bias=True, ties=P == 2)
    gate = torch.softmax(dev(logits), 1).to(TORCH_DT[gdt])           # 16-bit priorities tie massively
    rounded = gate.float().cpu().numpy()
    d_data = dev(data)
    for pid in {0, P // 2, P - 1}:
        if cf * (S0 // P) / E > 2000:
            cf = 2000.0 * E / (S0 // P)                                # everything fits
        got = ops.moe_encode_batch_prioritized(d_data, gate, P, pid, cf)
        want = ops.moe_encode_batch_prioritized(d_data, gate, P, pid, cf, scan_lookback=True)
        for a, b in zip(got, want):
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
        ref = mo.moe_encode_bpr(data, rounded, P, pid, cf, fast_scatter=True)
        for i in (1, 2, 3, 4):
            np.testing.assert_array_equal(to_np(got[i]), ref[i])
