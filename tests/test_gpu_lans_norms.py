"""Gradient norms of the tensors that LANS sweeps: summed by the step's first kernel up to 6144 chunks, by a sweep of their own
beyond, with the same bits."""
import numpy as np
import pytest
import torch

from tests.gpu_util import TORCH_DT

pytestmark = pytest.mark.gpu


# chunks that do and do not fill a workgroup of four, one element of a chunk, tensors small enough to be taken whole
@pytest.mark.parametrize("numels", [[3 * 8192], [4 * 8192 + 1, 700], [20011, 5 * 8192, 1, 8192 * 9 + 4095], [0, 16384 * 3 + 2, 5]])
@pytest.mark.parametrize("gdt", ["f32", "bf16", "f16"])
def test_norms_are_the_same_by_either_kernel(pkg, numels, gdt):
    ops, capi = pkg.ops, pkg.capi
    big = 6144 * 8192                                     # with any other chunk: one too many for the first kernel
    gen = torch.Generator(device="cuda").manual_seed(len(numels))
    normal = lambda n, std: torch.empty(n, device="cuda").normal_(0.0, std, generator=gen)  # noqa: E731
    g = [normal(n, 1e-2).to(TORCH_DT[gdt]) for n in numels]
    state = [[normal(n, 0.02) for n in numels] for _ in range(2)] + [[normal(n, 1e-3).square_() for n in numels]]
    results = []
    for extra in (0, big):
        mine = [[t.clone() for t in lst] for lst in state]
        plan = ops.LansPlan(numels + [extra], schedule=capi.LANS_SWEEPS)
        pad = [torch.zeros(extra, dtype=g[0].dtype, device="cuda")] + [torch.zeros(extra, device="cuda") for _ in range(3)]
        plan.step(g + [pad[0]], mine[0] + [pad[1]], mine[1] + [pad[2]], mine[2] + [pad[3]], 1,
                  capi.LansHyper(1e-3, 0.9, 0.999, 1e-6, 1, 0.01, 1, 1, 1))
        assert plan.error() == 0
        results.append([plan.norms()[:, :len(numels)].clone()] + [t for lst in mine for t in lst])
        plan.close()
    for a, b in zip(*results):
        assert torch.equal(a, b)
    want = np.array([float(t.double().norm()) for t in g])
    # a chunk's squares in fp32: 32 per thread one after the other, a tree over 256 threads; their sum in double
    np.testing.assert_allclose(results[0][0][0].cpu().numpy(), want, rtol=45 * 2.0 ** -24)
