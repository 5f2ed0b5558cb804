"""Calls of several threads on one stream: the scan workspace kept for the stream is theirs in turn."""
import threading

import pytest
import torch

from tests.gpu_util import dev, make_inputs

pytestmark = pytest.mark.gpu


def _calls(pkg, data, gate):
    """What a thread runs: short and long encodes, batch-prioritised ones with and without the scan, the routing alone, training."""
    ops, grad = pkg.ops, pkg.grad
    d, g = data.clone().requires_grad_(True), gate.clone().requires_grad_(True)
    return [lambda: ops.moe_encode(data[:2000], gate[:2000], None, 1.0, gate_is_logits=True),
            lambda: ops.moe_encode(data, gate, None, 1.0, top_k=2, gate_is_logits=True),
            lambda: ops.moe_encode_batch_prioritized(data[:1500], gate[:1500], 1, 0, 1.0),
            lambda: ops.moe_encode_batch_prioritized(data, gate, 2, 1, 1.0),
            lambda: ops.moe_route(gate, None, data.shape[1], 1.0, gate_is_logits=True),
            lambda: [t.detach() for t in grad.moe_encode(d, g, None, 1.0, top_k=2, gate_is_logits=True)]]


def test_threads_on_one_stream(pkg):
    S, M, E, rounds = 12000, 16, 16, 40
    inputs = [tuple(map(dev, make_inputs(seed, S, M, E, zipf_bias=True))) for seed in (1, 2, 3)]
    want = [[call() for call in _calls(pkg, *x)] for x in inputs]
    got, errors, start = [[] for _ in inputs], [], threading.Barrier(len(inputs))

    def run(i):
        try:
            calls = _calls(pkg, *inputs[i])
            start.wait()
            for _ in range(rounds):
                got[i].append([call() for call in calls])
        except BaseException as e:   # noqa: B902 - handed to the test's thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(inputs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for i in range(len(inputs)):
        for one in got[i]:
            for a, b in zip(one, want[i]):
                for x, y in zip(a, b):
                    assert torch.equal(x.contiguous().view(torch.uint8), y.contiguous().view(torch.uint8))
