"""Gradient wiring of the MoE dispatch operators, as RAF registers it (src/op/grad/moe.cc:30-93), for callers
that differentiate with torch.autograd.

  moe_encode, moe_encode_batch_prioritized (MoeEncodeGrad, :30-58):
      d data = moe_encode_dx(dy[4], y[1]);  d gate = moe_encode_dg(dy[0], y[1], E);  used_capacity: none
  moe_decode (MoeDecodeGrad, :60-90):
      d data = moe_decode_dx(dy, gate, indices_locations, E, C);  d gate = moe_decode_dg(dy, data, indices_locations)
      (moe_decode_grad: both in one pass over the rows)

The reference differentiates the one form of the op it has: top-1 on a gate that holds probabilities.  The forms
this library adds (top_k = 2 with GShard's normalised combine weights, docker/resources/sharded_moe.py:253-324, and
the softmax fused into the op, gate_is_logits) do more to a gate value than select it, so their gate gradient is
    d gate = moe_encode_dgate(dy[0], gate, y[1])
which goes back through the normalisation and the softmax (ops.moe_encode_dgate); moe_decode's rules take top_k.
Every gradient is computed by the HIP backward kernels; nothing here falls back to torch arithmetic.  The rules are native
autograd nodes (torch_host/torch_host.cc): forward-mode differentiation and torch.func transforms are refused, as they are of
any function with a backward rule alone.
"""
from . import capi, ops


def moe_encode(data, gate, used_capacity=None, capacity_factor=1.0, top_k=1, gate_is_logits=False, gate2_noise=None,
               capacity=None):
    """Differentiable raf.op.moe_encode: gradients flow to data (through dispatched) and to gate (through gates_s);
    with top_k = 2 or gate_is_logits the gate gradient goes back through the normalisation of the combine weights
    and through the fused softmax.  gate2_noise only moves the second choice and gets no gradient."""
    return capi.host().moe_encode_diff(data, gate, gate2_noise, used_capacity, float(capacity_factor),
                                       None if capacity is None else int(capacity), int(top_k), ops._flags(gate_is_logits, True),
                                       None, None)


def moe_encode_batch_prioritized(data, gate, n_partitions=1, partition_id=0, capacity_factor=1.0, gate_is_logits=False):
    """Differentiable raf.op.moe_encode_batch_prioritized (same gradient as moe_encode, src/op/grad/moe.cc:58)."""
    return capi.host().moe_encode_diff(data, gate, None, None, float(capacity_factor), None, 1, ops._flags(gate_is_logits, True),
                                       int(n_partitions), int(partition_id))


def moe_decode(data, gate, indices_locations, top_k=1):
    """Differentiable raf.op.moe_decode: gradients flow to data (expert outputs) and to gate (gates_s)."""
    return capi.host().moe_decode_diff(data, gate, indices_locations, int(top_k))
