"""Decodes of many units on their default split plan against one split per unit.

Both sum the same float32 terms in another order: a sum of S terms in float32 is within S 2^-24 of the exact one
relative to the sum of magnitudes, and far inside it in practice (3e-7 at 32K tokens), so 1e-5 of the output's root
mean square leaves a wide margin at these lengths.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers,kv,group,dim,bits,seq,scale_mode", [
    (24, 8, 4, 128, 3, 1500, "none"),
    (24, 4, 3, 256, 2, 3001, "none"),
    (24, 4, 3, 64, 4, 9001, "rms"),
    (24, 8, 1, 128, 4, 4111, "none"),
])
def test_default_plan_matches_one_split(hip_device, layers, kv, group, dim, bits, seq, scale_mode):
    import torque_hip as th
    from torque_hip import ops

    flags = th._lib.TQ_F32_PRODUCTS if scale_mode == "rms" else 0
    assert ops.plan_splits(layers, kv, kv * group, dim, seq, hip_device, bit_width=bits, flags=flags) > 1
    config = th.TorqueConfig(bit_width=bits, head_dim=dim, num_layers=layers, kv_heads=kv, scale_mode=scale_mode)
    cache = th.TorqueKVCacheHIP(config=config, initial_capacity=seq)
    g = torch.Generator(device="cuda").manual_seed(seq)
    rows = lambda n: torch.randn((layers, n, dim), generator=g, device="cuda")
    for _ in range(2):  # two appends: the second half of the sequence has other norms
        k, v = (torch.randn((layers, kv, seq // 2, dim), generator=g, device="cuda") for _ in range(2))
        cache.append_many(key=k, value=2.0 * v)
    q = rows(kv * group)
    split = cache._store.decode(q, rotate_query=True, inverse_output=True)
    whole = cache._store.decode(q, rotate_query=True, inverse_output=True, n_splits=1)
    error = (split - whole).abs().max().item()
    assert error <= 1e-5 * whole.square().mean().sqrt().item()
    assert np.array_equal(split.cpu().numpy(), cache._store.decode(q, rotate_query=True, inverse_output=True).cpu().numpy())
