"""Units of 8 query heads on the matrix split kernel, forced at small sizes, against a float64 decode of the same codes.

Tile and block edges, one and several splits, the current token and the fused append, score ranges that move the running
maximum.  Tolerance: that of the matrix kernel's other tests, 2e-6 of the output's scale at unit-scale inputs (see
test_gpu_mx.py), doubled for the wider scores here.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import torque_oracle as o

pytestmark = pytest.mark.gpu


def _decode64(cache, q, current=None):
    """Float64 attention of rotated queries [Hq, D] over the cache's dequantized rows, rotated back."""
    keys, values = (x[0].double() for x in cache._store.export_dequantized())
    if current is not None:
        keys, values = (torch.cat([x, c[0][:, None].double()], dim=1) for x, c in zip((keys, values), current))
    left, right = (s.double().cpu().numpy() for s in cache.rotation.device_signs())
    pi = torch.from_numpy(o.rotation_matrix(left, right)).to(q.device).double()
    qr = q.double() @ pi.t().contiguous()
    group = q.shape[0] // keys.shape[0]
    out = []
    for h in range(q.shape[0]):
        k, v = keys[h // group], values[h // group]
        out.append(torch.softmax((k @ qr[h]) / k.shape[1] ** 0.5, dim=0) @ v)
    return torch.stack(out) @ pi


@pytest.mark.parametrize("bits,dim", [(4, 64), (4, 128), (4, 256), (2, 128)])
@pytest.mark.parametrize("kv,group,seq,splits", [
    (1, 8, 1, 1), (2, 8, 15, 1), (1, 8, 16, 1), (1, 16, 17, 1), (2, 8, 129, 2), (1, 8, 1000, 3), (1, 24, 2500, 5), (2, 8, 3333, 0),
])
def test_units_of_8(hip_device, bits, dim, kv, group, seq, splits):
    import torque_hip as th
    from torque_hip import ops

    cache = th.TorqueKVCacheHIP(config=th.TorqueConfig(bit_width=bits, head_dim=dim, kv_heads=kv), initial_capacity=seq + 1)
    g = torch.Generator(device="cuda").manual_seed(seq + dim)
    k, v = (torch.randn(1, kv, seq, dim, generator=g, device="cuda") for _ in range(2))
    cache.append_many(key=k, value=v)
    nk, nv = (torch.randn(1, kv, 1, dim, generator=g, device="cuda") for _ in range(2))
    store = cache._store
    slab = dict(num_layers=1, query_heads=kv * group, kv_heads=kv, head_dim=dim, bit_width=bits, key_codes=store.key_codes,
                value_codes=store.value_codes, capacity=store.capacity, seq_len=seq, key_centroids=store.key_centroids,
                value_centroids=store.value_centroids, signs_left=store.signs_left, signs_right=store.signs_right,
                rotate_query=True, inverse_output=True, n_splits=splits, matrix_products=True)
    current = store.quantize_current(nk, nv, rotate_keys=True, rotate_values=True)
    for scale, dtype in ((1.0, torch.float32), (1.0, torch.float16), (6.0, torch.float32)):
        q = (scale * torch.randn(1, kv * group, dim, generator=g, device="cuda")).to(dtype)
        tol = 4e-6 * scale
        for cur in (None, current):
            got = ops.packed_decode(q, **slab, current_keys=None if cur is None else cur[0], current_values=None if cur is None else cur[1])[0]
            want = _decode64(cache, q[0], cur)
            assert (got - want).abs().max().item() <= tol * want.abs().max().item()
            again = ops.packed_decode(q, **slab, current_keys=None if cur is None else cur[0], current_values=None if cur is None else cur[1])[0]
            assert torch.equal(got, again)
        fused = ops.packed_decode_append(q, nk[:, :, 0].contiguous(), nv[:, :, 0].contiguous(), **slab, key_boundaries=store.key_boundaries,
                                         value_boundaries=store.value_boundaries)[0]
        assert (fused - want).abs().max().item() <= tol * want.abs().max().item()
