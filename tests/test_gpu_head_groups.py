"""Groups of query heads that are no multiple of 4: units of 4 heads with slots to spare, against the oracle.

Lengths on both sides of the line where they take over, decodes of one and several splits, the current token and the
fused append.  Tolerances are the float32 ones of the cache tests.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import torque_oracle as o

pytestmark = pytest.mark.gpu


def _caches(bits, dim, kv, seq, seed, scale_mode="none"):
    import torque_hip as th

    cache = th.TorqueKVCacheHIP(config=th.TorqueConfig(bit_width=bits, head_dim=dim, kv_heads=kv, scale_mode=scale_mode), initial_capacity=seq)
    rng = np.random.default_rng(seed)
    k, v = (rng.normal(size=(1, kv, seq, dim)).astype(np.float32) for _ in range(2))
    cache.append_many(key=k, value=v)
    return cache, k, v, rng


@pytest.mark.parametrize("bits,dim,kv,group,seq", [
    (3, 128, 2, 3, 33000), (3, 128, 2, 3, 500), (4, 128, 2, 7, 7001), (4, 64, 1, 5, 44000), (2, 256, 2, 6, 17000), (4, 256, 1, 7, 6600),
])
def test_odd_groups_match_oracle(hip_device, bits, dim, kv, group, seq):
    cache, k, v, rng = _caches(bits, dim, kv, seq, seq)
    model = o.OracleCache(bit_width=bits, head_dim=dim, num_layers=1, kv_heads=kv, key_centroids=cache.key_codebook.centroids,
                          value_centroids=cache.value_codebook.centroids, signs_left=cache.rotation.signs_left,
                          signs_right=cache.rotation.signs_right)
    model.append(k, v)
    q = rng.normal(size=(1, kv * group, dim)).astype(np.float32)
    expected = model.decode(q)[0]
    for n in (None, 1, 7):
        got = cache._store.decode(torch.from_numpy(q).to(hip_device), rotate_query=True, inverse_output=True, n_splits=n)
        np.testing.assert_allclose(got[0].cpu().numpy(), expected, atol=1e-5)
    nk, nv = (rng.normal(size=(1, kv, dim)).astype(np.float32) for _ in range(2))
    current = cache.decode_with_current(query=q, key=nk, value=nv)
    fused = cache.decode_append(query=q, key=nk, value=nv)
    model.append(nk[:, :, None], nv[:, :, None])
    expected = model.decode(q)[0]
    np.testing.assert_allclose(current, expected, atol=1e-5)
    np.testing.assert_allclose(fused, expected, atol=1e-5)
    np.testing.assert_array_equal(cache._key_codes[:, :, : seq + 1].cpu().numpy().view(np.uint32), model.k_codes)


@pytest.mark.parametrize("group,seq", [(3, 9000), (5, 30000), (6, 40000), (7, 30000)])
def test_odd_groups_of_dense_and_scaled_rows(hip_device, group, seq):
    """The same head decoded alone (groups of 1) sums the same float32 terms in another order."""
    from torque_hip import ops

    g = torch.Generator(device="cuda").manual_seed(group)
    q = torch.randn(1, 2 * group, 128, generator=g, device="cuda")
    k, v = (torch.randn(1, 2, seq, 128, generator=g, device="cuda").half() for _ in range(2))
    shape = dict(num_layers=1, head_dim=128, capacity=seq, seq_len=seq)
    got = ops.dense_decode(q, k, v, query_heads=2 * group, kv_heads=2, **shape)
    cache, _, _, _ = _caches(4, 128, 2, seq, 5, "rms")
    scaled = cache._store.decode(q, rotate_query=True, inverse_output=True)
    for h in range(group):
        mine = q[:, h::group].contiguous()
        alone = ops.dense_decode(mine, k, v, query_heads=2, kv_heads=2, **shape)
        assert torch.allclose(got[:, h::group], alone, atol=2e-6, rtol=1e-5)
        alone = cache._store.decode(mine, rotate_query=True, inverse_output=True)
        assert torch.allclose(scaled[:, h::group], alone, atol=2e-6, rtol=1e-5)
