"""The adapter's rotary and gate kernels against the torch operations they stand for."""

from __future__ import annotations

import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu

TYPES = [torch.float32, torch.float16, torch.bfloat16]


def _rotary_reference(x, cos, sin):
    r = cos.shape[-1]
    a, rest = x[..., :r], x[..., r:]
    half = torch.cat((-a[..., r // 2:], a[..., : r // 2]), dim=-1)
    return torch.cat([a * cos[:, None] + half * sin[:, None], rest], dim=-1)


@pytest.mark.parametrize("head_dim,rotary_dim", [(64, 64), (64, 2), (128, 32), (256, 64), (256, 130)])
@pytest.mark.parametrize("tokens,q_heads,k_heads", [(1, 4, 1), (37, 5, 2)])
def test_rotary_bit_exact(hip_device, head_dim, rotary_dim, tokens, q_heads, k_heads):
    from torque_hip import qwen_torch as qt

    g = torch.Generator(device=hip_device).manual_seed(head_dim + rotary_dim + tokens)
    for x_type, table_type in itertools.product(TYPES, TYPES):
        q, k = (torch.randn(1, tokens, h, head_dim + 3, generator=g, device=hip_device).to(x_type)[..., 1 : 1 + head_dim].transpose(1, 2)
                for h in (q_heads, k_heads))
        cos, sin = (torch.randn(1, tokens, rotary_dim, generator=g, device=hip_device).to(table_type) for _ in range(2))
        got = qt._rotary_fused(q, k, cos, sin)
        assert got is not None
        for y, x in zip(got, (q, k)):
            expected = _rotary_reference(x, cos, sin)
            assert y.dtype == expected.dtype and y.is_contiguous()
            assert torch.equal(y, expected), (x_type, table_type)


@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("tokens,heads", [(1, 4), (37, 5)])
def test_unrotate_gate(hip_device, head_dim, tokens, heads):
    """Two float32 operations after the bit-identical rotation, and a sigmoid of two more: the result is within 4 ulp
    (4 x 2^-23) of the torch composition in float32, one unit of the output type more where that rounds."""
    from torque_hip import RotationSpec
    from torque_hip import qwen_torch as qt

    rotation = RotationSpec.from_seed(head_dim, 3)
    g = torch.Generator(device=hip_device).manual_seed(head_dim + tokens)
    for gate_type, out_type in itertools.product(TYPES, TYPES):
        attn = torch.randn(1, tokens, heads, head_dim, generator=g, device=hip_device).transpose(1, 2)
        both = 4.0 * torch.randn(1, tokens, heads, 2 * head_dim, generator=g, device=hip_device)
        gate = both.to(gate_type)[..., head_dim:]
        got = qt._unrotate_gate(attn, gate, rotation=rotation, dtype=out_type)
        rotated = qt.runtime_unrotate_attention_output(attn, rotation=rotation)
        expected = rotated.transpose(1, 2).reshape(1, tokens, -1) * torch.sigmoid(gate.reshape(1, tokens, -1).float())
        assert got.dtype == out_type and got.shape == expected.shape
        unit = {torch.float32: 0.0, torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7}[out_type]
        torch.testing.assert_close(got.float(), expected, rtol=4 * 2.0**-23 + unit, atol=1e-7 if unit else 1e-30)


def test_gradients_and_transforms_keep_the_torch_operations(hip_device):
    from torque_hip import RotationSpec
    from torque_hip import qwen_torch as qt

    q, k = torch.randn(1, 2, 3, 64, device=hip_device), torch.randn(1, 1, 3, 64, device=hip_device)
    cos, sin = torch.randn(1, 3, 16, device=hip_device), torch.randn(1, 3, 16, device=hip_device)
    want = _rotary_reference(q, cos, sin)
    leaf = q.clone().requires_grad_()
    out = qt.apply_rotary(leaf, k, cos, sin)[0]
    assert out.requires_grad and torch.equal(out, want)
    with torch.no_grad():
        assert qt._rotary_fused(leaf, k, cos, sin) is not None
    stacked = torch.func.vmap(lambda x: qt.apply_rotary(x, k, cos, sin)[0])(torch.stack([q, q]))
    assert torch.equal(stacked[1], want)
    tangent = torch.func.jvp(lambda x: qt.apply_rotary(x, k, cos, sin)[0], (q,), (torch.ones_like(q),))[1]
    assert torch.allclose(tangent, _rotary_reference(torch.ones_like(q), cos, sin))
    assert qt._rotary_fused(q.cpu(), k.cpu(), cos.cpu(), sin.cpu()) is None
    assert qt._rotary_fused(q.double(), k.double(), cos, sin) is None
    assert all(torch.equal(a, b) for a, b in zip(qt.apply_rotary(q, k, cos[..., :0], sin[..., :0]), (q, k)))
    gate = torch.randn(1, 3, 2, 64, device=hip_device, requires_grad=True)
    rotation = RotationSpec.from_seed(64, 1)
    qt._unrotate_gate(q, gate, rotation=rotation, dtype=torch.float32).sum().backward()
    assert gate.grad is not None and gate.grad.abs().sum() > 0


def test_rows_past_one_launch(hip_device):
    """More rows than the 2^32 - 1 work-items of one launch hold at a wavefront each (2^26): a call is cut into several."""
    from torque_hip import RotationSpec
    from torque_hip import qwen_torch as qt

    g = torch.Generator(device=hip_device).manual_seed(1)
    tokens = 2**25 + 3
    q, k = (torch.randn(1, 1, tokens, 2, generator=g, device=hip_device, dtype=torch.float16) for _ in range(2))
    cos, sin = (torch.randn(1, tokens, 2, generator=g, device=hip_device, dtype=torch.float16) for _ in range(2))
    for y, x in zip(qt.apply_rotary(q, k, cos, sin), (q, k)):
        assert torch.equal(y, _rotary_reference(x, cos, sin))
    del q, k, cos, sin, x, y
    heads, tokens = 64, 2**20 + 1
    attn = torch.randn(1, 1, tokens, 64, generator=g, device=hip_device).expand(1, heads, tokens, 64)
    gate = torch.randn(1, tokens, 1, 64, generator=g, device=hip_device).expand(1, tokens, heads, 64)
    rotation = RotationSpec.from_seed(64, 3)
    one = qt._unrotate_gate(attn[:, :1], gate[:, :, :1], rotation=rotation, dtype=torch.bfloat16)
    got = qt._unrotate_gate(attn, gate, rotation=rotation, dtype=torch.bfloat16).view(tokens, heads, 64)
    for h in range(heads):
        assert torch.equal(got[:, h], one[0])


def test_operands_of_another_device_keep_the_torch_operations(hip_device, monkeypatch):
    """The library launches on the current device: tensors of another one go through torch, which guards its calls."""
    from torque_hip import _lib
    from torque_hip import qwen_torch as qt

    q, k = torch.randn(1, 2, 3, 64, device=hip_device), torch.randn(1, 1, 3, 64, device=hip_device)
    cos, sin = torch.randn(1, 3, 16, device=hip_device), torch.randn(1, 3, 16, device=hip_device)
    assert qt._plain(q, k, cos, sin)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: hip_device.index + 1)
    monkeypatch.setattr(_lib, "call", lambda *args: pytest.fail("launched on the current device"))
    assert not qt._plain(q, k, cos, sin)
    for y, x in zip(qt.apply_rotary(q, k, cos, sin), (q, k)):
        assert torch.equal(y, _rotary_reference(x, cos, sin))


def _check_attention(q, k, v, scale, offset, rows=slice(None)):
    """Against float64, as float32 attention.  A float32 score is a sum of D products, off by at most (D + 1) 2^-24 of
    its sum of magnitudes A however the products are grouped, and in fact by a few 2^-24; with 2 A 2^-22 allowed to a
    score every weight is off by that, relatively, in the numerator and the sum, and the sums of weights and values add
    a few 2^-22.  An output is then within (4 A + 16) 2^-22 of the same weighted sum of the values' magnitudes: its own
    keys' values, whatever keys it does not attend, or barely attends, hold."""
    from torque_hip import qwen_torch as qt

    got = qt._dense_attention(q, k, v, scale=scale, offset=offset)
    assert got.dtype == torch.float32 and got.shape == q.shape
    q, k, v = q[0].double(), k[0].double(), v[0].double()
    group = q.shape[0] // k.shape[0]
    allowed = torch.arange(k.shape[1], device=q.device)[None] <= torch.arange(offset, offset + q.shape[1], device=q.device)[:, None]
    for h in range(q.shape[0]):
        kt, vh = k[h // group].t().contiguous(), v[h // group].contiguous()
        weights = torch.softmax((torch.matmul(q[h], kt) * scale).masked_fill(~allowed, float("-inf")), dim=-1)
        most = torch.matmul(q[h].abs(), kt.abs()).masked_fill(~allowed, 0.0).amax(dim=-1, keepdim=True) * scale
        error = (got[0, h] - torch.matmul(weights, vh)).abs()
        bound = (4 * most + 16) * 2.0**-22 * torch.matmul(weights, vh.abs()) + 1e-38
        assert torch.all((error <= bound)[rows])


@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("tokens,offset,heads,kv_heads", [
    (1, 0, 1, 1), (2, 0, 4, 4), (16, 0, 5, 1), (17, 15, 6, 2), (31, 1, 8, 2), (33, 64, 7, 7), (130, 3, 16, 4), (257, 0, 3, 1),
])
def test_prompt_attention(hip_device, head_dim, tokens, offset, heads, kv_heads):
    """Short and ragged chunks, operands of every type, strided rows."""
    g = torch.Generator(device=hip_device).manual_seed(head_dim + tokens)
    keys = tokens + offset
    for types in ((torch.float32,) * 3, (torch.float32, torch.float32, torch.bfloat16), (torch.float16,) * 3):
        rows = lambda n, h: torch.randn(1, n, h, head_dim + 8, generator=g, device=hip_device)[..., 3 : 3 + head_dim].transpose(1, 2)
        q, k, v = (x.to(t) for x, t in zip((rows(tokens, heads), rows(keys, kv_heads), rows(keys, kv_heads)), types))
        # keys and values whose scale changes along the sequence
        k = k * torch.linspace(0.2, 2.0, keys, device=hip_device)[:, None].to(k.dtype)
        v = v * torch.exp2(torch.arange(keys, device=hip_device) % 97 / 12.0 - 4.0)[:, None].to(v.dtype)
        _check_attention(q, k, v, head_dim**-0.5, offset)


def test_prompt_attention_zero_and_extreme_rows(hip_device):
    """Zero values, one-key rows and magnitudes far from 1 keep the accuracy."""
    g = torch.Generator(device=hip_device).manual_seed(3)
    q, k, v = (torch.randn(1, h, 100, 64, generator=g, device=hip_device) for h in (2, 1, 1))
    v[:, :, 32:64] = 0.0
    for a, b in ((1.0, 1.0), (1e-20, 1e12), (1e15, 1e-18)):
        _check_attention(q / a, k * a, v * b, 0.125, 0)


@pytest.mark.parametrize("spread", [12, 20, 24, 28])
@pytest.mark.parametrize("where", ["masked value", "masked key", "barely attended value", "channel"])
def test_prompt_attention_keeps_every_value_s_own_precision(hip_device, where, spread):
    """A row's result has float32's precision of what the row attends, next to values 2^spread larger that it does not
    attend (a later key's value or key), that it gives no weight to (an early key far off the query) or that sit in
    other channels."""
    g = torch.Generator(device=hip_device).manual_seed(spread)
    q, k, v = (torch.randn(1, h, 96, 64, generator=g, device=hip_device) for h in (2, 1, 1))
    if where == "masked value":
        v[:, :, 29] *= 2.0**spread
    elif where == "masked key":
        k[:, :, 29] *= 2.0**spread
    elif where == "barely attended value":
        q[..., 0], k[..., 0] = 8.0, 20.0
        k[:, :, 3, 0] = -20.0  # a score 40 below the others'
        v[:, :, 3] *= 2.0**spread
    else:
        v[..., 1::2] *= 2.0**-spread
    # the rows that come before the key that is out of scale, computed beside the ones after it
    _check_attention(q, k, v, 0.125, 0, rows=slice(0, 29) if where.startswith("masked") else slice(None))
