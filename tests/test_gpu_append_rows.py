"""The append kernel at its edges: packed words bit for bit against the oracle.

Row counts around the line between the two kernels (4096 to 8192 rows of both streams when packing), around a workgroup's rows (64, 32, 16
at head_dim 64, 128, 256) and groups that end inside a wavefront,
sources that are not 16-byte aligned, quotients that tie with a boundary, values without an ordinary quotient (zeros,
subnormals, infinities, NaN), and codebooks that the bucket lookup cannot take (equal, unordered, infinite boundaries).
Whole-number outputs: no tolerance.

The forms with per-vector scales and those that write centroid values run here on both sides of their lines, where the
other tests of those entry points stay below them: bit for bit the same as calls of few rows, codes and centroids against the oracle on
the kernel's own scales.
"""

from __future__ import annotations

from math import sqrt

import numpy as np
import pytest
import torch

from oracle import torque_oracle as o

pytestmark = pytest.mark.gpu

DIMS = [64, 128, 256]


def _append(x, signs, boundaries, bits, *, seq_new, rotate=True, shift=0):
    """tq_append of rows x [groups * seq_new, D] (keys, and negated as values) into slabs with two spare tokens."""
    import torque_hip as th

    head_dim = x.shape[1]
    groups = x.shape[0] // seq_new
    words = head_dim * bits // 32

    def source(a):
        buf = torch.zeros(a.size + shift, dtype=torch.float16 if a.dtype == np.float16 else torch.float32, device="cuda")
        buf[shift:] = torch.from_numpy(a.reshape(-1)).cuda()
        return buf[shift:]

    k, v = source(x), source(-x)
    left, right = (torch.from_numpy(s.astype(np.float32)).cuda() for s in signs)
    bnd = torch.from_numpy(np.asarray(boundaries, dtype=np.float32)).cuda()
    codes = [torch.full((groups, seq_new + 2, words), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
    th._lib.call("tq_append", k.data_ptr(), v.data_ptr(), th._lib.TQ_F16 if x.dtype == np.float16 else th._lib.TQ_F32, 1, groups,
                 seq_new, head_dim, bits, left.data_ptr(), right.data_ptr(), 3 if rotate else 0, bnd.data_ptr(), bnd.data_ptr(),
                 codes[0].data_ptr(), codes[1].data_ptr(), seq_new + 2, 1, torch.cuda.current_stream().cuda_stream)
    got = [c.cpu().numpy().view(np.uint32) for c in codes]
    for g in got:  # the slots around the appended tokens are left alone
        assert (g[:, 0] == 0xFFFFFFFF).all() and (g[:, -1] == 0xFFFFFFFF).all()
    return [g[:, 1:-1].reshape(-1, words) for g in got]


def _expect(x, signs, boundaries, bits, rotate=True):
    with np.errstate(all="ignore"):
        y = x.astype(np.float32)
        y = o.rotation_apply(y, *signs) if rotate else y
        return o.pack_indices_batched(o.quantize_boundary_count(y, np.asarray(boundaries, dtype=np.float32)), bits)


def _check(x, signs, boundaries, bits, **kwargs):
    got = _append(x, signs, boundaries, bits, **kwargs)
    rotate = kwargs.get("rotate", True)
    np.testing.assert_array_equal(got[0], _expect(x, signs, boundaries, bits, rotate))
    np.testing.assert_array_equal(got[1], _expect(-x, signs, boundaries, bits, rotate))


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("head_dim", DIMS)
@pytest.mark.parametrize("groups,seq_new,dtype,shift", [
    (1, 1, np.float16, 0), (3, 1, np.float32, 0), (1, 15, np.float16, 0), (5, 7, np.float32, 1), (1, 65, np.float16, 3),
    (2, 64, np.float32, 0), (7, 33, np.float16, 0), (3, 1367, np.float32, 0), (2048, 1, np.float16, 0), (5, 411, np.float16, 1),
    (1, 4111, np.float32, 1), (300, 7, np.float16, 0), (5, 823, np.float16, 1), (600, 7, np.float32, 0),
])
def test_row_counts_and_alignment(hip_device, bits, head_dim, groups, seq_new, dtype, shift):
    rng = np.random.default_rng(bits * 1000 + head_dim + seq_new)
    x = rng.normal(0.0, 1.3, size=(groups * seq_new, head_dim)).astype(dtype)
    signs = o.rotation_signs_from_seed(head_dim, 3)
    bnd = o.codebook_boundaries(o.build_gaussian_codebook(bits, sample_size=5000, seed=1))
    _check(x, signs, bnd, bits, seq_new=seq_new, shift=shift)


@pytest.mark.parametrize("head_dim", DIMS)
@pytest.mark.parametrize("rotate", [True, False])
def test_ties_and_special_values(hip_device, head_dim, rotate):
    """One element of a row sets every element of its transform to +-x, so quotients sit on and beside the boundaries."""
    bits = 4
    signs = o.rotation_signs_from_seed(head_dim, 5)
    for bnd in (o.codebook_boundaries(o.uniform_codebook(bits)),  # has a boundary at 0 (or next to it)
                np.array([0.0] + [k * 0.37 for k in range(1, 15)], dtype=np.float32),
                np.linspace(-3e38, 3e38, 15).astype(np.float32)):
        points = []
        for b in bnd:
            with np.errstate(all="ignore"):
                y = np.float32(b * np.float32(sqrt(head_dim))) if rotate else np.float32(b)
            for _ in range(6):
                y = np.nextafter(y, np.float32(-np.inf), dtype=np.float32)
            for _ in range(13):
                points.append(y)
                y = np.nextafter(y, np.float32(np.inf), dtype=np.float32)
        points += [0.0, -0.0, 1e-45, -1e-45, 6e-45, 1e-42, 1e-38, 3.4e38, -3.4e38, np.inf, -np.inf, np.nan]
        x = np.zeros((len(points), head_dim), dtype=np.float32)
        x[np.arange(len(points)), np.arange(len(points)) % head_dim] = points
        mixed = np.random.default_rng(1).normal(size=(9, head_dim)).astype(np.float32)
        mixed[0, :], mixed[1, 3], mixed[2, 5], mixed[3, :] = 0.0, np.inf, np.nan, 2e38
        mixed[4] *= 1e-40
        x = np.concatenate([x, mixed])
        for rows in (x, np.resize(x, (2100, head_dim)), np.resize(x, (4200, head_dim))):  # a wavefront per row, then 16 elements to a lane
            _check(rows, signs, bnd, bits, seq_new=rows.shape[0], rotate=rotate)


@pytest.mark.parametrize("bits", [2, 3, 4])
def test_codebooks_without_buckets(hip_device, bits):
    head_dim, n = 128, (1 << bits) - 1
    rng = np.random.default_rng(bits)
    x = rng.normal(size=(4200, head_dim)).astype(np.float32)
    signs = o.rotation_signs_from_seed(head_dim, 2)
    close = np.linspace(-1e-3, 1e-3, n)
    close[-1] = 4.0  # all but one share a bucket
    boundaries = [np.zeros(n), rng.permutation(np.linspace(-2, 2, n)), close, np.where(np.arange(n) == 1, np.inf, np.linspace(-1, 1, n)),
                  np.where(np.arange(n) == 0, -np.inf, np.linspace(-1, 1, n)), np.where(np.arange(n) == n - 1, np.nan, np.linspace(-1, 1, n))]
    for bnd in boundaries:
        for rotate in (True, False):
            _check(x, signs, bnd, bits, seq_new=35, rotate=rotate)


@pytest.mark.parametrize("head_dim", DIMS)
def test_signs_of_any_size(hip_device, head_dim):
    """Sign vectors that are not +-1 take the division per element."""
    rng = np.random.default_rng(head_dim)
    x = rng.normal(size=(4200, head_dim)).astype(np.float32)
    signs = [(s * rng.uniform(0.5, 2.0, size=head_dim)).astype(np.float32) for s in o.rotation_signs_from_seed(head_dim, 4)]
    bnd = o.codebook_boundaries(o.build_gaussian_codebook(4, sample_size=5000, seed=1))
    _check(x, signs, bnd, 4, seq_new=4200)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _codebooks(bits):
    books = [o.build_gaussian_codebook(bits, sample_size=5000, seed=s) for s in (1, 2)]
    return [torch.from_numpy(np.asarray(a, dtype=np.float32)).cuda() for b in books for a in (o.codebook_boundaries(b), b)]


def _sources(rows, head_dim, dtype, shift, seed):
    """Two streams of rows over a few decades of norms, `shift` elements off a 16-byte boundary, with rows whose mean
    square is zero, infinite, subnormal or no number."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for _ in range(2):
        x = torch.randn(rows, head_dim, generator=g, device="cuda") * torch.randn(rows, 1, generator=g, device="cuda").exp()
        x[7], x[rows - 2], x[100, 3], x[4096 % rows, 5], x[9] = 0.0, 0.0, float("inf"), float("nan"), x[9] * 1e-23
        buf = torch.zeros(rows * head_dim + shift, dtype=dtype, device="cuda")
        buf[shift:] = x.reshape(-1).to(dtype)
        out.append(buf[shift:].view(rows, head_dim))
    return out


def _unpack(words, bits, head_dim):
    """Codes of packed rows: element e at bit e * bits of the row."""
    at = torch.arange(head_dim, device=words.device) * bits
    wide = words.to(torch.int64) & 0xFFFFFFFF
    pair = wide | torch.nn.functional.pad(wide, (0, 1))[:, 1:] << 32  # bits up to 31 of the next word: the last row word has none
    return (pair[:, at // 32] >> (at % 32)) & ((1 << bits) - 1)


def _type(x):
    import torque_hip as th

    return th._lib.TQ_F16 if x.dtype == torch.float16 else th._lib.TQ_F32


FORMS = [(2053, torch.float16, 0, 3), (2053, torch.float32, 1, 3), (4500, torch.float32, 0, 3), (4500, torch.float16, 3, 0), (9001, torch.float16, 0, 1)]
LINES = {4: 16000, 3: 60000, 2: 165000}  # rows of two streams past the largest line of the bit width, when writing values


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("head_dim", DIMS)
@pytest.mark.parametrize("rows,dtype,shift,flags", FORMS)
def test_scaled_rows(hip_device, bits, head_dim, rows, dtype, shift, flags):
    import torque_hip as th

    keys, values = _sources(rows, head_dim, dtype, shift, bits + head_dim)
    signs = o.rotation_signs_from_seed(head_dim, 6)
    left, right = (torch.from_numpy(s).cuda() for s in signs)
    kb, _, vb, _ = _codebooks(bits)
    words = head_dim * bits // 32

    def append(cuts):
        codes = [torch.full((rows + 2, words), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
        scales = [torch.full((rows + 2,), -1.0, device="cuda") for _ in range(2)]
        for t0, t1 in cuts:
            th._lib.call("tq_append_scaled", keys[t0:t1].data_ptr(), values[t0:t1].data_ptr(), _type(keys), 1, 1, t1 - t0, head_dim, bits,
                         left.data_ptr(), right.data_ptr(), flags, kb.data_ptr(), vb.data_ptr(), codes[0].data_ptr(), codes[1].data_ptr(),
                         scales[0].data_ptr(), scales[1].data_ptr(), rows + 2, 1 + t0, _stream())
        return codes, scales

    codes, scales = append([(0, rows)])
    few_codes, few_scales = append([(t, min(t + 1000, rows)) for t in range(0, rows, 1000)])
    for i, (x, rotate, bnd) in enumerate(((keys, flags & 1, kb), (values, flags & 2, vb))):
        assert torch.equal(codes[i], few_codes[i]) and torch.equal(scales[i].view(torch.int32), few_scales[i].view(torch.int32))
        assert codes[i][0].eq(-1).all() and codes[i][-1].eq(-1).all() and scales[i][0] == scales[i][-1] == -1.0
        with np.errstate(all="ignore"):
            y = x.float().cpu().numpy()
            y = o.rotation_apply(y, *signs) if rotate else y
            s = scales[i][1:-1].cpu().numpy()
            exp, _ = o.quantize_scaled(y, bnd.cpu().numpy(), s)
        np.testing.assert_array_equal(codes[i][1:-1].cpu().numpy().view(np.uint32), o.pack_indices_batched(exp, bits))
        ordinary = np.isfinite(y).all(axis=1) & (np.abs(y).max(axis=1) > 1e-15)  # whose squares float32 holds
        np.testing.assert_allclose(s[ordinary], o.rms_scales(y[ordinary]), rtol=3e-6)  # as test_gpu_scaled.py
        assert s[7] == s[rows - 2] == 1.0 and ordinary.sum() >= rows - 6


@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("head_dim", DIMS)
@pytest.mark.parametrize("rows,dtype,shift,flags", [(2053, torch.float16, 1, 3), (None, torch.float32, 0, 3), (None, torch.float16, 1, 1)])
def test_dequantized_rows(hip_device, bits, head_dim, rows, dtype, shift, flags, scaled):
    import torque_hip as th

    rows = rows or LINES[bits] // 2 + 37
    keys, values = _sources(rows, head_dim, dtype, shift, bits + head_dim)
    left, right = (torch.from_numpy(s).cuda() for s in o.rotation_signs_from_seed(head_dim, 6))
    kb, kc, vb, vc = _codebooks(bits)
    words = head_dim * bits // 32
    name = "_scaled" if scaled else ""

    def dequantize(cuts, off=0):
        out = [torch.full((rows * head_dim + 8,), 99.0, device="cuda") for _ in range(2)]
        for t0, t1 in cuts:
            ptrs = [x[off + t0 * head_dim :].data_ptr() for x in out]
            th._lib.call("tq_quantize_dequantize" + name, keys[t0:t1].data_ptr(), values[t0:t1].data_ptr(), _type(keys), t1 - t0, head_dim,
                         bits, left.data_ptr(), right.data_ptr(), flags, kb.data_ptr(), vb.data_ptr(), kc.data_ptr(), vc.data_ptr(), *ptrs,
                         _stream())
        for x in out:
            assert x[:off].eq(99.0).all() and x[off + rows * head_dim :].eq(99.0).all()
        return [x[off : off + rows * head_dim].view(rows, head_dim) for x in out]

    got = dequantize([(0, rows)])
    few = dequantize([(t, min(t + 1000, rows)) for t in range(0, rows, 1000)])
    moved = dequantize([(0, rows)], off=1)  # outputs off a 16-byte boundary
    # the packing form's codes (and scales), which the tests above compare with the oracle
    codes = [torch.zeros(rows, words, dtype=torch.int32, device="cuda") for _ in range(2)]
    scales = [torch.zeros(rows, device="cuda") for _ in range(2)]
    extra = [s.data_ptr() for s in scales] if scaled else []
    th._lib.call("tq_append" + name, keys.data_ptr(), values.data_ptr(), _type(keys), 1, 1, rows, head_dim, bits, left.data_ptr(),
                 right.data_ptr(), flags, kb.data_ptr(), vb.data_ptr(), codes[0].data_ptr(), codes[1].data_ptr(), *extra, rows, 0, _stream())
    for i, cent in enumerate((kc, vc)):
        index = _unpack(codes[i], bits, head_dim)
        want = cent[index] * scales[i][:, None] if scaled else cent[index]
        for y in (got[i], few[i], moved[i]):
            assert torch.equal(y.view(torch.int32), want.view(torch.int32))
