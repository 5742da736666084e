"""The append kernel at its edges: packed words bit for bit against the oracle.

Row counts around the line between the two kernels (4096 rows of both streams), around a workgroup's rows (64, 32, 16
at head_dim 64, 128, 256) and groups that end inside a wavefront,
sources that are not 16-byte aligned, quotients that tie with a boundary, values without an ordinary quotient (zeros,
subnormals, infinities, NaN), and codebooks that the bucket lookup cannot take (equal, unordered, infinite boundaries).
Whole-number outputs: no tolerance.
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
    (1, 4111, np.float32, 1), (300, 7, np.float16, 0),
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
        for rows in (x, np.resize(x, (2100, head_dim))):  # a wavefront per row, then 16 elements to a lane
            _check(rows, signs, bnd, bits, seq_new=rows.shape[0], rotate=rotate)


@pytest.mark.parametrize("bits", [2, 3, 4])
def test_codebooks_without_buckets(hip_device, bits):
    head_dim, n = 128, (1 << bits) - 1
    rng = np.random.default_rng(bits)
    x = rng.normal(size=(2100, head_dim)).astype(np.float32)
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
    x = rng.normal(size=(2100, head_dim)).astype(np.float32)
    signs = [(s * rng.uniform(0.5, 2.0, size=head_dim)).astype(np.float32) for s in o.rotation_signs_from_seed(head_dim, 4)]
    bnd = o.codebook_boundaries(o.build_gaussian_codebook(4, sample_size=5000, seed=1))
    _check(x, signs, bnd, 4, seq_new=2100)
