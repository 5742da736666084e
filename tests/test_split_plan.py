"""The default split plan of calls with many units, on the host: sizes that callers rely on."""

from __future__ import annotations

import random

import pytest

from torque_hip import _lib

CUS = 256
SCRATCH = 8 << 20  # tq_decode_noalloc's


def _splits(layers, kv, group, dim, bits, flags, seq):
    return _lib.call("tq_decode_default_splits", layers, kv, kv * group, dim, bits, flags, seq, CUS)


def _bytes(layers, kv, group, dim, n):
    return _lib.call("tq_decode_workspace_bytes", layers, kv, kv * group, dim, n, CUS)


def test_default_workspace_covers_every_plan():
    rng = random.Random(0)
    for _ in range(5000):
        shape = (rng.choice([1, 2, 3, 6, 12, 16, 24, 32, 64]), rng.choice([1, 2, 4, 8]), rng.randint(1, 8), rng.choice([64, 128, 256]))
        n = _splits(*shape, rng.choice([0, 2, 3, 4]), rng.choice([0, _lib.TQ_F32_PRODUCTS]), int(10 ** rng.uniform(0, 5.3)))
        need = _bytes(*shape, n)
        assert need <= _bytes(*shape, 0)
        if n > 1:  # more than the scratch holds only where one split does not fit either
            assert need <= SCRATCH or _bytes(*shape, 1) > SCRATCH, (shape, n)


@pytest.mark.parametrize("layers,kv,group,dim,bits,seq,most", [
    (24, 8, 4, 128, 3, 8192, 4),  # 192 units: 3 workgroups to a CU
    (24, 8, 1, 128, 4, 8192, 4),
    (24, 4, 4, 256, 3, 8192, 5),  # one round, 480 workgroups: more splits would save less than 1/16
    (1, 8, 4, 128, 3, 32768, 64),  # one round fills the CUs evenly: unchanged
    (24, 8, 1, 128, 4, 200, 1),  # short: one launch
    (1, 8, 1, 128, 4, 384, 1),  # one split as far as it is the faster one on the GPU: 6 iterations
    (1, 8, 1, 128, 4, 385, 4),
    (1, 8, 4, 128, 3, 320, 1),  # 5 for units of several heads
    (1, 8, 4, 128, 3, 321, 3),
    (1, 8, 1, 128, 4, 513, 5),
    (1, 8, 1, 256, 4, 256, 1),  # 8 shorter ones
    (1, 4, 4, 256, 4, 224, 1),
    (1, 4, 4, 256, 4, 225, 2),
    (24, 8, 4, 128, 3, 512, 1),  # more units than half of the CUs
    (24, 8, 4, 128, 3, 513, 2),
    (1, 4, 4, 256, 4, 257, 3),
    (1, 4, 4, 64, 3, 512, 1),
    (1, 4, 4, 64, 3, 513, 5),
    (1, 8, 1, 128, 0, 512, 4),  # dense rows: as long as any
])
def test_workgroups_spread_over_the_cus(layers, kv, group, dim, bits, seq, most):
    assert _splits(layers, kv, group, dim, bits, 0, seq) == most


@pytest.mark.parametrize("dim,bits,most", [(64, 4, 512), (128, 2, 512), (128, 3, 512), (256, 4, 256)])
@pytest.mark.parametrize("kv,group", [(8, 1), (4, 4), (4, 6)])
def test_one_launch_on_request(dim, bits, most, kv, group):
    """TQ_ONE_LAUNCH: one split up to 512 tokens and 8 iterations, on the kernel the call runs on without it."""
    one = _lib.TQ_ONE_LAUNCH
    assert _splits(1, kv, group, dim, bits, one, most) == 1 < _splits(1, kv, group, dim, bits, one, most + 1)
    for seq in (100, most, most + 1, 20000):
        name = lambda flags: _lib.split_kernel(kv, kv * group, dim, bits, flags, _lib.TQ_F16, seq, num_cus=CUS).split("<")[0]
        assert name(one) == name(0)
        assert _splits(1, kv, group, dim, bits, one, seq) == 1 or _splits(1, kv, group, dim, bits, 0, seq) == _splits(1, kv, group, dim, bits, one, seq)


@pytest.mark.parametrize("layers,kv,group,dim,bits,seq,default", [
    (1, 4, 8, 128, 4, 30001, 64),  # units of 8 heads: 4 x 64 workgroups
    (1, 8, 16, 128, 4, 32768, 16),
    (24, 2, 8, 256, 4, 8192, 5),
    (1, 4, 8, 128, 4, 8192, 64),  # too few blocks for the matrix kernel: units of 4 heads on the float32 kernel
])
def test_default_count_names_its_own_kernel(layers, kv, group, dim, bits, seq, default):
    """The default count passed explicitly runs the kernel that the default runs."""
    assert _splits(layers, kv, group, dim, bits, 0, seq) == default
    name = lambda n: _lib.split_kernel(kv, kv * group, dim, bits, 0, _lib.TQ_F16, seq, num_layers=layers, n_splits=n, num_cus=CUS)
    assert name(0) == name(default)
    assert ("mx" in name(0)) == (seq != 8192 or layers > 1)


@pytest.mark.parametrize("layers,kv,group,dim,bits", [
    (24, 8, 4, 64, 4), (24, 8, 4, 128, 4), (24, 8, 4, 128, 2), (48, 4, 4, 128, 4), (12, 8, 8, 128, 4), (24, 8, 8, 64, 4), (24, 4, 16, 128, 2),
])
def test_one_split_of_many_units_keeps_the_matrix_kernel(layers, kv, group, dim, bits):
    """Where the matrix kernel's own plan is one split of at least 4 blocks of 128 rows, a short sequence runs on it; with
    fewer rows, or with units too few for one split each, on the float32 kernel."""
    name = lambda seq, layers: _lib.split_kernel(kv, kv * group, dim, bits, 0, _lib.TQ_F16, seq, num_layers=layers, n_splits=0, num_cus=CUS)
    for seq in (385, 450, 512):
        assert _splits(layers, kv, group, dim, bits, 0, seq) == 1
        assert "mx" in name(seq, layers)
        assert "mx" not in name(seq, 1)
    assert "mx" not in name(384, layers)


@pytest.mark.parametrize("kv,group,dim,bits,seq", [(4, 7, 64, 3, 30000), (8, 3, 128, 4, 32768), (2, 5, 256, 2, 20000)])
def test_explicit_counts_of_few_workgroups_keep_units_of_one(kv, group, dim, bits, seq):
    """An odd group is cut into units of 4 heads only where its units of 1 would be more workgroups than CUs."""
    heads = lambda n: _lib.split_kernel(kv, kv * group, dim, bits, 0, _lib.TQ_F16, seq, n_splits=n, num_cus=CUS).rstrip(">").split(",")[2]
    most = CUS // (kv * group)
    assert [heads(n) for n in (1, most, most + 1, 64, 0)] == ["1", "1", "4", "4", "4"]


@pytest.mark.parametrize("kv,group,dim,bits,seq", [(4, 8, 128, 4, 30001), (8, 16, 128, 2, 32768), (2, 24, 256, 4, 131072), (8, 8, 64, 4, 32768)])
def test_units_of_8_have_their_own_name(kv, group, dim, bits, seq):
    """The 8-head instance is named apart from the 4-head one, so an explicit count shows which of them it runs."""
    name = lambda n, g=group: _lib.split_kernel(kv, kv * g, dim, bits, 0, _lib.TQ_F16, seq, n_splits=n, num_cus=CUS)
    eight = f"decode_mx_kernel<{dim},true,{bits},8>"
    default = _splits(1, kv, group, dim, bits, 0, seq)
    assert name(0) == name(default) == eight
    assert name(1) == f"decode_mx_kernel<{dim},true{'' if bits == 4 else ',2'}>"  # too few workgroups for units of 8
    assert name(1, 4) == name(1)


@pytest.mark.parametrize("layers,kv,group,dim,bits,seq,most", [
    (16, 8, 8, 128, 4, 1309, 1), (16, 8, 8, 128, 4, 5376, 1), (16, 8, 8, 128, 4, 5377, 2),  # 128 units: from 43 blocks on
    (24, 4, 8, 128, 2, 768, 1), (12, 8, 8, 64, 4, 3968, 1), (12, 8, 8, 128, 4, 8192, 2),  # 96 units: from 32
    (9, 8, 8, 128, 4, 2176, 1), (9, 8, 8, 128, 4, 2177, 3),  # 72 units, 3 splits: from 18
    (16, 8, 8, 256, 4, 3968, 1), (16, 8, 8, 256, 4, 3969, 2),  # head_dim 256: from 32
    (8, 8, 8, 128, 4, 1024, 4),  # units of 4 have splits of their own to merge
])
def test_units_of_8_take_splits_that_pay_for_their_merge(layers, kv, group, dim, bits, seq, most):
    assert _splits(layers, kv, group, dim, bits, 0, seq) == most
    name = _lib.split_kernel(kv, kv * group, dim, bits, 0, _lib.TQ_F16, seq, num_layers=layers, n_splits=0, num_cus=CUS)
    assert name == f"decode_mx_kernel<{dim},true,{bits},8>"


@pytest.mark.parametrize("units,group,dim,bits,seq,most,cut", [
    (96, 5, 128, 3, 768, 1, True), (96, 5, 128, 3, 1536, 1, True), (96, 5, 128, 3, 2048, 2, True),
    (128, 3, 128, 3, 768, 1, True), (128, 3, 128, 3, 1024, 4, True), (64, 3, 128, 3, 768, 6, True),  # 64 units: CUs left idle
    (40, 7, 128, 4, 341, 1, True), (40, 7, 128, 4, 512, 1, True), (36, 7, 128, 4, 400, 3, True),  # 280 and 252 units of 1
    (96, 7, 64, 4, 768, 1, True), (128, 6, 256, 4, 768, 1, True), (128, 5, 128, 3, 600, 1, True),
    (128, 4, 128, 3, 768, 4, True),  # units that divide the group keep their plan
    (64, 7, 128, 0, 767, 1, False), (64, 7, 128, 0, 768, 4, True), (96, 5, 128, 0, 768, 1, True),  # dense rows: cut from 768 tokens on
])
def test_cut_groups_take_splits_that_pay_for_their_merge(units, group, dim, bits, seq, most, cut):
    assert _splits(units, 1, group, dim, bits, 0, seq) == most
    if bits:
        name = _lib.split_kernel(1, group, dim, bits, 0, _lib.TQ_F16, seq, num_layers=units, n_splits=0, num_cus=CUS)
        assert name == f"decode_kernel<PackedB{bits},{dim},{4 if cut else 1}>"


@pytest.mark.parametrize("kv,group,dim,bits,seq,expected", [
    (4, 6, 128, 3, 65536, {1: 4, 21: 4, 22: 4, 33: 2, 42: 2, 43: 4}),  # 12 and 8 units: 33 to 42 are two rounds of either
    (8, 10, 64, 2, 32768, {6: 4, 11: 2, 12: 2, 13: 4}),
])
def test_explicit_counts_that_save_no_round_keep_units_of_two(kv, group, dim, bits, seq, expected):
    heads = lambda n: _lib.split_kernel(kv, kv * group, dim, bits, 0, _lib.TQ_F16, seq, n_splits=n, num_cus=CUS).rstrip(">").split(",")[2]
    assert {n: int(heads(n)) for n in expected} == expected


@pytest.mark.parametrize("units,group,dim,bits,seq,most", [
    (384, 4, 256, 3, 2048, 1), (384, 4, 256, 3, 3072, 2), (640, 4, 256, 3, 3072, 1), (300, 4, 256, 3, 1536, 1),
    (384, 1, 256, 3, 1536, 2),  # one head at a time has half the set-up
    (384, 4, 256, 0, 768, 1), (384, 2, 256, 0, 2048, 1), (192, 8, 256, 0, 1331, 1), (320, 4, 128, 0, 1331, 1),
    (300, 1, 256, 0, 3072, 5), (192, 4, 128, 0, 2048, 2),
])
def test_balanced_counts_leave_plans_that_more_splits_slow_down(units, group, dim, bits, seq, most):
    assert _splits(units, 1, group, dim, bits, 0, seq) == most


@pytest.mark.parametrize("units,group,dim,bits,seq,expected", [
    (160, 6, 128, 4, 1311, 2), (96, 10, 64, 2, 1317, 2), (160, 6, 128, 4, 12000, 4), (176, 6, 128, 4, 1311, 4),
])
def test_one_split_of_two_rounds_keeps_units_of_two(units, group, dim, bits, seq, expected):
    """480 units of 2 and 320 (288) units of 4 are two rounds of workgroups either way; 528 are three."""
    name = lambda n: _lib.split_kernel(1, group, dim, bits, 0, _lib.TQ_F16, seq, num_layers=units, n_splits=n, num_cus=CUS)
    assert name(0) == name(_splits(units, 1, group, dim, bits, 0, seq)) == f"decode_kernel<PackedB{bits},{dim},{expected}>"
