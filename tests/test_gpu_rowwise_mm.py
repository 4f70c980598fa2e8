"""The rowwise matrix-core product (batches, and one-row calls whose rows are
ragged or not dword-aligned) against the float64 product of the oracle's
dequantised weights.

Bound per output: the fp16 rounding (half a step) of a value within the fp32
error of the sum, (K / 32 + 16) roundings of partial sums no larger than
sum |x w| -- an MFMA rounds once per 32 k, then one FMA per scale group, one add
per wave.
"""
from __future__ import annotations

import numpy as np
import pytest

from oracle import lowbit_oracle as O
from tests.gpu_util import print_case, to_dev, to_np

pytestmark = pytest.mark.gpu


def _check(got, x, packed, scales, cols, group, bits, what):
    w = O.rowwise_dequant_f32(packed, scales, cols, group, bits).astype(np.float64)
    x64 = np.asarray(x, dtype=np.float16)[:, :cols].astype(np.float64)
    ref = x64 @ w.T
    err32 = (cols / 32 + 16) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w).T)
    half_step = np.spacing(np.abs(ref).astype(np.float16) + np.float16(0)).astype(np.float64) / 2
    bad = np.abs(got.astype(np.float64) - ref) > half_step * (1 + 2.0 ** -10) + err32
    assert np.isfinite(got).all() and not bad.any(), f"{what}: {int(bad.sum())} of {bad.size} outside the bound"


def _gemm(dev, packed, scales, x, cols, group, bits):
    import torch
    from neurova_amd import capi

    y = torch.full((x.shape[0], packed.shape[0]), float("nan"), dtype=torch.float16, device=dev)
    st = capi.lowbit_gemm(to_dev(packed, dev), to_dev(scales, dev), to_dev(x, dev), y, cols, group, bits)
    assert st == 0, capi.status_string(st)
    return to_np(y)


@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("rows,cols,group", [
    (1, 1, 32), (17, 7, 128), (33, 127, 32), (16, 128, 64), (31, 129, 64), (48, 257, 32), (37, 300, 96),
    (130, 1024, 128), (19, 2051, 256), (40, 515, 1000),  # one group longer than the row
])
@pytest.mark.parametrize("batch", [1, 2, 16, 17, 33])
def test_edges_vs_oracle(dev, bits, rows, cols, group, batch):
    print_case("mm", bits, rows, cols, group, batch)
    _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, group, batch=batch, seed=bits + rows + batch)
    _check(_gemm(dev, packed, scales, x, cols, group, bits), x, packed, scales, cols, group, bits, f"b{bits}")


# (batch, rows): one of each launch form on 256 compute units -- output blocks of 16 and 32
# rows, one, two and four row blocks, eight and four waves, and the four tile shapes
@pytest.mark.parametrize("batch,rows", [(16, 4100), (32, 4100), (32, 8200), (64, 4100), (130, 4100), (65, 16400),
                                        (130, 5504), (512, 6144), (512, 12300)])
@pytest.mark.parametrize("bits,cols,group", [(2, 256, 64), (3, 300, 32), (4, 384, 128), (7, 270, 32), (8, 256, 128)])
def test_launch_forms_vs_oracle(dev, batch, rows, bits, cols, group):
    print_case("mm-form", batch, rows, bits, cols, group)
    _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, group, batch=batch, seed=bits + rows + batch)
    _check(_gemm(dev, packed, scales, x, cols, group, bits), x, packed, scales, cols, group, bits, f"{batch}x{rows}")


@pytest.mark.parametrize("batch", [8, 9, 17, 32])
@pytest.mark.parametrize("rows", [8192, 8193, 16385])
@pytest.mark.parametrize("bits,cols,group", [(2, 1152, 128), (4, 1300, 128), (3, 300, 32), (8, 257, 64)])
def test_workgroups_per_cu_vs_oracle(dev, batch, rows, bits, cols, group):
    """Up to one, up to two and more workgroups of 32 rows for each of 256 compute
    units: blocks of 32 or 48 rows, four or eight waves, one or two stages in
    flight, the last block of a single row."""
    print_case("mm-cu", batch, rows, bits, cols, group)
    _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, group, batch=batch, seed=bits + rows + batch)
    _check(_gemm(dev, packed, scales, x, cols, group, bits), x, packed, scales, cols, group, bits, f"{batch}x{rows}")


@pytest.mark.parametrize("bits", [3, 4, 8])
@pytest.mark.parametrize("batch", [3, 40])
def test_wide_activation_rows(dev, bits, batch):
    """Activation rows longer than the product's columns, at an odd stride: what
    lies past them (infinities) is not used; wider code and scale rows likewise."""
    cols, group, rows = 200, 64, 50
    print_case("mm-wide", bits, batch)
    _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, group, batch=batch, seed=bits)
    wide = np.concatenate([x, np.full((batch, 5), np.inf, dtype=np.float16)], axis=1)
    packed = np.concatenate([packed, np.full((rows, 3), 0xA5, dtype=np.uint8)], axis=1)
    scales = np.concatenate([scales, np.full((rows, 2), np.nan, dtype=np.float16)], axis=1)
    _check(_gemm(dev, np.ascontiguousarray(packed), np.ascontiguousarray(scales), wide, cols, group, bits), x, packed,
           scales, cols, group, bits, f"b{bits}")


@pytest.mark.parametrize("bits", [2, 5, 8])
def test_special_values(dev, bits):
    """An infinity or NaN in one activation row stays in that row's outputs."""
    cols, group, rows = 256, 128, 40
    print_case("mm-special", bits)
    _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, group, batch=20, seed=bits)
    x[3, 70], x[18, 5] = np.inf, np.nan
    got = _gemm(dev, packed, scales, x, cols, group, bits)
    assert not np.isfinite(got[3]).any() and np.isnan(got[18]).all()
    keep = [i for i in range(20) if i not in (3, 18)]
    _check(got[keep], x[keep], packed, scales, cols, group, bits, f"b{bits}")


@pytest.mark.parametrize("batch", [3, 40])
@pytest.mark.parametrize("rows", [40, 16400])
@pytest.mark.parametrize("cols,group", [(160, 32), (190, 64)])
def test_infinite_scale_of_the_last_group(dev, batch, rows, cols, group):
    """An infinite scale of a ragged row's last group gives infinities, not NaN."""
    print_case("mm-inf-scale", batch, rows, cols, group)
    _, packed, scales, x = O.make_rowwise_inputs(rows, cols, 4, group, batch=batch, seed=rows + batch)
    scales[5, -1] = np.inf
    got = _gemm(dev, packed, scales, np.abs(x) + np.float16(1), cols, group, 4)
    w = O.rowwise_dequant_f32(packed, np.ones_like(scales), cols, group, 4).astype(np.float64)
    last = cols - (scales.shape[1] - 1) * group
    dot = (np.abs(x) + np.float16(1)).astype(np.float64)[:, -last:] @ w[5, -last:]
    assert np.array_equal(got[:, 5], np.where(dot > 0, np.inf, -np.inf).astype(np.float16))
    assert np.isfinite(np.delete(got, 5, axis=1)).all()


@pytest.mark.parametrize("bits", [5, 6, 7])
@pytest.mark.parametrize("rows,cols,group", [
    (7, 32, 32), (9, 2016, 32), (16, 2080, 128), (5, 4128, 64), (33, 6176, 128), (8, 10240, 64), (3, 10272, 128),
    (5127, 10272, 128), (5120, 10240, 64),  # two rows a wave above five lane steps, one below
])
def test_staged_row_of_whole_units(dev, bits, rows, cols, group):
    """One activation row at 5, 6 and 7 bits, staged in LDS: one to five lane
    steps prefetched, more than five, ragged last workgroups; the pair of
    matrices equals two single calls."""
    import torch
    from neurova_amd import capi

    print_case("staged-row", bits, rows, cols, group)
    _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, group, seed=bits + rows)
    q, s, xd = to_dev(packed, dev), to_dev(scales, dev), to_dev(x[0], dev)
    y = torch.full((rows,), float("nan"), dtype=torch.float16, device=dev)
    assert capi.lowbit_gemv(q, s, xd, y, cols, group, bits) == 0
    got = to_np(y)
    _check(got.reshape(1, -1), x, packed, scales, cols, group, bits, f"b{bits}")
    if rows < 100:
        import langburst_cuda as lc

        q2 = torch.flip(q, (0,)).contiguous()
        a, b = lc.lowbit_gemv_pair(q, s, q2, s, xd, cols, group, bits)
        assert torch.equal(a, y) and torch.equal(b, lc.lowbit_gemv(q2, s, xd, cols, group, bits))
