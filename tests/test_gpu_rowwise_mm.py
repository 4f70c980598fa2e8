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


# (batch, rows): output blocks of 16 and 32 rows, one, two and four row blocks, eight and four
# waves, and the four tile shapes, at rows of up to three stages
@pytest.mark.parametrize("batch,rows", [(16, 4100), (32, 4100), (32, 8200), (64, 4100), (130, 4100), (65, 16400),
                                        (130, 5504), (512, 6144), (512, 12300)])
@pytest.mark.parametrize("bits,cols,group", [(2, 256, 64), (3, 300, 32), (4, 384, 128), (7, 270, 32), (8, 256, 128)])
def test_launch_forms_vs_oracle(dev, batch, rows, bits, cols, group):
    print_case("mm-form", batch, rows, bits, cols, group)
    _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, group, batch=batch, seed=bits + rows + batch)
    _check(_gemm(dev, packed, scales, x, cols, group, bits), x, packed, scales, cols, group, bits, f"{batch}x{rows}")


# (batch, rows) for every launch form on 256 compute units, in the order of
# launch_sps (lb_rowwise_mm.hip): up to 16 rows -- 48, 32 (two stages in flight, then
# one) and 16 output rows a workgroup; up to 32 -- 48 and 32 rows on four waves, 32
# and 16 on eight, blocks of 16; split K above -- four row blocks on eight and on four
# waves, two row blocks of 16 output rows; the four tile shapes
_FORMS = [(16, 16400), (8, 4100), (16, 8200), (16, 2100), (32, 17408), (32, 8300), (32, 4100), (32, 2100), (32, 1100),
          (64, 4100), (130, 4100), (48, 1100), (512, 12300), (512, 6144), (65, 16400), (130, 5504)]


@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("group", [32, 64, 128])
def test_pipelines_vs_oracle(dev, bits, group):
    """Every launch form at every width and scale layout with several stages a wave
    (25 whole ones over four or eight waves, or for one tile) and a ragged end:
    slots issued again, LDS rows overwritten stage after stage.  Output rows of the
    first and last workgroups and some between are checked."""
    import torch
    from neurova_amd import capi

    cols = 25 * 128 + 7
    gen = torch.Generator(device=dev)
    gen.manual_seed(bits * 1000 + group)
    for batch, rows in _FORMS:
        print_case("mm-pipeline", bits, group, batch, rows)
        q = torch.randint(0, 256, (rows, (cols * bits + 7) // 8), dtype=torch.uint8, device=dev, generator=gen)
        s = (torch.rand((rows, -(-cols // group)), device=dev, generator=gen) * 0.01 + 1e-3).half()
        x = torch.randn((batch, cols), device=dev, generator=gen).half()
        y = torch.full((batch, rows), float("nan"), dtype=torch.float16, device=dev)
        assert capi.lowbit_gemm(q, s, x, y, cols, group, bits) == 0
        assert bool(torch.isfinite(y).all())
        pick = np.unique(np.concatenate([np.arange(0, 49, 3), [63, 64, 127, 128, 255, 256], np.linspace(300, rows - 50, 9).astype(int),
                                         np.arange(rows - 49, rows, 4), [rows - 1]]))
        idx = torch.from_numpy(pick).to(dev)
        _check(to_np(y[:, idx]), to_np(x), to_np(q[idx]), to_np(s[idx]), cols, group, bits, f"b{bits} g{group} {batch}x{rows}")


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


@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("batch", [1, 3, 40, 130])
def test_every_tail_length(dev, bits, batch):
    """Rows that end 1 to 127 columns into a stage of 128, with and without a whole
    stage before: the end of a row is loaded by 16-byte words shifted into place,
    rows below 16 bytes by bytes."""
    for cols in [*range(1, 34), 63, 64, 65, 100, 119, 120, 121, 127, *range(129, 146), 191, 192, 200, 247, 249, 255]:
        rows = 4100 if batch == 130 and cols == 249 else 21  # (four-wave tiles from 64 x 64 tiles for every CU)
        print_case("mm-tail", bits, batch, cols)
        _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, 32, batch=batch, seed=bits + cols + batch)
        got = _gemm(dev, packed, scales, x, cols, 32, bits)
        _check(got, x, packed, scales, cols, 32, bits, f"b{bits} K={cols}")


def test_tiny_rows_beyond_one_round_of_waves(dev):
    """Code rows below 16 bytes: the byte-wise kernel up to 80 waves per CU, the
    matrix-core product beyond."""
    for batch, rows in ((4, 20480), (4, 20481), (5, 20481)):
        print_case("mm-tiny", batch, rows)
        _, packed, scales, x = O.make_rowwise_inputs(rows, 7, 8, 32, batch=batch, seed=batch)
        _check(_gemm(dev, packed, scales, x, 7, 32, 8), x, packed, scales, 7, 32, 8, f"{batch}x{rows}")


def test_ragged_rows_run_like_whole_ones(dev):
    """A row that ends 120 columns into its last stage takes no longer than one that
    fills it, beyond 1.4 times for the noise of either (1.8 times when the end of a
    row was loaded by bytes)."""
    import torch
    from neurova_amd import capi

    rows, bits, best = 17408, 4, {}
    for cols in (5240, 5248):
        pc = cols * bits // 8
        q = torch.randint(0, 256, (rows, pc), dtype=torch.uint8, device=dev)
        s = torch.full((rows, 41), 0.01, dtype=torch.float16, device=dev)
        x, y = torch.ones((2, cols), dtype=torch.float16, device=dev), torch.empty((2, rows), dtype=torch.float16, device=dev)
        print_case("mm-ragged-time", cols)
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                assert capi.lowbit_gemm(q, s, x, y, cols, 128, bits) == 0
            b.record()
            torch.cuda.synchronize()
            best[cols] = min(best.get(cols, 1e9), a.elapsed_time(b))
    assert best[5240] < 1.4 * best[5248], best


@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("cols,group", [(8191, 128), (8193, 128), (8194, 64), (8290, 32), (12280, 128), (17400, 32), (17407, 64)])
def test_long_ragged_row_of_few_outputs(dev, bits, cols, group):
    """One row from K = 8192 on over blocks of 16 output rows on at most half of 256
    compute units (2048 output rows): sixteen waves share it, some with one stage more
    than others, and the ragged end is the next wave's; eight waves on either side."""
    import langburst_cuda as lc
    import torch

    for rows in (1, 17, 2048, 2049):
        if rows > 17 and cols != 8290:
            continue
        print_case("mm-long-row", bits, rows, cols, group)
        _, packed, scales, x = O.make_rowwise_inputs(rows, cols, bits, group, batch=1, seed=bits + cols)
        got = _gemm(dev, packed, scales, x, cols, group, bits)
        _check(got, x, packed, scales, cols, group, bits, f"b{bits} {rows}x{cols}")
        # two matrices in one launch: half the output rows each up to the same line
        q, s, xd = to_dev(packed, dev), to_dev(scales, dev), to_dev(x[0], dev)
        q2 = torch.flip(q, (0,)).contiguous()
        a, b = lc.lowbit_gemv_pair(q, s, q2, s, xd, cols, group, bits)
        _check(to_np(a)[None], x, packed, scales, cols, group, bits, "pair 0")
        _check(to_np(b)[None], x, packed[::-1].copy(), scales, cols, group, bits, "pair 1")


def test_long_ragged_row_of_few_outputs_time(dev):
    """Sixteen waves on such a row: no slower than 0.93 of the same row in a batch of
    two, which takes eight (measured 0.76 to 0.8)."""
    import torch
    from neurova_amd import capi

    rows, bits, cols, best = 2048, 4, 17400, {}
    q = torch.randint(0, 256, (rows, cols * bits // 8), dtype=torch.uint8, device=dev)
    s = torch.full((rows, -(-cols // 128)), 0.01, dtype=torch.float16, device=dev)
    for batch in (1, 2):
        x = torch.ones((batch, cols), dtype=torch.float16, device=dev)
        y = torch.empty((batch, rows), dtype=torch.float16, device=dev)
        print_case("mm-long-row-time", batch)
        assert capi.lowbit_gemm(q, s, x, y, cols, 128, bits) == 0
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                assert capi.lowbit_gemm(q, s, x, y, cols, 128, bits) == 0
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            graph.replay()
            a.record()
            graph.replay()
            b.record()
            torch.cuda.synchronize()
            best[batch] = min(best.get(batch, 1e9), a.elapsed_time(b))
    assert best[1] < 0.93 * best[2], best
