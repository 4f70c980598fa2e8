"""Prefill plans below one round of 128-row tiles: the tile heights and k
splits the planner chooses, with the split sums made by a second launch, and
whole tiles where the stream-K schedule was; plain and SiLU-gated A, both
scale modes, ragged last row blocks, every output against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import lowbit_oracle as O
from tests.gpu_util import assert_close_f16, assert_reference_rounding, print_case, to_dev, to_np

pytestmark = pytest.mark.gpu


def _buffers(dev, m, n, k, g):
    import torch
    from neurova_amd import capi

    c = torch.full((m, n), float("nan"), dtype=torch.float16, device=dev)
    ws = torch.zeros((n // 128 * 16,), dtype=torch.int32, device=dev)
    # partials start as NaN: every one that is summed has to be written first
    sc = torch.full((capi.marlin_scratch_bytes(m, n, k, g),), 255, dtype=torch.uint8, device=dev)
    return c, ws, sc


@pytest.mark.parametrize("m,k,n,group,height,split", [
    (33, 2560, 1280, 128, 2, True),    # 32-row tiles, the last one of a single row
    (65, 1024, 2048, -1, 2, True),
    (40, 5120, 14336, 128, 4, True),   # 64-row tiles
    (180, 2048, 5120, -1, 4, True),
    (200, 5120, 7168, 128, 8, True),   # 128-row tiles split over K
    (200, 5120, 5120, 128, None, True),
    (1000, 2304, 9216, 128, 8, False),  # 288 whole tiles, 96 rows of the last block missing
    (40, 256, 512, 128, None, None),    # two scale groups
    (1000, 1024, 8448, 128, 8, False),  # few stages: whole tiles are ahead of stream-K from half a round on too
    (1536, 2048, 8448, -1, 8, False),
])
def test_shapes_vs_oracle(dev, m, k, n, group, height, split):
    import torch
    from neurova_amd import capi

    plan = capi.marlin_describe_plan(m, n, k, group)
    assert plan["form"] == "prefill", plan
    if height is not None:
        assert plan["chunks_or_row_blocks"] == height, plan
    if split is not None:
        assert (plan["splits"] > 1) == split and (plan["row_blocks_or_full_tiles"] == 0) == split, plan
    print_case("gemm-shape", m, k, n, group)
    codes, qw, _, sp, x = O.make_marlin_inputs(m, k, n, group, seed=3000 + m + k)
    c, ws, sc = _buffers(dev, m, n, k, group)
    a, b, s = to_dev(x, dev), to_dev(qw, dev), to_dev(sp, dev)
    got = []
    for _ in range(2):
        assert capi.marlin_gemm(a, b, c, s, ws, group, sc) == 0
        torch.cuda.synchronize()
        got.append(to_np(c).copy())
    ref = O.marlin_gemm(x, qw, sp, group)
    assert_close_f16(got[0], ref, what=f"m={m} k={k} n={n} g={group}")
    if group == 128:
        assert_reference_rounding(got[0], ref, x, qw, sp, group, what=f"m={m} k={k} n={n}")
    assert np.array_equal(got[0].view(np.uint16), got[1].view(np.uint16))
    assert int(ws.abs().sum()) == 0


@pytest.mark.parametrize("m,k,n", [(33, 1024, 768), (70, 2048, 1280), (130, 3072, 512), (260, 1024, 1280), (1100, 1024, 8448)])
def test_silu_packed_prefill_vs_oracle(dev, m, k, n):
    """The gated activations are formed once in scratch; the product over them
    takes the plain plans."""
    import torch
    from neurova_amd import capi

    print_case("silu-prefill", m, k, n)
    _, qw, _, sp, _ = O.make_marlin_inputs(m, k, n, 128, seed=3100 + m)
    mixed = np.random.default_rng(3100 + m).normal(0, 1, (m, 2 * k)).astype(np.float16)
    c, ws, sc = _buffers(dev, m, n, k, 128)
    assert capi.marlin_gemm_silu_packed(to_dev(mixed, dev), to_dev(qw, dev), c, to_dev(sp, dev), ws, 128, sc) == 0
    torch.cuda.synchronize()
    assert int(ws.abs().sum()) == 0
    assert_close_f16(to_np(c), O.marlin_gemm_silu_packed(mixed, qw, sp, k, 128), what=f"silu m={m}")


@pytest.mark.parametrize("m,k,n,group", [(29, 4096, 2048, 128), (31, 5120, 5120, -1), (32, 4224, 1280, 128),
                                         (30, 5120, 14336, 128), (28, 4096, 2048, 128)])
def test_wave_staged_decode_vs_oracle(dev, m, k, n, group):
    """M = 29..32 with a long K: each wave's batches of A go through its own LDS
    (M = 28: loaded as fragments); split and whole-K tiles, both scale modes."""
    import torch
    from neurova_amd import capi

    plan = capi.marlin_describe_plan(m, n, k, group)
    assert plan["form"] == "direct" and (plan["lds_bytes"] >= 4 * 32 * 272) == (m > 28), plan
    print_case("wave-staged", m, k, n, group)
    _, qw, _, sp, x = O.make_marlin_inputs(m, k, n, group, seed=3300 + m + k)
    c, ws, sc = _buffers(dev, m, n, k, group)
    assert capi.marlin_gemm(to_dev(x, dev), to_dev(qw, dev), c, to_dev(sp, dev), ws, group, sc) == 0
    torch.cuda.synchronize()
    ref = O.marlin_gemm(x, qw, sp, group)
    assert_close_f16(to_np(c), ref, what=f"m={m} k={k} n={n} g={group}")
    if group == 128:
        assert_reference_rounding(to_np(c), ref, x, qw, sp, group, what=f"m={m} k={k} n={n}")
    assert int(ws.abs().sum()) == 0


@pytest.mark.parametrize("m", [48, 300])
def test_workspace_of_one_entry(dev, m):
    """Plans whose splits are summed by a second launch use no workspace
    counters: the smallest workspace gives the same outputs."""
    import torch
    from neurova_amd import capi

    k, n = 2048, 2048
    print_case("one-entry workspace", m)
    _, qw, _, sp, x = O.make_marlin_inputs(m, k, n, 128, seed=3200 + m)
    a, b, s = to_dev(x, dev), to_dev(qw, dev), to_dev(sp, dev)
    outs = []
    for entries in (n // 128 * 16, 1):
        c, _, sc = _buffers(dev, m, n, k, 128)
        ws = torch.zeros((entries,), dtype=torch.int32, device=dev)
        assert capi.marlin_gemm(a, b, c, s, ws, 128, sc) == 0
        torch.cuda.synchronize()
        outs.append(to_np(c))
    assert np.array_equal(outs[0].view(np.uint16), outs[1].view(np.uint16))


@pytest.mark.parametrize("m,k,n", [(20, 256, 512), (48, 2048, 2048), (300, 1024, 2048)])
def test_one_entry_workspace_without_scratch(dev, m, k, n):
    """With neither split counters nor scratch the tiles run whole."""
    import torch
    from neurova_amd import capi

    print_case("no scratch", m, k, n)
    _, qw, _, sp, x = O.make_marlin_inputs(m, k, n, 128, seed=3300 + m)
    c, _, _ = _buffers(dev, m, n, k, 128)
    ws = torch.zeros((1,), dtype=torch.int32, device=dev)
    st = capi.marlin_gemm(to_dev(x, dev), to_dev(qw, dev), c, to_dev(sp, dev), ws, 128, None)
    assert st == 0, capi.status_string(st)
    assert_close_f16(to_np(c), O.marlin_gemm(x, qw, sp, 128), what=f"m={m} k={k} n={n}")


@pytest.mark.parametrize("m,k,n", [(20, 256, 512), (33, 1024, 768), (64, 2048, 1280), (200, 1024, 2048), (1030, 256, 256)])
@pytest.mark.parametrize("group", [128, -1])
def test_silu_packed_prefill_without_scratch(dev, m, k, n, group):
    """Without scratch for the gated activations every tile gates its own rows:
    whole tiles with a one-entry workspace and no scratch, split ones with scratch
    for the partials alone; the same outputs as with scratch up to the order of
    the sums."""
    import torch
    from neurova_amd import capi

    print_case("silu no scratch", m, k, n, group)
    _, qw, _, sp, _ = O.make_marlin_inputs(m, k, n, group, seed=3400 + m)
    mixed = np.random.default_rng(3400 + m).normal(0, 1, (m, 2 * k)).astype(np.float16)
    a, b, s = to_dev(mixed, dev), to_dev(qw, dev), to_dev(sp, dev)
    ref = O.marlin_gemm_silu_packed(mixed, qw, sp, k, group)
    c, ws, sc = _buffers(dev, m, n, k, group)
    act = -(-m * k * 2 // 256) * 256
    assert capi.marlin_describe_plan(m, n, k, group, 1)["form"] == "prefill" and sc.numel() >= act
    one = torch.zeros((1,), dtype=torch.int32, device=dev)
    for workspace, scratch in ((one, None), (one, sc[1:]), (ws, sc[:act - 256])):
        c.fill_(float("nan"))
        st = capi.marlin_gemm_silu_packed(a, b, c, s, workspace, group, scratch)
        if st == capi.LB_ERR_SCRATCH and workspace is ws:  # its partials need more than that
            torch.cuda.synchronize()
            assert bool(torch.isnan(c).all())
            continue
        assert st == 0, capi.status_string(st)
        torch.cuda.synchronize()
        assert int(ws.abs().sum()) == 0 and int(one.abs().sum()) == 0
        assert_close_f16(to_np(c), ref, what=f"m={m} k={k} n={n} g={group}")


def test_scratch_is_refused_as_missing_before_anything_runs(dev):
    """A workspace that holds the split counters asks for splits: without scratch
    for their partials the call is refused, plain and SiLU-gated."""
    import torch
    from neurova_amd import capi

    m, k, n = 48, 2048, 2048
    print_case("scratch refused", m, k, n)
    _, qw, _, sp, x = O.make_marlin_inputs(m, k, n, 128, seed=3500)
    c, ws, _ = _buffers(dev, m, n, k, 128)
    b, s = to_dev(qw, dev), to_dev(sp, dev)
    mixed = np.concatenate([x, x], axis=1)
    assert capi.marlin_gemm(to_dev(x, dev), b, c, s, ws, 128, None) == capi.LB_ERR_SCRATCH
    assert capi.marlin_gemm_silu_packed(to_dev(mixed, dev), b, c, s, ws, 128, None) == capi.LB_ERR_SCRATCH
    torch.cuda.synchronize()
    assert bool(torch.isnan(c).all()) and int(ws.abs().sum()) == 0


@pytest.mark.parametrize("op,m,k,n", [("plain", 2048, 17408, 256), ("plain", 1024, 1024, 4096), ("gated", 300, 2048, 1024),
                                      ("argmax", 40, 1024, 2048), ("plain", 4, 5120, 5120)])
def test_op_scratch_is_its_plans_own(dev, op, m, k, n):
    """The torch ops keep scratch for the plans they run, in whole MiB a stream: a
    plain product none for gated activations."""
    import torch
    import langburst_cuda as lc
    from neurova_amd import capi

    need = capi.marlin_describe_plan(m, n, k, 128, ("plain", "gated", "argmax").index(op))["scratch_bytes"]
    print_case("op scratch", op, m, k, n, need)
    q = torch.zeros((k // 16, 2 * n), dtype=torch.int32, device=dev)
    s = torch.ones((k // 128, n), dtype=torch.float16, device=dev)
    x = torch.zeros((m, k * (2 if op == "gated" else 1)), dtype=torch.float16, device=dev)
    out = torch.empty((m, n), dtype=torch.float16, device=dev)
    ws = torch.zeros((n // 128 * 16,), dtype=torch.int32, device=dev)
    best, state = (torch.zeros((m,), dtype=torch.int64, device=dev) for _ in range(2))
    sync = torch.zeros((2,), dtype=torch.int32, device=dev)
    side = torch.cuda.Stream()  # scratch is kept per stream
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        before = torch.cuda.memory_allocated(dev)
        if op == "plain":
            lc.lowbit_marlin_gemm_out(q, s, x, out, ws, k, 128)
        elif op == "gated":
            lc.lowbit_marlin_gemm_silu_packed_out(q, s, x, out, ws, k, 128)
        else:
            lc.lowbit_marlin_gemm_argmax_out(q, s, x, out, ws, state, best, sync, 1, k, 128)
        kept = torch.cuda.memory_allocated(dev) - before
    torch.cuda.synchronize()
    assert kept <= -(-need // 2 ** 20) * 2 ** 20, (kept, need)
