"""Tile items shared by a workgroup's four waves, and the launch order that puts
long items first: same sums in another order, so the MFMA routes keep their bar,
1e-5 of |A||B| against fp64 of the quantised inputs."""
import numpy as np
import pytest
import torch

from conftest import assert_close_scaled

pytestmark = pytest.mark.gpu

import ra_spmm  # noqa: E402
from ra_spmm import synthetic as S  # noqa: E402

MAKE = {0: ra_spmm.make_tc_direct_plan, 1: ra_spmm.make_community_tc_plan, 2: ra_spmm.make_segment_hybrid_plan}


def _check(oracle, g, kind, N, rows=0, dtype="fp16", build="auto", columns=None):
    B = np.random.default_rng(N + rows).standard_normal((g.K, N)).astype(np.float32)
    rp, ci, vl = g.torch("cuda") if build != "host" else [torch.from_numpy(x) for x in (g.rowptr, g.colind, g.vals)]
    plan = MAKE[kind](rp, ci, vl, g.M, g.K, N, value_dtype=dtype, build=build, rows_per_window=rows)
    C = ra_spmm.run_tile_plan_route(plan, torch.from_numpy(B).cuda(), dtype)
    assert torch.equal(C, ra_spmm.run_tile_plan_route(plan, torch.from_numpy(B).cuda(), dtype))
    quant = oracle.quantize_f16 if dtype == "fp16" else oracle.quantize_bf16
    qv, qb = quant(g.vals), quant(B)
    assert_close_scaled(C.cpu().numpy(), oracle.spmm_tile_f64(g.rowptr, g.colind, g.vals, B, dtype.replace("fp", "f")),
                        oracle.spmm_f64(g.rowptr, g.colind, np.abs(qv), np.abs(qb)), 1e-5, f"{kind} {N} {rows}")
    return plan


# Every column-run width (1, 2, 4, 8) and ragged widths; all items are shared here (few windows of several steps).
@pytest.mark.parametrize("N", [16, 17, 32, 63, 64, 100, 128, 250, 257])
@pytest.mark.parametrize("rows", [8, 16, 32])
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_shared_items(oracle, N, rows, kind):
    print(f"[shared] N={N} rows={rows} kind={kind}", flush=True)
    g = S.random_csr(301, 900, 60.0, seed=N, skew=1.0, empty_frac=0.1)
    _check(oracle, g, kind, N, rows, dtype="bf16" if N % 2 else "fp16")


# Windows of equal length on both sides of the room for four times the waves: 8 rows, N = 128, 2 * 4096 (6.3 steps); 16 rows,
# N = 128, 0.8 * 4096 (4 steps); 32 rows, N = 128, 0.6 * 3072 (8 steps).  Also items of just under and over 6 steps.
@pytest.mark.parametrize("rows,windows,degree", [(8, 2040, 26), (8, 2300, 26), (8, 400, 22), (8, 400, 25), (16, 800, 8),
                                                 (16, 1000, 8), (32, 440, 8), (32, 480, 8)])
def test_room_for_shared_items(oracle, rows, windows, degree):
    print(f"[room] rows={rows} windows={windows} degree={degree}", flush=True)
    _check(oracle, S.random_csr(rows * windows - 3, 1500, degree, seed=rows), 0, 128, rows)


# Even windows over a B just below and just past the size from which their gathers keep the branches (N = 128: whole rows;
# N = 512: the slices of TC_DIRECT run outermost; N = 32: narrow runs), fp16 and bf16.
@pytest.mark.parametrize("K,N", [(31_249, 128), (31_250, 128), (31_250, 512), (62_500, 64), (109_374, 32), (109_375, 32)])
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_even_windows_over_a_large_B(oracle, K, N, kind):
    print(f"[even] K={K} N={N} kind={kind}", flush=True)
    _check(oracle, S.random_csr(805, K, 32.0 if N == 32 else 11.0, seed=K % 97), kind, N, 8, dtype="bf16" if kind else "fp16")


def _long_rows(M, K, every, length, seed):
    """Short rows with a long one every `every` rows."""
    rng = np.random.default_rng(seed)
    deg = np.full(M, 3)
    deg[::every] = length
    rowptr = np.zeros(M + 1, np.int32)
    np.cumsum(deg, out=rowptr[1:])
    cols = np.concatenate([np.sort(rng.choice(K, d, replace=False)) for d in deg]).astype(np.int32)
    return S.Graph(rowptr, cols, rng.standard_normal(cols.size).astype(np.float32), M, K)


# Windows of 1024, 1025 (just long) and 1600 vectors among short ones, in enough items (M / 8 > 2048) that only the
# long ones are shared; with column partitions every partition has its own order.
@pytest.mark.parametrize("length", [1003, 1005, 1600])
@pytest.mark.parametrize("parts", [1, 2])
@pytest.mark.parametrize("build", ["auto", "host"])
def test_long_items_first(oracle, monkeypatch, length, parts, build):
    if build == "host" and parts > 1:
        pytest.skip("the host builder makes no column partitions")
    monkeypatch.setenv("RA_TILE_COL_PARTS", str(parts))
    g = _long_rows(17_000, 2500, 1500, length, seed=length)
    plan = _check(oracle, g, 0, 64, 8, build=build)
    assert plan.num_segments * plan.col_parts > 2048
    _check(oracle, g, 1, 40, 8, build=build)


def test_order_only_where_items_are_long():
    """A window of SEGMENT_HYBRID is cut into segments that are never long: its plan has no launch order of its own,
    however long the window.  A whole window of TC_DIRECT comes first."""
    g = _long_rows(1700, 2500, 1500, 1600, seed=9)
    rp, ci, vl = g.torch("cuda")
    for rows in (8, 32):
        plan = ra_spmm.make_segment_hybrid_plan(rp, ci, vl, g.M, g.K, 64, rows_per_window=rows)
        assert plan.max_window_blocks * (8 if rows == 8 else 32) > 1024
        assert ra_spmm.export_tile_plan(plan, "item_order").numel() == 0
        plan = ra_spmm.make_tc_direct_plan(rp, ci, vl, g.M, g.K, 64, rows_per_window=rows)
        first = sorted({0, 1500 // rows})
        rest = [w for w in range(plan.num_windows) if w not in first]
        assert ra_spmm.export_tile_plan(plan, "item_order").tolist() == first + rest
    host = ra_spmm.make_segment_hybrid_plan(*(t.cpu() for t in (rp, ci, vl)), g.M, g.K, 64, build="host")
    assert ra_spmm.export_tile_plan(host, "item_order").numel() == 0
