"""Packets of four columns and of one at any width N and alignment, and the depth of the gather rounds.

A row's last packet starts at column N - 4 and stores only the columns that no
other packet owns; launches of fewer waves keep more gathers in flight.  Neither
changes the fma chain of an output element, so every result is the oracle's bit
for bit (rows of ZERO_OVERHEAD_CSR over 256 nonzeros: 1e-5 of |A||B|).
"""
import numpy as np
import pytest
import torch

from conftest import assert_close_scaled, assert_fp32_route

pytestmark = pytest.mark.gpu

import ra_spmm  # noqa: E402
from ra_spmm import synthetic as S  # noqa: E402


def _B(K, N, seed):
    return np.random.default_rng(seed).standard_normal((K, N)).astype(np.float32)


# 1-3: one column a lane, as where ragged rows are narrow; 4-9, 15-17: one to five packets; 63-65, 127-129: lane-group edges; 253-259: column slices.
@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7, 9, 15, 17, 31, 33, 63, 65, 127, 129, 253, 257, 259, 510, 1001])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_every_width_and_alignment(oracle, N, shift):
    print(f"[packets] N={N} shift={shift}", flush=True)
    g = S.random_csr(601, 500, 9.0, seed=N, skew=0.4, empty_frac=0.05, max_deg=450)
    deg = np.diff(g.rowptr)
    assert deg.max() > 256 and (deg == 0).any()
    B = _B(g.K, N, seed=N + shift)
    seq = oracle.spmm_seq_f32(g.rowptr, g.colind, g.vals, B)
    rp, ci, vl = g.torch("cuda")
    storage = torch.full((B.size + shift,), float("nan"), device="cuda")
    Bd = storage[shift:].view(g.K, N)  # a view `shift` floats into its storage
    Bd.copy_(torch.from_numpy(B))
    np.testing.assert_array_equal(ra_spmm.spmm_csr_direct(rp, ci, vl, Bd).cpu().numpy(), seq)
    plan = ra_spmm.make_zero_overhead_plan(rp, g.M, g.K)
    C = ra_spmm.run_zero_overhead_plan(plan, rp, ci, vl, Bd).cpu().numpy()
    np.testing.assert_array_equal(C[deg <= 256], seq[deg <= 256])
    assert_close_scaled(C, oracle.spmm_f64(g.rowptr, g.colind, g.vals, B),
                        oracle.spmm_f64(g.rowptr, g.colind, np.abs(g.vals), np.abs(B)), 1e-5, f"zo N={N}")


# Ragged widths at the bounds of the rule for one column a lane (N = 8, 16, 32, 128; mean row 8, 16; 3,000 bytes a wave and
# 8 MB of B) and of the rule for slices (N = 385, 441; 16,000 and 25,000 rows).
@pytest.mark.parametrize("rows,mean,widths", [(2000, 3.0, (9, 13, 401)), (2000, 10.0, (8, 11, 17, 31)), (2000, 18.0, (30, 33, 127)),
                                              (17_000, 14.0, (126, 130, 385)), (26_000, 3.0, (301, 441))])
def test_packets_and_slices_of_ragged_rows(oracle, rows, mean, widths):
    g = S.random_csr(rows, rows, mean, seed=rows, skew=0.9, empty_frac=0.02, max_deg=700)
    deg = np.diff(g.rowptr)
    rp, ci, vl = g.torch("cuda")
    plan = ra_spmm.make_zero_overhead_plan(rp, g.M, g.K)
    host = ra_spmm.make_zero_overhead_plan(rp.cpu(), g.M, g.K, build="host")
    for N in widths:
        print(f"[ragged] rows={rows} N={N}", flush=True)
        B = _B(g.K, N, seed=N)
        seq = oracle.spmm_seq_f32(g.rowptr, g.colind, g.vals, B)
        Bd = torch.from_numpy(B).cuda()
        np.testing.assert_array_equal(ra_spmm.spmm_csr_direct(rp, ci, vl, Bd).cpu().numpy(), seq)
        C = ra_spmm.run_zero_overhead_plan(plan, rp, ci, vl, Bd).cpu().numpy()
        np.testing.assert_array_equal(ra_spmm.run_zero_overhead_plan(host, rp, ci, vl, Bd).cpu().numpy(), C)
        np.testing.assert_array_equal(C[deg <= 256], seq[deg <= 256])
        assert_close_scaled(C, oracle.spmm_f64(g.rowptr, g.colind, g.vals, B),
                            oracle.spmm_f64(g.rowptr, g.colind, np.abs(g.vals), np.abs(B)), 1e-5, f"zo N={N}")


# (30, 210,000): 25 MB of B, one column a lane.
@pytest.mark.parametrize("N,K", [(47, 900), (129, 900), (258, 900), (30, 210_000)])
def test_resumed_chains_at_ragged_widths(oracle, monkeypatch, N, K):
    """The FP32 route over column partitions continues each element's chain from C: a packet that overlaps its
    neighbour must neither add to the neighbour's columns twice nor store them."""
    monkeypatch.setenv("RA_TILE_COL_PARTS", "4")
    g = S.random_csr(400, K, 40.0, seed=N)
    B = _B(g.K, N, seed=N)
    rp, ci, vl = g.torch("cuda")
    plan = ra_spmm.make_tc_direct_plan(rp, ci, vl, g.M, g.K, N)
    assert plan.col_parts == 4
    C = ra_spmm.run_tc_direct_plan_tf32(plan, torch.from_numpy(B).cuda()).cpu().numpy()
    stored = oracle.quantize_f16_scaled(g.vals, plan.value_scale_log2)
    assert_fp32_route(C, g.rowptr, g.colind, stored, B, oracle)


# Lanes a row, rows a wave: N = 16 -> 16 rows, 64 -> 4, 128 -> 2.  The row counts lie on both sides of 2^13 and 2^16 waves.
@pytest.mark.parametrize("N,rows", [(32, 65_000), (32, 66_000), (64, 32_000), (64, 33_500), (128, 16_300), (128, 16_500),
                                    (128, 131_000), (128, 131_200)])
def test_depths_of_the_gather_rounds(oracle, N, rows):
    print(f"[depth] N={N} rows={rows}", flush=True)
    g = S.random_csr(rows, 300, 5.0, seed=rows, empty_frac=0.05)
    B = _B(g.K, N, seed=N)
    seq = oracle.spmm_seq_f32(g.rowptr, g.colind, g.vals, B)
    rp, ci, vl = g.torch("cuda")
    Bd = torch.from_numpy(B).cuda()
    np.testing.assert_array_equal(ra_spmm.spmm_csr_direct(rp, ci, vl, Bd).cpu().numpy(), seq)
    plan = ra_spmm.make_zero_overhead_plan(rp, g.M, g.K)
    np.testing.assert_array_equal(ra_spmm.run_zero_overhead_plan(plan, rp, ci, vl, Bd).cpu().numpy(), seq)


# A launch of 16 gathers in flight (N = 64 and 128, few rows), one of 8 (N = 48, 40,000 rows) and several packets a lane
# with rows of under 3 nonzeros (N = 300, over 2^16 waves).  Rows of 0..4, 0..8 and 0..9 nonzeros: a wave whose rows fit
# a shorter round takes it.
@pytest.mark.parametrize("longest", [4, 5, 8, 9])
@pytest.mark.parametrize("N,rows", [(64, 1000), (128, 515), (48, 40_000), (300, 66_000)])
def test_rounds_of_short_rows(oracle, N, rows, longest):
    print(f"[short] N={N} rows={rows} longest={longest}", flush=True)
    rng = np.random.default_rng(rows + longest)
    deg = rng.integers(0, 3 if N == 300 else longest + 1, rows)
    deg[::97] = longest
    rowptr = np.zeros(rows + 1, np.int32)
    np.cumsum(deg, out=rowptr[1:])
    colind = rng.integers(0, 200, rowptr[-1]).astype(np.int32)
    vals = rng.standard_normal(rowptr[-1]).astype(np.float32)
    B = _B(200, N, seed=N)
    seq = oracle.spmm_seq_f32(rowptr, colind, vals, B)
    rp, ci, vl, Bd = (torch.from_numpy(x).cuda() for x in (rowptr, colind, vals, B))
    np.testing.assert_array_equal(ra_spmm.spmm_csr_direct(rp, ci, vl, Bd).cpu().numpy(), seq)
    plan = ra_spmm.make_zero_overhead_plan(rp, rows, 200)
    np.testing.assert_array_equal(ra_spmm.run_zero_overhead_plan(plan, rp, ci, vl, Bd).cpu().numpy(), seq)


def test_infinities_stay_in_their_rows(oracle):
    """Rounds past the end of a row gather nothing: an infinity or NaN in B reaches only the rows that refer to it."""
    g = S.random_csr(300, 200, 6.0, seed=3, empty_frac=0.1)
    B = _B(g.K, 40, seed=1)
    B[0] = np.inf
    B[g.K - 1] = np.nan
    rp, ci, vl = g.torch("cuda")
    with np.errstate(invalid="ignore"):
        seq = oracle.spmm_seq_f32(g.rowptr, g.colind, g.vals, B)
    Bd = torch.from_numpy(B).cuda()
    np.testing.assert_array_equal(ra_spmm.spmm_csr_direct(rp, ci, vl, Bd).cpu().numpy(), seq)
    plan = ra_spmm.make_zero_overhead_plan(rp, g.M, g.K)
    np.testing.assert_array_equal(ra_spmm.run_zero_overhead_plan(plan, rp, ci, vl, Bd).cpu().numpy(), seq)
