"""32-bit gather offsets up to their limit, and the 64-bit addresses past it.

CSR kernels gather through a buffer descriptor while K * N * 4 <= 0xFFFF0000 and N <= 16,000; the tile
kernels while row -1 of the 16-bit B, whose offset wraps, still lies past its end.  Few rows reach all of
B: the first, the last, and those around 2 GiB, where a signed offset would turn negative.
"""
import numpy as np
import pytest
import torch

from conftest import assert_close_scaled

pytestmark = pytest.mark.gpu

import ra_spmm  # noqa: E402


def _matrix(K, row_bytes, M, per_row, seed):
    """CSR of M rows with ascending distinct columns; (rowptr, colind, vals, used columns, colind in the used ones)."""
    rng = np.random.default_rng(seed)
    middle = (1 << 31) // row_bytes
    special = np.unique(np.clip([0, 1, middle - 1, middle, middle + 1, K - 2, K - 1], 0, K - 1))
    rows = [np.unique(np.concatenate([special, rng.integers(0, K, per_row - special.size)])) for _ in range(M)]
    rowptr = np.concatenate([[0], np.cumsum([r.size for r in rows])]).astype(np.int32)
    colind = np.concatenate(rows).astype(np.int32)
    used, sub = np.unique(colind, return_inverse=True)
    # k / 64: exact in fp16 and bf16
    vals = (rng.integers(1, 65, colind.size) / 64.0).astype(np.float32)
    return rowptr, colind, vals, used, sub.astype(np.int32)


def _need_memory(gib):
    if torch.cuda.get_device_properties(0).total_memory < gib << 30:
        pytest.skip(f"needs a GPU with {gib} GiB")


# Whole rows, one column a lane (33 on CSR_DIRECT, 31 on both), four a lane on ragged rows.
@pytest.mark.parametrize("N", [64, 31, 33, 130])
@pytest.mark.parametrize("past", [0, 1])
def test_csr_gathers_around_4_gib(oracle, N, past):
    _need_memory(32)
    K = 0xFFFF0000 // (4 * N) + past
    print(f"[offsets] csr N={N} K={K}", flush=True)
    rowptr, colind, vals, used, sub = _matrix(K, 4 * N, 70, 40, seed=N)
    B = torch.randn(K, N, device="cuda", generator=torch.Generator("cuda").manual_seed(N))
    seq = oracle.spmm_seq_f32(rowptr, sub, vals, B[torch.from_numpy(used).cuda()].cpu().numpy())
    rp, ci, vl = (torch.from_numpy(x).cuda() for x in (rowptr, colind, vals))
    np.testing.assert_array_equal(ra_spmm.spmm_csr_direct(rp, ci, vl, B).cpu().numpy(), seq)
    plan = ra_spmm.make_zero_overhead_plan(rp, 70, K)
    np.testing.assert_array_equal(ra_spmm.run_zero_overhead_plan(plan, rp, ci, vl, B).cpu().numpy(), seq)


@pytest.mark.parametrize("N", [16_000, 16_001, 16_004])
def test_csr_gathers_of_the_widest_rows(oracle, N):
    print(f"[offsets] csr N={N}", flush=True)
    rowptr, colind, vals, used, sub = _matrix(90, 4 * N, 30, 20, seed=N)
    B = np.random.default_rng(N).standard_normal((90, N)).astype(np.float32)
    seq = oracle.spmm_seq_f32(rowptr, colind, vals, B)
    rp, ci, vl, Bd = (torch.from_numpy(x).cuda() for x in (rowptr, colind, vals, B))
    np.testing.assert_array_equal(ra_spmm.spmm_csr_direct(rp, ci, vl, Bd).cpu().numpy(), seq)
    plan = ra_spmm.make_zero_overhead_plan(rp, 30, 90)
    np.testing.assert_array_equal(ra_spmm.run_zero_overhead_plan(plan, rp, ci, vl, Bd).cpu().numpy(), seq)


# Rows whose last block is partly padding; 8-row windows of 100 columns a row are shared and gather through the
# descriptor, as the tall ones do; with 9 a row (under 6 steps, even windows, a large B) they go by pointers.
@pytest.mark.parametrize("N", [64, 128])
@pytest.mark.parametrize("past", [0, 1])
@pytest.mark.parametrize("rows,per_row", [(8, 100), (8, 9), (16, 33), (32, 33)])
def test_tile_gathers_around_4_gib(oracle, N, past, rows, per_row):
    _need_memory(16)
    K = 0xFFFFFFFF // (2 * N) - 1 + past
    print(f"[offsets] tile N={N} K={K} rows={rows}", flush=True)
    rowptr, colind, vals, used, sub = _matrix(K, 2 * N, 67, per_row, seed=N + rows)
    B = torch.randn(K, N, device="cuda", dtype=torch.float16, generator=torch.Generator("cuda").manual_seed(N))
    Bu = B[torch.from_numpy(used).cuda()].float().cpu().numpy()
    rp, ci, vl = (torch.from_numpy(x).cuda() for x in (rowptr, colind, vals))
    plan = ra_spmm.make_tc_direct_plan(rp, ci, vl, 67, K, N, rows_per_window=rows)
    C = ra_spmm.run_tile_plan_route(plan, B, "fp16").cpu().numpy()
    assert_close_scaled(C, oracle.spmm_f64(rowptr, sub, vals, Bu), oracle.spmm_f64(rowptr, sub, vals, np.abs(Bu)), 1e-5,
                        f"tile {N} {rows}")
