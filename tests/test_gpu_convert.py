"""fp32 -> fp16 / bf16 conversion of B: every run remainder, unaligned inputs and
rows that end in the middle of a 16-byte load, bit for bit as torch rounds; and
the merge of split windows over more slots than one round loads."""
import ctypes

import numpy as np
import pytest
import torch

from conftest import assert_close_scaled

pytestmark = pytest.mark.gpu

import ra_spmm  # noqa: E402
from ra_spmm import capi  # noqa: E402
from ra_spmm import synthetic as S  # noqa: E402


@pytest.mark.parametrize("cols", [1, 4, 7, 8, 9, 15, 16, 17, 47, 100, 128, 250])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_convert_every_remainder(cols, shift):
    lib = capi.load()
    rows, ldo = 333, (cols + 7) // 8 * 8
    storage = torch.full((rows * cols + shift,), float("nan"), device="cuda")
    x = storage[shift:].view(rows, cols)
    x.copy_(torch.randn(rows, cols, device="cuda") * torch.logspace(-7, 5, rows, device="cuda")[:, None])
    for dtype, torch_dtype in ((1, torch.float16), (2, torch.bfloat16)):
        out = torch.full((rows, ldo), 7.0, device="cuda", dtype=torch_dtype)
        capi.check(lib.ra_convert_f32(capi.ptr(x), capi.ptr(out), rows, cols, ldo, dtype,
                                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        assert torch.equal(out[:, :cols], x.to(torch_dtype)), (cols, shift, torch_dtype)
        assert not out[:, cols:].float().any()


# One window of 8 rows and 64 blocks (512 vectors) per segment: 1 to 20 slots a window.
@pytest.mark.parametrize("slots", [2, 8, 9, 10, 17, 20])
@pytest.mark.parametrize("N", [16, 33, 128])
def test_merge_of_many_slots(oracle, slots, N):
    K = 512 * slots
    g = S.random_csr(16, K, K - 7, seed=slots, max_deg=K - 1)
    B = np.random.default_rng(N).standard_normal((K, N)).astype(np.float32)
    rp, ci, vl = g.torch("cuda")
    plan = ra_spmm.make_segment_hybrid_plan(rp, ci, vl, g.M, g.K, N, rows_per_window=8)
    assert plan.num_split_windows == 2 and plan.num_split_segs == 2 * slots
    C = ra_spmm.run_tile_plan_route(plan, torch.from_numpy(B).cuda(), "fp16").cpu().numpy()
    qv, qb = oracle.quantize_f16(g.vals), oracle.quantize_f16(B)
    assert_close_scaled(C, oracle.spmm_tile_f64(g.rowptr, g.colind, g.vals, B, "f16"),
                        oracle.spmm_f64(g.rowptr, g.colind, np.abs(qv), np.abs(qb)), 1e-5, "merge")
