"""Device tile-format build (hipCUB sorts and scans) against the host builder.

Both builders must emit the same plan bit for bit: every array of the format
(win_rows, block_offsets, atox, fp16/bf16 value bits, segment and merge
tables) and every count in the plan info.  The host builder is itself pinned
against the oracle's tile_format (tests/test_oracle_structures.py), so
equality here carries that pin over to the device build.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import ra_spmm  # noqa: E402
from ra_spmm import synthetic as S  # noqa: E402

MAKE = {0: ra_spmm.make_tc_direct_plan, 1: ra_spmm.make_community_tc_plan,
        2: ra_spmm.make_segment_hybrid_plan}
ARRAYS = ("win_rows", "block_offsets", "atox", "vals", "seg_window", "seg_bbegin", "seg_bend",
          "seg_slot", "split_windows", "split_offsets")
INFO = ("active", "num_windows", "num_blocks", "num_segments", "num_split_windows",
        "num_split_segs", "nnz", "num_vectors", "plan_bytes", "avg_tc_tile_density",
        "value_scale_log2", "max_window_blocks")


def _dups(seed=21):
    """CSR with repeated (row, column) entries, unsorted columns and empty windows."""
    rng = np.random.default_rng(seed)
    M, K = 300, 120
    deg = rng.integers(0, 30, M)
    deg[40:72] = 0                                      # four empty windows
    rp = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    ci = rng.integers(0, K // 3, rp[-1]).astype(np.int32)   # many duplicates
    vl = rng.standard_normal(rp[-1]).astype(np.float32)
    return S.Graph(rp, ci, vl, M, K, "dups")


GRAPHS = {
    "skewed": lambda: S.random_csr(1003, 900, 9.0, seed=3, skew=1.1, empty_frac=0.05),
    "community": lambda: S.sbm(64, 50, 12.0, 0.9, seed=6),
    "hub_windows": lambda: S.random_csr(40, 40000, 2500.0, seed=8),
    "dense_rows": lambda: S.random_csr(200, 3000, 150.0, seed=4),
    "duplicates": _dups,
    "one_row": lambda: S.random_csr(1, 50, 20.0, seed=2),
}


def _compare(g, kind, value_dtype, N=64):
    rp, ci, vl = (torch.from_numpy(np.ascontiguousarray(a)) for a in (g.rowptr, g.colind, g.vals))
    host = MAKE[kind](rp, ci, vl, g.M, g.K, N, value_dtype, build="host")
    dev = MAKE[kind](rp.cuda(), ci.cuda(), vl.cuda(), g.M, g.K, N, value_dtype, build="gpu", rows_per_window=8)
    for f in INFO:
        assert getattr(host, f) == getattr(dev, f), f
    for a in ARRAYS:
        h = ra_spmm.export_tile_plan(host, a).numpy()
        d = ra_spmm.export_tile_plan(dev, a).numpy()
        np.testing.assert_array_equal(h, d, err_msg=a)
    return host, dev


@pytest.mark.parametrize("gname", list(GRAPHS))
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("value_dtype", ["fp16", "bf16"])
def test_device_build_matches_host(gname, kind, value_dtype):
    print(f"[tile-build] {gname} kind={kind} {value_dtype}", flush=True)
    host, dev = _compare(GRAPHS[gname](), kind, value_dtype)
    assert host.active


def test_device_build_runs_identically():
    g = GRAPHS["skewed"]()
    B = torch.randn(g.K, 96, device="cuda")
    for kind in (0, 1, 2):
        host, dev = _compare(g, kind, "fp16", 96)
        for route in ("fp16", "fp32"):
            assert torch.equal(ra_spmm.run_tile_plan_route(host, B, route),
                               ra_spmm.run_tile_plan_route(dev, B, route))


def test_device_build_inactive_and_invalid():
    g = GRAPHS["skewed"]()
    rp, ci, vl = g.torch("cuda")
    p = ra_spmm.make_tc_direct_plan(rp, ci, vl, g.M, g.K, 8, build="gpu", rows_per_window=8)
    assert p.valid and not p.active
    bad = ci.clone()
    bad[5] = g.K
    with pytest.raises(RuntimeError, match="out of range"):
        ra_spmm.make_tc_direct_plan(rp, bad, vl, g.M, g.K, 64, build="gpu")


def test_c3_device_build_matches_host():
    g = S.CONFIGS["C3"]()
    for kind in (0, 1):
        _compare(g, kind, "fp16", 256)


@pytest.mark.parametrize("seed", range(16))
def test_device_build_matches_host_random(seed):
    """Seeded shapes, densities, skew, empty rows and duplicates: the device
    build equals the host build array for array."""
    rng = np.random.default_rng(500 + seed)
    M, K = int(rng.integers(1, 2500)), int(rng.integers(1, 4000))
    d = float(rng.choice([1.0, 6.0, 30.0, 120.0]))
    g = S.random_csr(M, K, min(d, K), seed=int(rng.integers(1 << 30)), skew=float(rng.choice([0.0, 1.1])),
                     empty_frac=float(rng.choice([0.0, 0.2])), max_deg=K)
    if rng.random() < 0.4 and g.nnz > 1:  # repeated (row, column) entries
        ci = g.colind.copy()
        ci[1::3] = ci[0:-1:3][: len(ci[1::3])]
        g = S.Graph(g.rowptr, ci, g.vals, M, K, "dups")
    kind = int(rng.integers(0, 3))
    value_dtype = "bf16" if rng.random() < 0.3 else "fp16"
    print(f"[tile-build] random seed={seed} M={M} K={K} nnz={g.nnz} kind={kind} {value_dtype}", flush=True)
    _compare(g, kind, value_dtype, N=int(rng.choice([16, 64, 200])))


def _window_graph(per_window, K, seed, shuffle):
    """Windows of 32 rows with exactly per_window nonzeros, spread unevenly, duplicates and (shuffle) unsorted columns."""
    rng = np.random.default_rng(seed)
    deg = np.concatenate([rng.multinomial(n, rng.dirichlet(np.full(32, 0.3))) for n in per_window])[:-3]
    rp = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    ci = rng.integers(0, K, rp[-1]).astype(np.int32)
    if not shuffle:
        for r in range(deg.size):
            ci[rp[r]:rp[r + 1]].sort()
    return S.Graph(rp, ci, rng.standard_normal(rp[-1]).astype(np.float32), deg.size, K, "windows")


# Either side of each size that the window sort has a kernel for, and one past the largest (the global sort).
@pytest.mark.parametrize("longest", [1, 255, 1024, 1025, 2048, 2049, 4096, 4097])
@pytest.mark.parametrize("K", [64, 1 << 16])
@pytest.mark.parametrize("kind", [0, 2])
def test_window_sort_matches_host(longest, K, kind):
    g = _window_graph([longest, longest // 2, 0, longest, longest // 3 + 4], K, seed=longest, shuffle=longest % 2 == 1)
    _compare(g, kind, "fp16")


# The counts behind the choice of the window height come from the same sort.
@pytest.mark.parametrize("longest", [900, 3000, 6000])
def test_window_height_choice(longest):
    dense = _window_graph([longest] * 8, 96, seed=3, shuffle=False)    # rows share their columns: tall windows
    sparse = _window_graph([longest] * 8, 1 << 18, seed=4, shuffle=False)
    for g, tall in ((dense, True), (sparse, False)):
        rp, ci, vl = g.torch("cuda")
        plans = [mk(rp, ci, vl, g.M, g.K, 64) for mk in (ra_spmm.make_tc_direct_plan, ra_spmm.make_segment_hybrid_plan)]
        assert all((p.rows_per_window > 8) == tall for p in plans), [p.rows_per_window for p in plans]
        B = torch.randn(g.K, 64, device="cuda", generator=torch.Generator("cuda").manual_seed(longest))
        ref = ra_spmm.spmm_csr_baseline(rp, ci, vl, B)
        # fp16 rounds a value and a feature to 2^-11 of themselves each; a feature below 2^-14 to a multiple of 2^-24,
        # so to 2^-25 absolute.
        bound = 2.0 ** -10 * ra_spmm.spmm_csr_baseline(rp, ci, vl.abs(), B.abs()) + \
            2.0 ** -25 * ra_spmm.spmm_csr_baseline(rp, ci, vl.abs(), torch.ones_like(B)) + 1e-30
        for p in plans:
            assert bool(((ra_spmm.run_tile_plan_route(p, B, "fp16") - ref).abs() <= bound).all())


def test_more_windows_than_a_grid():
    """134 million rows: more 8-row windows than one workgroup each would fit a grid."""
    if torch.cuda.get_device_properties(0).total_memory < 64 << 30:
        pytest.skip("needs a GPU with 64 GiB")
    M, K, N = (1 << 27) + 11, 500, 16
    print(f"[windows] M={M}", flush=True)
    rows = torch.cat([torch.arange(300), torch.arange(1 << 26, (1 << 26) + 300), torch.arange(M - 300, M)])
    deg = torch.zeros(M, dtype=torch.int32, device="cuda")
    deg[rows.cuda()] = 7
    rowptr = torch.zeros(M + 1, dtype=torch.int32, device="cuda")
    rowptr[1:] = torch.cumsum(deg, 0)
    gen = torch.Generator("cuda").manual_seed(1)
    ci = torch.sort(torch.rand(rows.numel(), K, device="cuda", generator=gen).topk(7, dim=1).indices, dim=1).values
    ci = ci.to(torch.int32).flatten()
    vl = torch.randint(1, 65, (ci.numel(),), device="cuda", generator=gen) / 64.0
    B = torch.randn(K, N, device="cuda", generator=gen).half().float()
    plan = ra_spmm.make_tc_direct_plan(rowptr, ci, vl, M, K, N)
    assert plan.nnz == ci.numel() and plan.num_windows == (M + 7) // 8
    C = ra_spmm.run_tc_direct_plan(plan, B)
    want = (vl.double()[:, None] * B.double()[ci.long()]).view(-1, 7, N).sum(1)
    scale = (vl.double()[:, None] * B.double().abs()[ci.long()]).view(-1, 7, N).sum(1)
    assert ((C[rows.cuda()].double() - want).abs() <= 1e-5 * scale).all()
    assert int((C != 0).any(1).sum()) <= rows.numel()
