"""Device memory kept between plans: reused, bounded, given back, and never
handed on while a stream may still be using it."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

import ra_spmm  # noqa: E402
from ra_spmm import synthetic as S  # noqa: E402


def _free():
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0] + torch.cuda.memory_reserved()


def test_reuse_and_release():
    """Four plans after the first take no memory of their own (each converts B into a buffer of 256 MB)."""
    g = S.sbm(256, 100, 24.0, 0.9, seed=2)
    rp, ci, vl = g.torch("cuda")
    B = torch.randn(g.K, 5008, device="cuda")
    one = g.K * 5008 * 2

    def once():
        plan = ra_spmm.make_tc_direct_plan(rp, ci, vl, g.M, g.K, 5008)
        return ra_spmm.run_tc_direct_plan(plan, B)

    ref = once()
    _free()
    assert torch.equal(once(), ref)  # the one-time allocations of the runtime are done after this
    kept = _free()
    for _ in range(4):
        assert torch.equal(once(), ref)
    assert abs(_free() - kept) < one // 2
    ra_spmm.release_memory()
    assert _free() - kept >= one  # the blocks of the dead plans went back
    assert torch.equal(once(), ref)


def test_bound_and_large_blocks():
    """Dropped plans keep at most 4 GiB, and a block above that takes what was asked for and goes back at once."""
    ra_spmm.release_memory()
    g = S.random_csr(4096, 600_000, 4.0, seed=3)
    rp, ci, vl = g.torch("cuda")

    def run(n):
        plan = ra_spmm.make_tc_direct_plan(rp, ci, vl, g.M, g.K, n)
        ra_spmm.run_tc_direct_plan(plan, torch.zeros(g.K, n, device="cuda"))
        torch.cuda.synchronize()
        return plan

    run(64)
    ra_spmm.release_memory()
    start = _free()
    plans = [run(1024) for _ in range(5)]  # 1.2 GB each
    assert start - _free() > 5 * g.K * 1024 * 2
    plans.clear()
    assert start - _free() < (4 << 30) + (64 << 20)
    ra_spmm.release_memory()
    assert start - _free() < (64 << 20)
    plan = run(3712)  # 4.45 GB: eighths of its power of two would be 4.83
    need = g.K * 3712 * 2
    assert abs(start - _free() - need) < (256 << 20)  # the runtime's own memory comes and goes by some MiB
    del plan
    assert start - _free() < (256 << 20)


def test_plans_of_other_streams_and_threads():
    """A plan dropped right after its run was queued on a side stream: the next plans, on other streams and threads,
    must not get its memory before the run is done."""
    graphs = [S.random_csr(4000, 4000, 20.0 + i, seed=i, skew=1.2) for i in range(3)]
    inputs = []
    for i, g in enumerate(graphs):
        rp, ci, vl = g.torch("cuda")
        B = torch.randn(g.K, 96, device="cuda", generator=torch.Generator("cuda").manual_seed(i))
        plan = ra_spmm.make_segment_hybrid_plan(rp, ci, vl, g.M, g.K, 96)
        inputs.append((g, rp, ci, vl, B, ra_spmm.run_segment_hybrid_plan(plan, ci, vl, B)))
    torch.cuda.synchronize()
    wrong, errors, done = [], [], [0, 0, 0]

    def work(i):
        g, rp, ci, vl, B, ref = inputs[i]
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(20):
                    plan = ra_spmm.make_segment_hybrid_plan(rp, ci, vl, g.M, g.K, 96)
                    out = ra_spmm.run_segment_hybrid_plan(plan, ci, vl, B)
                    del plan
                    stream.synchronize()
                    if not torch.equal(out, ref):
                        wrong.append(i)
                    done[i] += 1
        except Exception as e:  # noqa: BLE001
            errors.append((i, e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not any(t.is_alive() for t in threads)
    assert not errors and not wrong and done == [20, 20, 20]
