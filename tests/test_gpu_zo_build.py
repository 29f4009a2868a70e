"""ZERO_OVERHEAD_CSR binning on the GPU against the host's, list for list, around
the edges of a round (256 rows), of a tile (1,024) and of the bins."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import ra_spmm  # noqa: E402

LISTS = ("short_rows", "chunk_rows", "chunk_starts", "chunk_slot", "split_rows", "split_off")
INFO = ("num_tiny", "num_short", "num_medium", "num_long", "num_empty", "num_chunks", "num_split_rows",
        "max_long_chunks", "num_split_chunks", "plan_bytes")
EDGES = [0, 1, 4, 5, 16, 17, 64, 65, 256, 257, 512, 513, 3000]  # either side of every bin and chunk


@pytest.mark.parametrize("M", [1, 63, 64, 255, 256, 257, 1023, 1024, 1025, 5000])
@pytest.mark.parametrize("mix", ["edges", "long", "empty", "short"])
def test_lists_equal_the_host_binning(M, mix):
    rng = np.random.default_rng(M)
    deg = {"edges": rng.choice(EDGES, M), "long": rng.integers(60, 700, M), "empty": np.zeros(M, np.int64),
           "short": rng.integers(0, 20, M)}[mix]
    rowptr = torch.from_numpy(np.concatenate([[0], np.cumsum(deg)]).astype(np.int32))
    host = ra_spmm.make_zero_overhead_plan(rowptr, M, M, build="host")
    dev = ra_spmm.make_zero_overhead_plan(rowptr.cuda(), M, M)
    for f in INFO:
        assert getattr(host, f) == getattr(dev, f), f
    for name in LISTS:
        assert torch.equal(ra_spmm.export_zero_overhead_plan(host, name), ra_spmm.export_zero_overhead_plan(dev, name)), name


@pytest.mark.parametrize("at", [0, 255, 1024, 2999])
def test_decreasing_rowptr_is_refused(at):
    rowptr = np.arange(0, 3001 * 5, 5, dtype=np.int32)
    rowptr[at + 1] = rowptr[at] - 1
    with pytest.raises(RuntimeError, match="monotone"):
        ra_spmm.make_zero_overhead_plan(torch.from_numpy(rowptr).cuda(), 3000, 3000)
