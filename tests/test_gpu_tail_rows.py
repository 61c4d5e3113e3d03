"""The tail's block list at the edges of its one-workgroup form (256 rows): the
set of the rows' last finalized blocks, each once, in range, with the byte map
left zero -- the same set that the two-launch form lists past 256 rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rows,listed", [(1, True), (64, True), (255, False), (256, True), (257, True), (700, False)])
def test_tail_block_list(n_rows, listed):
    import torch
    from locks import _lib
    print(f"[case] tail rows {n_rows} listed {listed}", flush=True)
    rng = np.random.default_rng(n_rows)
    R, MB, NB, page = (n_rows if not listed else n_rows + 5), 6, 400, 16
    bt = rng.integers(0, NB, (R, MB)).astype(np.int32)           # shared blocks: duplicates
    bt[rng.random((R, MB)) < 0.05] = -1
    bt[rng.random((R, MB)) < 0.05] = NB + 3
    sl = rng.integers(0, page * (MB + 2), R).astype(np.int32)    # also shorter than a page, past the table
    rows = rng.integers(-1, R + 2, n_rows).astype(np.int32) if listed else np.arange(n_rows, dtype=np.int32)
    exp = set()
    for r in rows:
        if 0 <= r < R:
            blk = int(bt[r, min(max(int(sl[r]) // page - 1, 0), MB - 1)])
            if 0 <= blk < NB:
                exp.add(blk)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    dbt, dsl, drows = dev(bt), dev(sl), dev(rows)
    mark = torch.zeros(NB, dtype=torch.uint8, device="cuda")
    blocks = torch.full((NB,), -7, dtype=torch.int32, device="cuda")
    count = torch.full((1,), 99, dtype=torch.int32, device="cuda")
    lib = _lib.load()
    for _ in range(2):
        _lib.check(lib.locks_refresh_blocks(
            0, dbt.data_ptr(), MB, dsl.data_ptr(), R, drows.data_ptr() if listed else None, n_rows, 0, page, NB,
            None, 0, 0, 0, 0, 0, None, 0, mark.data_ptr(), blocks.data_ptr(), count.data_ptr(), _lib.stream_ptr()),
            "refresh_blocks")
        torch.cuda.synchronize()
        n = int(count.item())
        got = blocks[:n].cpu().tolist()
        assert n == len(exp) and set(got) == exp
        assert int(mark.sum()) == 0
