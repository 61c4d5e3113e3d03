"""Selection over rows whose page count is not a multiple of 4 (vector accesses
of 4-byte alignment, a last vector that runs past the row): the page tables
equal the oracle's, and equal those of the same scores in a row padded to a
multiple of 4 bit for bit; nothing is written past a row."""
import numpy as np
import pytest

from oracle import locks_oracle as O

pytestmark = pytest.mark.gpu


# row lengths at the edges of the routes: 1-3, 4 k + 1 .. 3, one thread's
# vector, 4096 / 8192 (pages per thread), 64K (head, page) entries, chunks of
# 1024 and 2048 pages, the large-budget route
@pytest.mark.parametrize("MP,G,b,combine", [
    (1, 4, 5, "nrm"), (2, 16, 1, "max"), (3, 1, 1, "max"), (5, 4, 2, "nrm"), (6, 4, 3, "max"), (7, 8, 2, "nrm"),
    (1023, 4, 126, "nrm"), (2049, 8, 77, "nrm"), (4097, 4, 126, "nrm"), (4094, 1, 117, "max"), (5626, 4, 126, "nrm"),
    (8191, 8, 126, "max"), (9381, 16, 126, "nrm"), (18751, 4, 126, "nrm"), (18749, 4, 1875, "nrm"),
    (8193, 1, 64, "max")])
def test_odd_rows(MP, G, b, combine):
    import torch
    from locks.selection import Rki4State, derive_page_params, rki4_select_only
    print(f"[case] MP {MP} G {G} b {b} {combine}", flush=True)
    rng = np.random.default_rng(MP * 17 + G)
    n_kv, lens = 2, [MP * 16, max(MP * 16 - 33, 1), 1 + (MP * 16) // 2]
    R = len(lens)
    npg, nsh, bfix = O.derive_page_params(lens, 16, 1, 1, b)
    sh = np.round(rng.standard_normal((R, n_kv, G, MP)) * 64).astype(np.float32) / 64    # ties
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")

    def run(width):
        st = Rki4State("cuda", num_layers=1, num_blocks=4, n_kv=n_kv, G=G, head_dim=128, page=16, max_reqs=R,
                       max_pages=width, budget_pages=b, combine=combine)
        st.score_h.zero_()
        st.score_h[..., :MP] = torch.from_numpy(sh).cuda()
        pm = np.full((R, n_kv, 16, st.score_chunks), -np.inf, np.float32)
        for r in range(R):
            for z in range(st.score_chunks):
                lo, hi = z * st.score_chunk, min((z + 1) * st.score_chunk, int(nsh[r]))
                if hi > lo:
                    pm[r, :, :G, z] = sh[r, :, :, lo:hi].max(axis=-1)
        st.page_max.copy_(torch.from_numpy(pm))
        derive_page_params(st, sl, R)
        for _ in range(2):                                # the second call reuses the workspace
            st.score.fill_(-7.0)
            st.page_table.fill_(-9)
            rki4_select_only(st, R)
        torch.cuda.synchronize()
        return st.page_table.cpu().numpy(), st.page_cnt.cpu().numpy(), st.score.cpu().numpy()

    tab, cnt, score = run(MP)
    tab4, cnt4, score4 = run(-(-MP // 4) * 4)
    assert np.array_equal(tab, tab4[..., :MP]) and np.array_equal(cnt, cnt4)
    assert np.array_equal(score.view(np.uint32), score4[..., :MP].copy().view(np.uint32))
    for r in range(R):
        assert (score[r, :, max(int(nsh[r]), 0):] == -7.0).all()       # nothing past the scored pages
    # exact top-b of the combined scores that the GPU wrote
    comb = np.where(score == -7.0, 0, score).astype(np.float32)
    ref, rcnt = O.topb_select(comb, npg, nsh, bfix, 1, MP)
    assert np.array_equal(cnt, rcnt) and np.array_equal(tab, ref)
