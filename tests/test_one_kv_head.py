"""States with one kv head: torch gives a dimension of size 1 any stride, so the
records' row stride is taken from the blocks."""
import numpy as np
import pytest

from oracle import locks_oracle as O
from tests.cases import load_slabs, make_case, to_dev


@pytest.mark.parametrize("d,page", [(64, 16), (128, 16), (256, 64)])
@pytest.mark.parametrize("L,NB", [(1, 7), (3, 20)])
def test_row_strides(d, page, L, NB):
    from locks.selection import Rki4State
    for n_kv in (1, 2):
        st = Rki4State("cpu", num_layers=L, num_blocks=NB, n_kv=n_kv, G=4, head_dim=d, page=page, max_reqs=1,
                       max_pages=4)
        assert list(st.slab_row_bytes) == [st.row_bytes] * 6


@pytest.mark.gpu
@pytest.mark.parametrize("G", [1, 16])
def test_step_equals_oracle(G):
    import torch
    from locks.attention import ensure_stage_b_buffers, sparse_paged_decode_batched
    from locks.selection import Rki4State, derive_page_params, rki4_score_only, rki4_select_only
    print(f"[case] one kv head, G {G}", flush=True)
    case = make_case(11 + G, 1, G, [1500, 801])
    st = Rki4State("cuda", num_layers=1, num_blocks=case.NB, n_kv=1, G=G, head_dim=128, page=16, max_reqs=2,
                   max_pages=case.MP, budget_pages=20)
    ensure_stage_b_buffers(st, torch.device("cuda"), 16)
    load_slabs(st, 0, case.slabs)
    d = to_dev(case)
    out = torch.zeros(2, G, 128, dtype=torch.float32, device="cuda")
    derive_page_params(st, d["sl"], 2)
    rki4_score_only(st, 0, d["q"], d["bt"], d["sl"], 2, case.scale)
    rki4_select_only(st, 2)
    sparse_paged_decode_batched(d["q"], d["kv"], d["bt"], d["sl"], st, out, scale=case.scale)
    torch.cuda.synchronize()
    _, nsh, _ = O.derive_page_params(case.seq_lens, 16, 1, 1, 20, 0.1)
    sh = O.score_rki4_twin(case.q, case.slabs, case.bt, nsh, 1, G, case.scale, case.MP)
    for r in range(2):
        P = int(nsh[r])
        assert np.abs(st.score_h.cpu().numpy()[r, ..., :P] - sh[r, ..., :P]).max() <= 2e-5
    tab, cnt = st.page_table.cpu().numpy(), st.page_cnt.cpu().numpy()
    assert (cnt == 22).all()
    ref, _ = O.decode_attention(case.q, case.k, case.v, case.bt, case.seq_lens, tab, cnt, G, case.scale)
    assert np.abs(out.cpu().numpy() - ref).max() <= 2e-3
