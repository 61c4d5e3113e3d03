"""The scorer rotates a request's chunks in the grid: with every kind of chunk
count (powers of two, multiples of one, odd) and more requests than chunks,
each chunk is scored once, and a request's scores and chunk maxima do not
depend on its place in the batch."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Z,n_kv,G,R", [
    (1, 2, 4, 3), (2, 8, 4, 5), (3, 8, 4, 4), (4, 8, 1, 9), (6, 4, 7, 5), (8, 2, 16, 11), (22, 4, 7, 3), (32, 2, 4, 37),
    (43, 1, 16, 3)])
def test_place_in_the_batch(Z, n_kv, G, R):
    import torch
    from locks.selection import Rki4State, derive_page_params, rki4_score_only
    print(f"[case] Z {Z} n_kv {n_kv} G {G} requests {R}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(Z * 64 + R)
    MP, NB = 8 * Z, 500
    lens = torch.randint(1, MP * 16 + 1, (R,), generator=g, device="cuda", dtype=torch.int32)
    lens[0] = MP * 16
    bt = torch.randint(0, NB, (R, MP), generator=g, device="cuda", dtype=torch.int32)
    q = torch.randn(R, n_kv * G, 128, generator=g, device="cuda").to(torch.bfloat16)
    st = Rki4State("cuda", num_layers=1, num_blocks=NB, n_kv=n_kv, G=G, head_dim=128, page=16, max_reqs=R, max_pages=MP,
                   zsplit=Z)
    assert st.score_chunks == Z
    st.pp_rows.random_(generator=g)
    for t in (st.pp_vs, st.pp_cs, st.pp_mus):
        t.copy_(torch.rand(t.shape, generator=g, device="cuda") * 0.05 + 0.01)

    def run(order):
        st.score_h.fill_(float("nan"))
        st.page_max.fill_(float("nan"))
        sl, tab, qq = lens[order].contiguous(), bt[order].contiguous(), q[order].contiguous()
        derive_page_params(st, sl, R)
        rki4_score_only(st, 0, qq, tab, sl, R, 0.088)
        torch.cuda.synchronize()
        back = torch.argsort(order)
        return st.score_h[back], st.page_max[back]

    first = torch.arange(R, device="cuda")
    score, pmax = run(first)
    assert not pmax[:, :, :G].isnan().any()
    page = torch.arange(MP, device="cuda")
    scored = page < ((lens + 15) // 16 - 1)[:, None]                 # all but the window page
    want = scored[:, None, None, :].expand_as(score)
    assert torch.equal(~score.isnan(), want)
    chunk_max = torch.where(want, score, float("-inf")).unflatten(-1, (Z, 8)).amax(-1)
    assert torch.equal(pmax[:, :, :G], chunk_max)
    for order in (first.flip(0), torch.randperm(R, generator=g, device="cuda")):
        s2, p2 = run(order)
        assert torch.equal(s2.nan_to_num(7.0), score.nan_to_num(7.0)) and torch.equal(p2[:, :, :G], pmax[:, :, :G])
