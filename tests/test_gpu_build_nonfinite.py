"""Pages with infinite, NaN or overflowing keys: a finite value over an infinite
scale is a zero code (IEEE division), and such a page leaves the records of the
pages that share its wave byte for byte alone."""
import pytest

pytestmark = pytest.mark.gpu

SLABS = ("pp_v4", "pp_vs", "pp_c8", "pp_cs", "pp_mu8", "pp_mus", "pp_tag")
INF, NAN = float("inf"), float("nan")


def _bits(t):
    import torch
    return t.contiguous().view(torch.int16) if t.dtype == torch.bfloat16 else t


# item counts that put 4, 2 and 1 pages into a wave
@pytest.mark.parametrize("d,page,n_blocks", [
    (128, 16, 1601), (64, 16, 1601), (256, 16, 551), (512, 16, 3201), (128, 32, 551), (128, 64, 41)])
def test_nonfinite_pages(d, page, n_blocks):
    import torch
    from locks.selection import MlaState, Rki4State, rki4_build_blocks
    print(f"[case] d {d} page {page} blocks {n_blocks}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(d + page)
    n_kv, row = (1, d + 64) if d == 512 else (2, d)
    h = n_kv - 1                                       # the special pages' head
    K = torch.randn(n_blocks, page, n_kv, row, generator=g, device="cuda").to(torch.bfloat16)[..., :d]
    bad = K.clone()
    inf_at = {5: INF, 18: -INF, n_blocks - 1: INF}     # a page's infinite key, in channel 3
    nan_at, huge_at = (10, 23), (14, 29, 30)
    for b, x in inf_at.items():
        bad[b, page // 2, h, 3] = x
    for b in nan_at:
        bad[b, 1, h, 3] = NAN
    for b in huge_at:                                  # finite keys, the gram overflows
        bad[b, :, h] *= 1e20
    ids = torch.arange(n_blocks, dtype=torch.int32, device="cuda")

    def build(keys):
        kw = dict(num_layers=1, num_blocks=n_blocks, max_reqs=1, max_pages=4)
        st = MlaState("cuda", n_heads=16, **kw) if d == 512 else \
            Rki4State("cuda", n_kv=n_kv, G=1, head_dim=d, page=page, **kw)
        rki4_build_blocks(st, 0, keys, ids)
        torch.cuda.synchronize()
        return st

    clean, st = build(K), build(bad)
    others = torch.ones(n_blocks, n_kv, dtype=torch.bool, device="cuda")
    for b in (*inf_at, *nan_at, *huge_at):
        others[b, h] = False
    for name in SLABS:
        assert torch.equal(_bits(getattr(st, name)[0])[others], _bits(getattr(clean, name)[0])[others]), name
    for b in inf_at:                                   # the centroid's scale is infinite
        mu8 = st.pp_mu8[0, b, h].cpu().tolist()
        assert float(st.pp_mus[0, b, h]) == INF
        assert mu8[3] == -127 and not any(mu8[:3] + mu8[4:]), mu8
    for b in nan_at:                                   # a NaN is no maximum; the other channels keep their codes
        top = clean.pp_mu8[0, b, h].abs().argmax()
        same = st.pp_mu8[0, b, h] == clean.pp_mu8[0, b, h]
        same[3] = True
        assert int(top) == 3 or bool(same.all())
    for b in huge_at:                                  # singular values infinite: an empty basis
        assert int(st.pp_v4[0, b, h].sum()) == 0
        assert (st.pp_vs[0, b, h] == torch.tensor(1e-8, dtype=torch.bfloat16)).all()
