"""The latent decode on both sides of its pages-per-split rule against 64-bit
attention over the attended pages: full and short rows, an empty row, more
pages than the budget (longer splits), fewer splits allocated than the rule asks."""
import math

import pytest


def test_rule():
    from locks.attention.mla_decode import _launch_shape, _pps_min
    assert [_pps_min(n, 128) for n in (1, 4, 8, 16, 17, 32, 128)] == [4, 4, 4, 4, 8, 8, 8]
    assert [_pps_min(n, 200) for n in (1, 10, 11, 64)] == [4, 4, 8, 8]

    class St:
        budget_abs, sink_pages, window_pages, split = 117, 1, 10, 32
    assert _launch_shape(St, 8) == (4, 32) and _launch_shape(St, 32) == (8, 16)
    St.split = 5                                     # a state's own split count is never exceeded
    assert _launch_shape(St, 8) == (4, 5) and _launch_shape(St, 32) == (8, 5)


@pytest.mark.gpu
@pytest.mark.parametrize("R,budget,split", [
    (1, 128, None), (8, 128, None), (16, 128, None), (17, 128, None), (40, 100, None), (11, 200, None), (33, 61, None),
    (20, 128, 5), (3, 40, 2)])
def test_decode_equals_64_bit(R, budget, split):
    import torch
    from locks.attention.mla_decode import mla_decode
    from locks.selection import MlaState
    print(f"[case] R {R} budget {budget} split {split}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(R * 1000 + budget)
    MP, NB = budget + 30, 600
    cache = torch.randn(NB, 16, 576, generator=g, device="cuda").to(torch.bfloat16)
    q = torch.randn(R, 16, 576, generator=g, device="cuda").to(torch.bfloat16)
    bt = torch.randint(0, NB, (R, MP), generator=g, device="cuda", dtype=torch.int32)
    st = MlaState("cuda", num_layers=1, num_blocks=NB, n_heads=16, max_reqs=R, max_pages=MP, budget_pages=budget,
                  split=split)
    cnt = torch.full((R,), budget, dtype=torch.int32)
    cnt[R // 2] = max(budget // 3, 1)
    if R > 2:
        cnt[0], cnt[1], cnt[2] = 1, MP, 0            # one page; more than the budget; none
    lens = torch.full((R,), MP * 16 - 5, dtype=torch.int32)
    st.page_cnt[:, 0] = cnt.cuda()
    keep = [torch.randperm(MP, generator=g, device="cuda")[:int(c)].sort().values for c in cnt]
    for r, p in enumerate(keep):
        st.page_table[r, 0, :len(p)] = p.to(torch.int32)
    scale = 1 / math.sqrt(192)
    out = torch.full((R, 16, 512), 7.0, device="cuda")
    lse = torch.full((R, 16), 7.0, device="cuda")
    mla_decode(st, q, cache, bt, lens.cuda(), R, scale, out, lse)
    torch.cuda.synchronize()
    for r, p in enumerate(keep):
        if not len(p):
            assert not out[r].any() and (lse[r] == -math.inf).all()
            continue
        rows = cache[bt[r, p].long()].double().flatten(0, 1)
        pos = (p[:, None] * 16 + torch.arange(16, device="cuda")).flatten()
        x = (q[r].double() @ rows.t().contiguous() * scale).masked_fill(pos >= int(lens[r]), -math.inf)
        ref = torch.softmax(x, -1) @ rows[:, :512].contiguous()
        # probabilities are rounded to fp16 (2^-11 relative each), the sum of |P V| is at most max |V|
        assert (out[r].double() - ref).abs().max() <= 2.0 ** -11 * float(rows.abs().max())
        assert (lse[r].double() - torch.logsumexp(x, -1)).abs().max() <= 1e-5
