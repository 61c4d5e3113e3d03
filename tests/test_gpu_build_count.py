"""All-layer builds whose device count is below the host's bound: the packing
follows the count.  Every packing (1 to 4 pages of 16 tokens a wave, 1 and 2 of
32, odd remainders, waves that take a second turn) writes the bytes that a page
built alone gets, and no record past the count is touched."""
import pytest

pytestmark = pytest.mark.gpu

SLABS = ("pp_v4", "pp_vs", "pp_c8", "pp_cs", "pp_mu8", "pp_mus", "pp_tag")


def _bits(t):
    import torch
    return t.contiguous().view(torch.int16) if t.dtype == torch.bfloat16 else t


@pytest.mark.parametrize("d,page,n_kv,L,bound,count", [
    (128, 16, 2, 1, 1200, 1100), (64, 16, 3, 1, 1100, 1001), (512, 16, 1, 2, 1700, 1301),       # 3 a wave
    (256, 16, 2, 1, 1200, 1103), (256, 16, 2, 1, 1700, 1601), (512, 16, 1, 1, 4000, 3333),      # 3; 4 a wave
    (128, 16, 5, 1, 777, 777), (64, 16, 2, 2, 900, 801),
    (128, 16, 4, 40, 450, 431),                                                                 # 68960: a second turn
    (128, 32, 2, 3, 500, 401), (64, 32, 2, 1, 513, 513), (256, 32, 1 + 1, 1, 700, 300),         # 1 and 2 a wave
    (128, 16, 2, 2, 4000, 3), (512, 16, 1, 4, 4000, 1), (64, 64, 2, 2, 300, 5), (128, 16, 8, 2, 300, 0)])
def test_count_below_the_bound(d, page, n_kv, L, bound, count):
    import torch
    from locks import _lib
    from locks.selection import MlaState, Rki4State, rki4_build_blocks
    print(f"[case] d {d} page {page} n_kv {n_kv} layers {L} bound {bound} count {count}", flush=True)
    NB = bound + 3
    g = torch.Generator(device="cuda").manual_seed(d + page + bound)
    row = d + (64 if d == 512 else 0)
    K = [torch.randn(NB, page, n_kv, row, generator=g, device="cuda").to(torch.bfloat16)[..., :d] for _ in range(L)]
    kw = dict(num_layers=L, num_blocks=NB, max_reqs=1, max_pages=4)

    def state():
        if d == 512:
            return MlaState("cuda", n_heads=16, **kw)
        return Rki4State("cuda", n_kv=n_kv, G=1, head_dim=d, page=page, **kw)

    st, alone = state(), state()
    ids = torch.randperm(NB, generator=g, device="cuda")[:bound].to(torch.int32)
    kp = torch.tensor([k.data_ptr() for k in K], dtype=torch.int64).cuda()
    n = torch.tensor([count], dtype=torch.int32, device="cuda")
    lib = _lib.load()
    _lib.check(lib.locks_build_rki4_layers(
        kp.data_ptr(), L, K[0].stride(0), K[0].stride(1), K[0].stride(2), NB, ids.data_ptr(), n.data_ptr(), bound, n_kv,
        d, page, NB, *[_lib.ptr(getattr(st, s)) for s in SLABS[:6]], _lib.rows_arg(st), st.pp_tag.data_ptr(),
        _lib.stream_ptr()), "build_rki4_layers")
    step = max(1, 1000 // n_kv)                       # few enough items for one page per wave
    for layer in range(L):
        for lo in range(0, count, step):
            rki4_build_blocks(alone, layer, K[layer], ids[lo:min(lo + step, count)])
    torch.cuda.synchronize()
    for name in SLABS:
        assert torch.equal(_bits(getattr(st, name)), _bits(getattr(alone, name))), name
    rest = torch.ones(NB, dtype=torch.bool, device="cuda")
    rest[ids[:count].long()] = False
    assert not st.pp_v4[:, rest].any() and st.pp_tag[:, rest].isnan().all()
