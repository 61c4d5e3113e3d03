"""The builder packs up to 64 / page pages into a wave once there are more items
than SIMDs to spread them over: one and two pages a wave (full waves, partial
last waves, masked block ids among them) write the bytes that a page built alone gets, and
leave every other record untouched.  A page's build depends on that page
alone and takes the same roundings in any packing, so the bytes are equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SLABS = ("pp_v4", "pp_vs", "pp_c8", "pp_cs", "pp_mu8", "pp_mus", "pp_tag")


# items per call: below, at and just above the spread limit (1024), with odd
# remainders of two pages a wave (page 64: always one)
@pytest.mark.parametrize("d,page,n_kv,n_blocks", [
    (128, 16, 2, 1), (128, 16, 8, 128), (128, 16, 5, 205), (128, 16, 3, 343), (64, 16, 2, 515),
    (256, 16, 2, 513), (512, 16, 1, 1027), (128, 32, 2, 513), (64, 64, 2, 514), (256, 64, 3, 343)])
def test_packed_pages_equal_single_pages(d, page, n_kv, n_blocks):
    import torch
    from locks.selection import MlaState, Rki4State, rki4_build_blocks
    print(f"[case] d {d} page {page} n_kv {n_kv} blocks {n_blocks}", flush=True)
    NB = n_blocks + 7
    g = torch.Generator(device="cuda").manual_seed(d + page + n_blocks)
    row = d + (64 if d == 512 else 0)
    K = torch.randn(NB, page, n_kv, row, generator=g, device="cuda").to(torch.bfloat16)[..., :d]
    K[3 % NB] = 0                                     # no variance: scale floors
    K[5 % NB, :, :, :] = K[5 % NB, :1, :, :]          # constant page
    kw = dict(num_layers=1, num_blocks=NB, max_reqs=1, max_pages=4)

    def state():
        if d == 512:
            return MlaState("cuda", n_heads=16, **kw)
        return Rki4State("cuda", n_kv=n_kv, G=1, head_dim=d, page=page, **kw)

    ids = torch.randperm(NB, generator=g, device="cuda")[:n_blocks].to(torch.int32)
    packed, alone = state(), state()
    masked = torch.cat([ids[:1], torch.tensor([-1, NB, NB + 9], dtype=torch.int32, device="cuda"), ids[1:]])
    rki4_build_blocks(packed, 0, K, masked)
    step = max(1, 1000 // n_kv)                       # few enough items for one page per wave
    for lo in range(0, n_blocks, step):
        rki4_build_blocks(alone, 0, K, ids[lo:lo + step])
    torch.cuda.synchronize()
    for name in SLABS:
        a, b = getattr(packed, name)[0], getattr(alone, name)[0]
        if a.dtype == torch.bfloat16:
            a, b = a.contiguous().view(torch.int16), b.contiguous().view(torch.int16)
        assert torch.equal(a, b), name
    rest = np.setdiff1d(np.arange(NB), ids.cpu().numpy())
    assert int(packed.pp_v4[0][torch.from_numpy(rest).cuda()].sum()) == 0
