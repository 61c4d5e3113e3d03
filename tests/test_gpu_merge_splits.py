"""The split merge in all its forms (one wave per head for up to 8, 16 and 32
splits, 256 threads past that and, at 17 to 32 splits, for few heads) against a
64-bit merge: ragged page counts, an empty row, splits without mass, NaN in the
partials that no split wrote."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (2, 3, 4): 24 heads; (30, 8, 8): 1920, past every head count at which the form changes
@pytest.mark.parametrize("R,n_kv,G", [(2, 3, 4), (30, 8, 8)])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("nsplit", [1, 8, 9, 16, 17, 32, 33])
def test_merge_equals_64_bit(R, n_kv, G, d, nsplit):
    import torch
    from locks.attention.decode import decode_merge
    print(f"[case] R {R} n_kv {n_kv} G {G} d {d} splits {nsplit}", flush=True)
    rng = np.random.default_rng(nsplit * 1000 + d + R)
    split, pps_min, max_cnt = nsplit + 3, 4, nsplit * 4
    cnt = rng.integers(1, max_cnt + 1, (R, n_kv)).astype(np.int32)
    cnt[0, 0], cnt[0, 1], cnt[-1, -1] = 0, max_cnt, 1
    g = torch.Generator(device="cuda").manual_seed(nsplit)
    m = torch.randn(R, n_kv, split, G, generator=g, device="cuda") * 3
    l = torch.rand(R, n_kv, split, G, generator=g, device="cuda") + 0.1
    acc = torch.randn(R, n_kv, split, G, d, generator=g, device="cuda")
    # a split whose tokens are all masked: m = -inf, l = 0, acc = 0
    empty = torch.rand(R, n_kv, split, G, generator=g, device="cuda") < 0.1
    empty[0, 1] = True                                  # a row without any mass: zeros
    m[empty], l[empty], acc[empty] = float("-inf"), 0.0, 0.0
    dcnt = torch.from_numpy(cnt).cuda()
    pps = torch.clamp(-(-dcnt // nsplit), min=pps_min)
    act = torch.arange(split, device="cuda") < torch.clamp(-(-dcnt // pps), max=nsplit)[..., None]
    for t in (m, l, acc):
        t[~act] = float("nan")                          # stale rows
    on = (act[..., None] & ~empty)
    md = torch.where(on, m, float("-inf")).double()
    top = md.amax(2, keepdim=True)
    w = torch.where(on, torch.exp(md - torch.where(top.isinf(), 0.0, top)), 0.0)
    lt = (w * torch.where(on, l, 0.0).double()).sum(2)
    ref = (w[..., None] * torch.where(on[..., None], acc, 0.0).double()).sum(2)
    ref = torch.where(lt[..., None] > 0, ref / lt[..., None], 0.0).reshape(R, n_kv * G, d)
    for dtype, tol in ((torch.float32, 2e-6), (torch.bfloat16, 2.0 ** -8)):
        out = torch.full((R, n_kv * G, d), 9.0, dtype=dtype, device="cuda")
        decode_merge(m, l, acc, dcnt, out, n_req=R, n_kv=n_kv, G=G, split=split, pps_min=pps_min, pt_cols=4096,
                     max_cnt=max_cnt)
        torch.cuda.synchronize()
        # fp32: at most 33 products and sums, each to 2^-24, and the exp to ~2 ulp, of terms up to |acc| max;
        # bf16: half an ulp of the value besides
        bound = tol * torch.clamp(ref.abs(), min=float(acc.nan_to_num(0).abs().max()) if dtype == torch.float32 else 1e-2)
        assert ((out.double() - ref).abs() <= bound).all(), float((out.double() - ref).abs().max())
        assert not out[0, :2 * G].any()                 # no pages; no mass
