"""GPU parity of the HIP hot path against the CPU oracle (calls go through
the C ABI via the locks package).

Bars:
  * scorer: |score_h - oracle| <= 2e-5 on every scored page (the documented
    near-tie band is |dscore| < 1e-5 for ranking decisions);
  * selection: page tables bit-exact for the "max" combine (exact fp32 max)
    and for identical combined scores; with the "nrm" combine (exp) the kept
    sets may differ only at pages whose oracle score lies within 1e-5
    (relative) of the oracle's b-th largest score;
  * attention: bf16 output within max-abs 2e-2 and mean-rel 1e-3 of the fp32
    oracle; fp32 output within 2e-3 max-abs.
"""
from __future__ import annotations

import numpy as np
import pytest

from oracle import locks_oracle as O
from tests.cases import load_slabs, make_case, to_dev

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


def _state(case, *, budget_pages=126, combine="nrm", split=128, sink=1, window=1, L=1):
    import torch
    from locks.attention import ensure_stage_b_buffers
    from locks.selection import Rki4State
    st = Rki4State("cuda", num_layers=L, num_blocks=case.NB, n_kv=case.n_kv, G=case.G,
                   head_dim=case.d, page=case.page, max_reqs=case.R, max_pages=case.MP,
                   budget=0.1, budget_pages=budget_pages, sink_pages=sink,
                   window_pages=window, combine=combine)
    ensure_stage_b_buffers(st, torch.device("cuda"), split)
    return st


def _derive_np(case, st):
    return O.derive_page_params(case.seq_lens, case.page, st.window_pages, st.sink_pages,
                                st.budget_abs, st.budget)


def _near_tie_ok(gpu_tab, gpu_cnt, ora_tab, ora_cnt, ora_score, npg, nsh, bfix, sink, rel=1e-5):
    """Kept sets equal except at oracle near-ties of the b-th largest score."""
    R, n_kv = gpu_cnt.shape
    n_diff = 0
    for r in range(R):
        for kh in range(n_kv):
            a = set(gpu_tab[r, kh, :gpu_cnt[r, kh]].tolist())
            b = set(ora_tab[r, kh, :ora_cnt[r, kh]].tolist())
            if a == b:
                continue
            assert gpu_cnt[r, kh] == ora_cnt[r, kh]
            sel = ora_score[r, kh, sink:nsh[r]]
            tau = np.sort(sel)[::-1][bfix[r] - 1]
            for p in a ^ b:
                assert abs(ora_score[r, kh, p] - tau) <= rel * max(abs(tau), 1e-30), \
                    f"page {p} differs and is not a near-tie (r={r} kh={kh})"
                n_diff += 1
    return n_diff


@pytest.mark.parametrize("n_kv,G,ctx", [(8, 4, 16384), (2, 16, 8192), (4, 8, 4096),
                                        (2, 3, 3000)])
def test_score_matches_oracle(n_kv, G, ctx):
    import torch
    from locks.selection import derive_page_params, rki4_score_only
    say("score", n_kv, G, ctx)
    case = make_case(0, n_kv, G, [ctx])
    st = _state(case)
    load_slabs(st, 0, case.slabs)
    d = to_dev(case)
    derive_page_params(st, d["sl"], case.R)
    rki4_score_only(st, 0, d["q"], d["bt"], d["sl"], case.R, case.scale)
    torch.cuda.synchronize()
    npg, nsh, b = _derive_np(case, st)
    ref = O.score_rki4_twin(case.q, case.slabs, case.bt, nsh, n_kv, G, case.scale, case.MP)
    ref64 = O.score_rki4_intpath(case.q, case.slabs, case.bt, nsh, n_kv, G, case.scale,
                                 case.MP, dtype=np.float64)
    got = st.score_h.cpu().numpy()
    P = int(nsh[0])
    err = np.abs(got[..., :P] - ref[..., :P]).max()
    err64 = np.abs(got[..., :P] - ref64[..., :P]).max()
    say(f"max|gpu-twin|={err:.3e} max|gpu-exact|={err64:.3e}")
    assert err <= 2e-5 and err64 <= 2e-5
    # per-chunk maxima published for the selector
    pm = st.page_max.cpu().numpy().transpose(0, 1, 3, 2)   # (R, n_kv, chunks, 16)
    for z in range(st.score_chunks):
        lo, hi = z * st.score_chunk, min((z + 1) * st.score_chunk, P)
        for kh in range(n_kv):
            for g in range(G):
                exp = got[0, kh, g, lo:hi].max() if hi > lo else -np.inf
                assert pm[0, kh, z, g] == exp


@pytest.mark.parametrize("n_kv,G", [(8, 4), (2, 16)])
def test_score_q_quantisation_ties(n_kv, G):
    """q rows whose q / qs quotients are exact half-integers (qs = 2^-4): the
    scorer must round them to even exactly as the reference's rint does.  A
    half-away-from-zero quantiser would move the scores by far more than the
    tolerance (checked on the oracle), so the test pins the tie path."""
    import torch
    from locks.selection import derive_page_params, rki4_score_only
    say("score q ties", n_kv, G)
    case = make_case(11, n_kv, G, [4096])
    rng = np.random.default_rng(12)
    H, d = n_kv * G, case.d
    k = rng.integers(-120, 120, size=(1, H, d))
    qv = (k + 0.5) / 16.0                                 # every quotient a tie
    qv[:, :, 0] = 127.0 / 16.0                             # row max -> qs = 2^-4
    away = np.where(k >= 0, k + 1, k) / 16.0               # ties rounded away from 0
    away[:, :, 0] = 127.0 / 16.0
    case.q = O.f32_to_bf16(qv.astype(np.float32))
    assert np.array_equal(O.bf16_to_f32(case.q), qv.astype(np.float32))   # bf16-exact
    q_away = O.f32_to_bf16(away.astype(np.float32))
    st = _state(case)
    load_slabs(st, 0, case.slabs)
    dv = to_dev(case)
    derive_page_params(st, dv["sl"], case.R)
    rki4_score_only(st, 0, dv["q"], dv["bt"], dv["sl"], case.R, case.scale)
    torch.cuda.synchronize()
    npg, nsh, b = _derive_np(case, st)
    P = int(nsh[0])
    ref = O.score_rki4_twin(case.q, case.slabs, case.bt, nsh, n_kv, G, case.scale, case.MP)
    ref_away = O.score_rki4_twin(q_away, case.slabs, case.bt, nsh, n_kv, G, case.scale, case.MP)
    got = st.score_h.cpu().numpy()
    assert np.abs(ref_away[..., :P] - ref[..., :P]).max() > 1e-3
    assert np.abs(got[..., :P] - ref[..., :P]).max() <= 2e-5


def _random_select_inputs(seed, n_kv, G, seq_lens, MP, st, ties=None):
    """Upload a synthetic score_h + consistent per-chunk maxima."""
    import torch
    rng = np.random.default_rng(seed)
    R = len(seq_lens)
    sh = rng.standard_normal((R, n_kv, G, MP)).astype(np.float32) * 3
    if ties == "all_equal":
        sh[:] = 1.5
    elif ties == "bands":
        sh = np.round(sh).astype(np.float32)          # few distinct values
    elif ties == "underflow":
        sh[..., ::7] = -200.0                         # exp underflows to +0
        sh = np.where(rng.random(sh.shape) < 0.5, -300.0, sh).astype(np.float32)
    elif ties == "sparse_peaks":
        # fewer normal pages than the budget: the b-th key sits far below
        # the row maximum (the selector's absolute-radix fallback)
        keep = np.zeros(sh.shape, bool)
        for idx in np.ndindex(*sh.shape[:3]):
            keep[idx][rng.choice(MP, size=min(40, MP), replace=False)] = True
        sh = np.where(keep, sh, -300.0).astype(np.float32)
    elif ties == "far":
        # a second cluster ~40 units (about 58 binades of exp) below
        sh = np.where(rng.random(sh.shape) < 0.025, sh, sh - 40.0).astype(np.float32)
    npg, nsh, b = O.derive_page_params(seq_lens, 16, st.window_pages, st.sink_pages,
                                       st.budget_abs, st.budget)
    pm = np.full((R, n_kv, st.score_chunks, 16), -np.inf, np.float32)
    for r in range(R):
        for z in range(st.score_chunks):
            lo, hi = z * st.score_chunk, min((z + 1) * st.score_chunk, nsh[r])
            if hi > lo:
                pm[r, :, z, :G] = sh[r, :, :, lo:hi].max(axis=-1)
    st.score_h.copy_(torch.from_numpy(sh))
    st.page_max.copy_(torch.from_numpy(np.ascontiguousarray(pm.transpose(0, 1, 3, 2))))
    return sh, npg, nsh, b


@pytest.mark.parametrize("combine", ["max", "nrm"])
@pytest.mark.parametrize("seq_lens,n_kv,G,bp", [
    ([16384], 8, 4, 126),            # whole-row kernel, 4 pages/thread
    ([131072], 8, 4, 126),           # Llama 128K: whole-row kernel, 8 pages/thread
    ([200000], 2, 16, 126),          # chunks of 1024 pages, G=16
    ([40000], 2, 4, 1000),           # whole-row kernel, 4 pages/thread, large b
    ([1 << 20], 2, 16, 126),         # 1M context, 32 chunks
    ([262144, 196608, 131072, 65536], 2, 16, 126),   # ragged batch
    ([100000], 2, 4, 5000),          # whole-row kernel, 8 pages/thread, large b
    ([400000], 2, 4, 5000),          # histogram (band) route: b * chunks > register finisher
    ([1 << 20], 2, 16, 6553),        # 1M at the default 10 % budget: band route
    ([262144], 2, 16, 1638),         # 16 candidates per thread in the finisher
    ([40, 17, 0, 33], 2, 4, 126),    # short rows, padded row, keep-all
])
def test_select_matches_oracle(combine, seq_lens, n_kv, G, bp):
    import torch
    from locks.selection import derive_page_params, rki4_select_only
    say("select", combine, seq_lens, n_kv, G, bp)
    MP = max(1, max((s + 15) // 16 for s in seq_lens))
    case = make_case(1, n_kv, G, seq_lens, MP=MP, kv=False)
    st = _state(case, budget_pages=bp, combine=combine)
    d = to_dev(case)
    derive_page_params(st, d["sl"], case.R)
    sh, npg, nsh, b = _random_select_inputs(2, n_kv, G, seq_lens, MP, st)
    rki4_select_only(st, case.R)
    torch.cuda.synchronize()
    first = (st.page_table.clone(), st.page_cnt.clone())
    for _ in range(2):                  # repeated calls: arrival counters reset
        st.page_table.fill_(7)
        rki4_select_only(st, case.R)
        torch.cuda.synchronize()
        assert torch.equal(st.page_table, first[0]) and torch.equal(st.page_cnt, first[1])
    assert (st.n_pages.cpu().numpy() == npg).all() and (st.n_sel_hi.cpu().numpy() == nsh).all()
    assert (st.b_fix.cpu().numpy() == b).all()
    comb = O.combine_nrm(sh, nsh) if combine == "nrm" else O.combine_max(sh, nsh)
    tab, cnt = O.topb_select(comb, npg, nsh, b, st.sink_pages, MP)
    gtab, gcnt = st.page_table.cpu().numpy(), st.page_cnt.cpu().numpy()
    gsc = st.score.cpu().numpy()
    for r in range(case.R):
        P = max(int(nsh[r]), 0)
        if combine == "max":
            assert np.array_equal(gsc[r, :, :P], comb[r, :, :P])
        else:
            assert np.abs(gsc[r, :, :P] - comb[r, :, :P]).max(initial=0) <= 1e-5 * G
    assert np.array_equal(gcnt, cnt)
    if combine == "max":
        assert np.array_equal(gtab, tab)
    else:
        nd = _near_tie_ok(gtab, gcnt, tab, cnt, comb, npg, nsh, b, st.sink_pages)
        say("near-tie differences:", nd)
        # ascending, -1 padded layout holds regardless
        for r in range(case.R):
            for kh in range(n_kv):
                row = gtab[r, kh]
                c = gcnt[r, kh]
                assert (np.diff(row[:c]) > 0).all() and (row[c:] == -1).all()
    # exact bit-level check of the selector itself: feed the GPU's own combined
    # scores to the oracle top-b
    tab2, cnt2 = O.topb_select(gsc, npg, nsh, b, st.sink_pages, MP)
    assert np.array_equal(gtab, tab2) and np.array_equal(gcnt, cnt2)


@pytest.mark.parametrize("combine", ["max", "nrm"])
def test_select_band_route_batch_size_changes(combine):
    """One state on the histogram (band) route called with n_req = 4, then 1,
    then 4: the row histograms must be zero on entry to every call whatever
    the previous call's batch size (the workspace layout is fixed by its
    capacity, not by n_req).  Every call is checked against the oracle."""
    import torch
    from locks.selection import derive_page_params, rki4_select_only
    seq_all = [400000, 300000, 350000, 380000]
    n_kv, G, bp = 2, 4, 5000
    MP = max((s + 15) // 16 for s in seq_all)
    case = make_case(5, n_kv, G, seq_all, MP=MP, kv=False)
    st = _state(case, budget_pages=bp, combine=combine)
    for it, R in enumerate((4, 1, 4, 1)):
        seq = seq_all[:R] if it < 2 else seq_all[::-1][:R]
        say("band route", combine, "call", it, "n_req", R, seq)
        sl = torch.tensor(seq, dtype=torch.int32, device="cuda")
        derive_page_params(st, sl, R)
        sh, npg, nsh, b = _random_select_inputs(40 + it, n_kv, G, seq, MP, st)
        st.page_table.fill_(7)
        rki4_select_only(st, R)
        torch.cuda.synchronize()
        gtab = st.page_table[:R].cpu().numpy()
        gcnt = st.page_cnt[:R].cpu().numpy()
        gsc = st.score[:R].cpu().numpy()
        tab2, cnt2 = O.topb_select(gsc, npg, nsh, b, st.sink_pages, MP)
        assert np.array_equal(gtab, tab2) and np.array_equal(gcnt, cnt2), f"call {it}"
        if combine == "max":
            comb = O.combine_max(sh[:R], nsh)
            tab, cnt = O.topb_select(comb, npg, nsh, b, st.sink_pages, MP)
            assert np.array_equal(gtab, tab) and np.array_equal(gcnt, cnt)


@pytest.mark.parametrize("ties", ["all_equal", "bands", "underflow", "sparse_peaks", "far"])
@pytest.mark.parametrize("ctx,bp", [(16384, 126), (131072, 126), (1 << 19, 126), (1 << 19, 3000)])
def test_select_tie_batteries(ties, ctx, bp):
    import torch
    from locks.selection import derive_page_params, rki4_select_only
    say("ties", ties, ctx, bp)
    n_kv, G = 2, 8
    case = make_case(3, n_kv, G, [ctx], kv=False)
    for combine in ("max", "nrm"):
        st = _state(case, budget_pages=bp, combine=combine)
        d = to_dev(case)
        derive_page_params(st, d["sl"], 1)
        sh, npg, nsh, b = _random_select_inputs(4, n_kv, G, [ctx], case.MP, st, ties=ties)
        rki4_select_only(st, 1)
        torch.cuda.synchronize()
        gsc = st.score.cpu().numpy()
        tab, cnt = O.topb_select(gsc, npg, nsh, b, st.sink_pages, case.MP)
        assert np.array_equal(st.page_table.cpu().numpy(), tab)
        assert np.array_equal(st.page_cnt.cpu().numpy(), cnt)


def _decode_check(case, st, d, out, tab, cnt, rel=1e-3, mabs=2e-2):
    import torch
    got = out.float().cpu().numpy()
    ref, _ = O.decode_attention(case.q, case.k, case.v, case.bt, case.seq_lens, tab, cnt,
                                case.G, case.scale)
    if out.dtype == torch.bfloat16:
        ref_cmp = O.bf16_round(ref.astype(np.float32))
        err = np.abs(got - ref_cmp)
        mr = err.sum() / max(np.abs(ref_cmp).sum(), 1e-30)
        say(f"bf16 out: max-abs {err.max():.3e} mean-rel {mr:.3e}")
        assert err.max() <= mabs and mr <= rel
    else:
        err = np.abs(got - ref)
        say(f"fp32 out: max-abs {err.max():.3e}")
        assert err.max() <= 2e-3
    assert np.isfinite(got).all()


@pytest.mark.parametrize("n_kv,G,seq_lens,split", [
    (8, 4, [16384], 128), (2, 16, [131072], 128), (2, 16, [65536, 49152, 32768, 16384], 64),
    (4, 5, [1000, 7, 0, 4099], 32), (2, 16, [20000], 1)])
@pytest.mark.parametrize("max_cnt", [0, 128, 10])
def test_decode_matches_oracle(n_kv, G, seq_lens, split, max_cnt):
    """max_cnt: the grid-sizing bound of page_cnt (0 none; 128 = b + sink +
    window, the true bound; 10 = a bound below the real counts, which must
    still decode every page, in fewer, longer splits)."""
    import torch
    from locks.attention import decode_merge, decode_splitk
    from locks.attention.decode import _pps_min, _split_kv
    say("decode", n_kv, G, seq_lens, split, max_cnt)
    MP = max(1, max((s + 15) // 16 for s in seq_lens))
    case = make_case(5, n_kv, G, seq_lens, MP=MP, build=False)
    rng = np.random.default_rng(6)
    npg, nsh, b = O.derive_page_params(seq_lens, 16, 1, 1, 126, 0.1)
    sc = rng.random((case.R, n_kv, MP)).astype(np.float32)
    tab, cnt = O.topb_select(sc, npg, nsh, b, 1, MP)
    st = _state(case, split=split)
    d = to_dev(case)
    st.page_table.copy_(torch.from_numpy(tab))
    st.page_cnt.copy_(torch.from_numpy(cnt))
    k, v = _split_kv(d["kv"])
    for dt in (torch.bfloat16, torch.float32):
        out = torch.full((case.R, n_kv * G, 128), float("nan"), dtype=dt, device="cuda")
        pps = _pps_min(case.R)
        decode_splitk(d["q"], k, v, d["bt"], d["sl"], st.page_table, st.page_cnt, st.m_part,
                      st.l_part, st.acc_part, n_req=case.R, G=G, split=st.split,
                      pps_min=pps, scale=case.scale, max_cnt=max_cnt)
        decode_merge(st.m_part, st.l_part, st.acc_part, st.page_cnt, out, n_req=case.R,
                     n_kv=n_kv, G=G, split=st.split, pps_min=pps,
                     pt_cols=st.page_table.shape[2], max_cnt=max_cnt)
        torch.cuda.synchronize()
        _decode_check(case, st, d, out, tab, cnt)


@pytest.mark.parametrize("n_kv,G,seq_lens,split", [
    (8, 4, [16384], 128), (2, 16, [131072], 128), (4, 5, [1000, 7, 0, 4099], 32),
    (2, 16, [65536, 49152, 32768, 16384], 64), (2, 16, [20000], 1)])
@pytest.mark.parametrize("max_cnt", [0, 128, 10])
def test_fused_decode_equals_split_and_merge(n_kv, G, seq_lens, split, max_cnt):
    """The one-launch decode (last split of a row merges it) equals split +
    the head-parallel merge up to fp32 reassociation (the two merges sum the
    splits in different orders), on repeated calls (the arrival counts
    return to zero) and for rows with nothing selected (exact zeros)."""
    import torch
    from locks.attention import decode_merge, decode_splitk
    from locks.attention.decode import _pps_min, _split_kv, decode_fused
    say("fused decode", n_kv, G, seq_lens, split, max_cnt)
    MP = max(1, max((s + 15) // 16 for s in seq_lens))
    case = make_case(9, n_kv, G, seq_lens, MP=MP, build=False)
    rng = np.random.default_rng(10)
    npg, nsh, b = O.derive_page_params(seq_lens, 16, 1, 1, 126, 0.1)
    st = _state(case, split=split)
    d = to_dev(case)
    k, v = _split_kv(d["kv"])
    pps = _pps_min(case.R, n_kv)
    for call in range(3):
        sc = rng.random((case.R, n_kv, MP)).astype(np.float32)
        tab, cnt = O.topb_select(sc, npg, nsh, b, 1, MP)
        st.page_table.copy_(torch.from_numpy(tab))
        st.page_cnt.copy_(torch.from_numpy(cnt))
        dt = torch.float32 if call == 1 else torch.bfloat16
        ref = torch.full((case.R, n_kv * G, 128), float("nan"), dtype=dt, device="cuda")
        out = torch.full_like(ref, float("nan"))
        decode_splitk(d["q"], k, v, d["bt"], d["sl"], st.page_table, st.page_cnt, st.m_part,
                      st.l_part, st.acc_part, n_req=case.R, G=G, split=st.split,
                      pps_min=pps, scale=case.scale, max_cnt=max_cnt)
        decode_merge(st.m_part, st.l_part, st.acc_part, st.page_cnt, ref, n_req=case.R,
                     n_kv=n_kv, G=G, split=st.split, pps_min=pps,
                     pt_cols=st.page_table.shape[2], max_cnt=max_cnt)
        decode_fused(d["q"], k, v, d["bt"], d["sl"], st.page_table, st.page_cnt, st.m_part,
                     st.l_part, st.acc_part, st.dec_counters, out, n_req=case.R, G=G,
                     split=st.split, pps_min=pps, scale=case.scale, max_cnt=max_cnt)
        torch.cuda.synchronize()
        a, b_ = out.float(), ref.float()
        assert torch.isfinite(a).all()
        if dt == torch.float32:
            assert (a - b_).abs().max().item() <= 1e-5 * max(1.0, b_.abs().max().item())
        else:                                    # at most one bf16 ulp apart
            assert ((a - b_).abs() <= b_.abs() * 2.0 ** -7 + 1e-30).all()
        assert torch.equal(a == 0, b_ == 0)
        assert int(st.dec_counters.abs().sum()) == 0


def test_dense_equality_and_split_invariance():
    """Selecting every page reproduces dense attention; any split count gives
    the same result up to fp32 reassociation."""
    import torch
    from locks.attention import decode_merge, decode_splitk
    from locks.attention.decode import _split_kv
    say("dense equality")
    n_kv, G, sl = 2, 16, [9000]
    case = make_case(7, n_kv, G, sl, build=False)
    npg = (sl[0] + 15) // 16
    tab = np.full((1, n_kv, case.MP), -1, np.int32)
    tab[:, :, :npg] = np.arange(npg)
    cnt = np.full((1, n_kv), npg, np.int32)
    d = to_dev(case)
    k, v = _split_kv(d["kv"])
    outs = []
    for split in (1, 7, 64, 512):
        st = _state(case, split=split)
        st.page_table.copy_(torch.from_numpy(tab))
        st.page_cnt.copy_(torch.from_numpy(cnt))
        out = torch.empty((1, n_kv * G, 128), dtype=torch.float32, device="cuda")
        decode_splitk(d["q"], k, v, d["bt"], d["sl"], st.page_table, st.page_cnt, st.m_part,
                      st.l_part, st.acc_part, n_req=1, G=G, split=split, pps_min=1,
                      scale=case.scale)
        decode_merge(st.m_part, st.l_part, st.acc_part, st.page_cnt, out, n_req=1,
                     n_kv=n_kv, G=G, split=split, pps_min=1,
                     pt_cols=st.page_table.shape[2])
        torch.cuda.synchronize()
        outs.append(out.cpu().numpy())
    # dense reference through torch SDPA in float64 (independent of the oracle)
    K = O.bf16_to_f32(case.k[case.bt[0, :npg]]).reshape(-1, n_kv, 128)[:sl[0]]
    V = O.bf16_to_f32(case.v[case.bt[0, :npg]]).reshape(-1, n_kv, 128)[:sl[0]]
    Q = O.bf16_to_f32(case.q[0]).reshape(n_kv, G, 128)
    qt = torch.from_numpy(Q).double()
    kt = torch.from_numpy(K).double().permute(1, 0, 2)[:, None]
    vt = torch.from_numpy(V).double().permute(1, 0, 2)[:, None]
    ref = torch.nn.functional.scaled_dot_product_attention(
        qt[:, :, None], kt.expand(-1, G, -1, -1), vt.expand(-1, G, -1, -1))
    ref = ref[:, :, 0].reshape(1, n_kv * G, 128).numpy()
    for o in outs:
        assert np.abs(o - ref).max() <= 2e-3
        # splits differ only by fp16 rounding of P relative to each split max
        assert np.abs(o - outs[0]).max() <= 1e-3


@pytest.mark.parametrize("n_kv,G,seq_lens", [(2, 16, [9000, 4097, 16, 1]), (8, 4, [20000])])
@pytest.mark.parametrize("split", [1, 37, 256])
def test_dense_comparator_matches_sdpa(n_kv, G, seq_lens, split):
    """The dense full-KV decode (every page of the row, no page table) equals
    float64 SDPA over the row's first seq_len tokens, for ragged rows
    (partial last page, a one-page row, a one-token row) and any split."""
    import torch
    from locks.attention import decode_dense
    from locks.attention.decode import _split_kv
    say("dense comparator", n_kv, G, seq_lens, split)
    case = make_case(8, n_kv, G, seq_lens, build=False)
    d = to_dev(case)
    k, v = _split_kv(d["kv"])
    R = case.R
    mp = torch.empty(R, n_kv, split, G, device="cuda")
    lp = torch.empty_like(mp)
    ap = torch.empty(R, n_kv, split, G, 128, device="cuda")
    for dt in (torch.float32, torch.bfloat16):
        out = torch.full((R, n_kv * G, 128), float("nan"), dtype=dt, device="cuda")
        decode_dense(d["q"], k, v, d["bt"], d["sl"], mp, lp, ap, out, n_req=R, G=G,
                     split=split, scale=case.scale)
        torch.cuda.synchronize()
        got = out.float().cpu().numpy()
        for r, sl in enumerate(seq_lens):
            npg = (sl + 15) // 16
            K = O.bf16_to_f32(case.k[case.bt[r, :npg]]).reshape(-1, n_kv, 128)[:sl]
            V = O.bf16_to_f32(case.v[case.bt[r, :npg]]).reshape(-1, n_kv, 128)[:sl]
            Q = O.bf16_to_f32(case.q[r]).reshape(n_kv, G, 128)
            qt = torch.from_numpy(Q).double()
            kt = torch.from_numpy(K).double().permute(1, 0, 2)[:, None]
            vt = torch.from_numpy(V).double().permute(1, 0, 2)[:, None]
            ref = torch.nn.functional.scaled_dot_product_attention(
                qt[:, :, None], kt.expand(-1, G, -1, -1), vt.expand(-1, G, -1, -1),
                scale=float(case.scale))
            ref = ref[:, :, 0].reshape(n_kv * G, 128).numpy()
            # north-star bar for both output types: P is fp16 (the reference's
            # P.V precision), ~2^-11 |v| per token, unaveraged on short rows
            rb = ref if dt == torch.float32 else O.bf16_round(ref.astype(np.float32))
            e = np.abs(got[r] - rb)
            assert e.max() <= 2e-2 and e.sum() / np.abs(rb).sum() <= 1e-3, f"row {r}: {e.max()}"


@pytest.mark.parametrize("budget_pages", [126, 128])
def test_end_to_end_runtime_path(budget_pages):
    """The reference's call sites (select adapter + decode dispatch) on one
    layer vs the oracle pipeline; budget 126 (+ sink + window = 128 attended
    pages) and the quickstart budget_pages=128."""
    import torch
    from locks.backend import _runtime
    from locks.config import LocksConfig
    from locks.selection import derive_page_params
    say("e2e runtime", budget_pages)
    n_kv, G, sl = 2, 16, [16384, 5000]
    case = make_case(9, n_kv, G, sl)
    st = _state(case, L=2, budget_pages=budget_pages)
    load_slabs(st, 1, case.slabs)
    d = to_dev(case)
    kv = d["kv"]
    st._layer_of = {kv.data_ptr(): 1}
    cfg = LocksConfig(budget_pages=budget_pages)
    derive_page_params(st, d["sl"], case.R)
    out = torch.zeros((case.R, n_kv * G, 128), dtype=torch.bfloat16, device="cuda")
    _runtime._rki4_select_adapter(d["q"], kv, d["bt"], d["sl"], st, case.R, case.scale, cfg)
    _runtime.decode_dispatch(d["q"], kv, d["bt"], d["sl"], st, out, None, case.scale, cfg)
    torch.cuda.synchronize()
    npg, nsh, b = _derive_np(case, st)
    sh = O.score_rki4_twin(case.q, case.slabs, case.bt, nsh, n_kv, G, case.scale, case.MP)
    comb = O.combine_nrm(sh, nsh)
    tab, cnt = O.topb_select(comb, npg, nsh, b, 1, case.MP)
    gtab, gcnt = st.page_table.cpu().numpy(), st.page_cnt.cpu().numpy()
    nd = _near_tie_ok(gtab, gcnt, tab, cnt, comb, npg, nsh, b, 1)
    say("near-tie differences:", nd)
    _decode_check(case, st, d, out, gtab, gcnt)


def _aliased_case(seed, n_kv, G, seq_len, NB=4096):
    """A long row (page ids up to seq_len / 16, a block table that wide) over
    a small physical pool: logical pages map to random blocks of NB, several
    pages per block.  The decode reads only what the block table names, so
    the index arithmetic runs at full length without a full-size cache."""
    import types
    rng = np.random.default_rng(seed)
    MP = (seq_len + 15) // 16
    k, v, _ = O.synth_kv(rng, NB, 16, n_kv, 128)
    q = O.f32_to_bf16(rng.standard_normal((1, n_kv * G, 128), dtype=np.float32))
    bt = rng.integers(0, NB, (1, MP), dtype=np.int32)
    return types.SimpleNamespace(n_kv=n_kv, G=G, seq_lens=[seq_len], MP=MP, NB=NB, k=k, v=v, q=q,
                                 bt=bt, page=16, d=128, R=1, scale=1.0 / np.sqrt(128))


@pytest.mark.parametrize("split,max_cnt", [(128, 128), (128, 0), (64, 10)])
def test_decode_matches_oracle_at_1m(split, max_cnt):
    """BASELINE configs[2]'s row: 1M tokens (65 536 pages, page ids to 65 535
    through a 65 536-wide block table), 2 kv heads x G 16, b = 126 + sink +
    window spread over the row; bf16 and fp32 outputs at the north-star bar."""
    import torch
    from locks.attention import decode_merge, decode_splitk
    from locks.attention.decode import _pps_min, _split_kv
    say("decode 1M", split, max_cnt)
    case = _aliased_case(41, 2, 16, 1 << 20)
    rng = np.random.default_rng(42)
    npg, nsh, b = O.derive_page_params(case.seq_lens, 16, 1, 1, 126, 0.1)
    sc = rng.random((1, 2, case.MP)).astype(np.float32)
    tab, cnt = O.topb_select(sc, npg, nsh, b, 1, case.MP)
    assert int(cnt[0, 0]) == 128 and int(tab[0, 0, 127]) == case.MP - 1
    st = _state(case, split=split)
    d = to_dev(case)
    st.page_table.copy_(torch.from_numpy(tab))
    st.page_cnt.copy_(torch.from_numpy(cnt))
    k, v = _split_kv(d["kv"])
    for dt in (torch.bfloat16, torch.float32):
        out = torch.full((1, 32, 128), float("nan"), dtype=dt, device="cuda")
        pps = _pps_min(1)
        decode_splitk(d["q"], k, v, d["bt"], d["sl"], st.page_table, st.page_cnt, st.m_part,
                      st.l_part, st.acc_part, n_req=1, G=16, split=st.split, pps_min=pps,
                      scale=case.scale, max_cnt=max_cnt)
        decode_merge(st.m_part, st.l_part, st.acc_part, st.page_cnt, out, n_req=1, n_kv=2,
                     G=16, split=st.split, pps_min=pps, pt_cols=st.page_table.shape[2],
                     max_cnt=max_cnt)
        torch.cuda.synchronize()
        _decode_check(case, st, d, out, tab, cnt)


@pytest.mark.parametrize("seq_len,split", [(131072, 128), (131072 + 7, 256)])
def test_dense_comparator_matches_sdpa_at_128k(seq_len, split):
    """The dense comparator over a whole 128K row (8 192 pages; a partial last
    page in the second case) against float64 SDPA over the same tokens."""
    import torch
    from locks.attention import decode_dense
    from locks.attention.decode import _split_kv
    say("dense comparator 128K", seq_len, split)
    n_kv, G = 8, 4
    case = _aliased_case(43, n_kv, G, seq_len)
    d = to_dev(case)
    k, v = _split_kv(d["kv"])
    mp = torch.empty(1, n_kv, split, G, device="cuda")
    lp = torch.empty_like(mp)
    ap = torch.empty(1, n_kv, split, G, 128, device="cuda")
    out = torch.full((1, n_kv * G, 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    decode_dense(d["q"], k, v, d["bt"], d["sl"], mp, lp, ap, out, n_req=1, G=G, split=split,
                 scale=case.scale)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()[0]
    npg = (seq_len + 15) // 16
    K = O.bf16_to_f32(case.k[case.bt[0, :npg]]).reshape(-1, n_kv, 128)[:seq_len]
    V = O.bf16_to_f32(case.v[case.bt[0, :npg]]).reshape(-1, n_kv, 128)[:seq_len]
    Q = O.bf16_to_f32(case.q[0]).reshape(n_kv, G, 128)
    qt = torch.from_numpy(Q).double()
    kt = torch.from_numpy(K).double().permute(1, 0, 2)[:, None]
    vt = torch.from_numpy(V).double().permute(1, 0, 2)[:, None]
    ref = torch.nn.functional.scaled_dot_product_attention(
        qt[:, :, None], kt.expand(-1, G, -1, -1), vt.expand(-1, G, -1, -1), scale=float(case.scale))
    rb = O.bf16_round(ref[:, :, 0].reshape(n_kv * G, 128).numpy().astype(np.float32))
    e = np.abs(got - rb)
    say(f"dense 128K: max-abs {e.max():.3e} mean-rel {e.sum() / np.abs(rb).sum():.3e}")
    assert e.max() <= 2e-2 and e.sum() / np.abs(rb).sum() <= 1e-3
