"""The work a program has the LOCKS path do on one GPU, as timed cases.

Four kinds, each through the entry points a serving program calls:

* ``decode``: the per-layer select + attend of a single-token decode step
  (``LocksEngine.forward``), one call or the layers of a step captured in a
  HIP graph, with K/V resident or (``mem-v``) V in the DRAM tier;
* ``mla``: the same step over a latent cache (``mla_forward_mqa``);
* ``build``: the summaries of a prompt's pages in every layer
  (``rki4_build_bulk``), and of a latent cache's (d 512);
* ``tail``: the summaries of the pages that a decode step has just filled
  (``rki4_build_tail``).

K, V and latents are N(0, 1) with a few channels scaled up, block tables are
drawn from one shuffled pool, and the summaries that a decode reads are made
here in plain torch, so a case's inputs do not depend on the code it times.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "locks-kv_amd"))

RANK, ROPE, LATENT = 8, 64, 512


def _decode(name, lens, n_kv, group, layers, *, d=128, page=16, budget_pages=126, combine="nrm",
            variant="fast", graph=True):
    return dict(name=name, kind="decode", lens=lens, n_kv=n_kv, group=group, d=d, page=page, layers=layers,
                budget_pages=budget_pages, combine=combine, variant=variant, graph=graph)


def listed():
    return [
        # one layer's attention call of a 16K chat, without a graph: the smallest call a program makes
        _decode("layer-16k-eager", "16384", 8, 4, 1, graph=False),
        # a long-document chat of one user at a 2048-token budget
        _decode("step-128k", "131072", 8, 4, 4),
        # the longest context one user has, wide query groups
        _decode("step-1m", "1048576", 2, 16, 2),
        # four users with contexts of very different lengths
        _decode("step-ragged-4", "262144,196608,131072,65536", 2, 16, 3),
        # a serving batch under the configuration's default budget (10 % of the context)
        _decode("step-batch16-10pct", "32768,31007,28123,24576,21333,19001,16384,15001,12288,11117,9999,8192,"
                "7001,5555,4097,3001", 8, 4, 2, budget_pages=0),
        # a model of another head size and cache page, with the "max" combine
        _decode("step-d64-page32", "50021,12345", 4, 8, 4, d=64, page=32, budget_pages=64, combine="max"),
        # one user of a latent-attention model
        dict(name="mla-128k", kind="mla", lens="131072", layers=4, budget_pages=128),
        # a serving batch of a latent-attention model
        dict(name="mla-batch8", kind="mla", lens="65536,50001,33333,24576,16001,8192,5001,2049", layers=2,
             budget_pages=128),
        # a 32K prompt's summaries, once per prompt
        dict(name="build-32k", kind="build", lens="32768", n_kv=8, d=128, page=16, layers=8),
        # a latent-attention model's prompt
        dict(name="build-latent-32k", kind="build", lens="32768", n_kv=1, d=LATENT, page=16, layers=8),
        # every sixteenth decode step: the pages that four users have just filled, all layers
        dict(name="tail-4", kind="tail", lens="1024,1008,528,272", n_kv=8, d=128, page=16, layers=32),
        # a decode step with V in the DRAM tier, the selected pages already hot
        _decode("step-mem-v", "24576", 8, 4, 2, variant="mem-v"),
    ]


def draw(rng):
    kind = rng.choice(["decode"] * 6 + ["mla"] * 2 + ["build"] * 2 + ["tail"])
    log = lambda lo, hi: int(math.exp(rng.uniform(math.log(lo), math.log(hi))))  # noqa: E731
    d, page = rng.choice([(128, 16)] * 5 + [(64, 16), (256, 16), (128, 32), (128, 64), (64, 32), (256, 64)])
    if kind == "decode":
        n_kv, group = rng.choice([(8, 4), (8, 4), (8, 8), (4, 8), (4, 7), (2, 16), (16, 1), (1, 16)])
        n = rng.choice([1, 1, 2, 4, 8])
        most = min(1 << 20, (1 << 21) * 64 // (n * n_kv * d))
        lens = ",".join(str(log(900, most)) for _ in range(n))
        return {k: v for k, v in _decode("", lens, n_kv, group, rng.choice([1, 2]), d=d, page=page,
                                         budget_pages=rng.choice([0, rng.randint(24, 260)]),
                                         combine=rng.choice(["nrm", "nrm", "max"])).items() if k != "name"}
    if kind == "mla":
        n = rng.choice([1, 1, 3, 6])
        return dict(kind="mla", lens=",".join(str(log(900, 131072 // n)) for _ in range(n)), layers=rng.choice([1, 2]),
                    budget_pages=rng.randint(40, 200))
    if kind == "build":
        if rng.random() < 0.25:
            return dict(kind="build", lens=str(log(500, 30000)), n_kv=1, d=LATENT, page=16, layers=rng.choice([2, 4]))
        return dict(kind="build", lens=str(log(500, 20000)), n_kv=rng.choice([2, 8]), d=d, page=page,
                    layers=rng.choice([1, 2, 4]))
    return dict(kind="tail", lens=",".join(str(log(100, 900)) for _ in range(rng.randint(1, 6))),
                n_kv=rng.choice([2, 8]), d=d, page=page, layers=rng.choice([16, 32]))


# ---- inputs ------------------------------------------------------------------
def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def _page(case):
    return case.get("page", 16)


def _inputs(case, seed):
    """Block table, lengths, and a function that makes one layer's tensors."""
    dev, page, lens = torch.device("cuda"), _page(case), _lens(case)
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    npg = [-(-s // page) for s in lens]
    NB, MP = sum(npg) + 5, max(npg)
    perm = torch.randperm(NB, generator=g, device=dev).to(torch.int32)
    bt = torch.zeros(len(lens), MP, dtype=torch.int32, device=dev)
    at = 0
    for r, n in enumerate(npg):
        bt[r, :n] = perm[at:at + n]
        at += n

    def keys(n_kv, d):
        """(NB, page, n_kv, d) bf16: N(0, 1), four channels of each head x8."""
        scale = torch.ones(n_kv, d, device=dev)
        for h in range(n_kv):
            scale[h, torch.randperm(d, generator=g, device=dev)[:4]] = 8.0
        return (torch.randn(NB, page, n_kv, d, generator=g, device=dev) * scale).to(torch.bfloat16)

    def latents():
        """(NB, page, 576) bf16 rows [latent | rope]."""
        scale = torch.exp(torch.randn(LATENT + ROPE, generator=g, device=dev) * 0.5)
        return (torch.randn(NB, page, LATENT + ROPE, generator=g, device=dev) * scale).to(torch.bfloat16)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev).to(torch.bfloat16)

    sl = torch.tensor(lens, dtype=torch.int32, device=dev)
    return dict(lens=lens, npg=npg, NB=NB, MP=MP, bt=bt, sl=sl, keys=keys, latents=latents, normal=normal)


def _summaries(K):
    """rki4 records of every page of K (NB, page, n_kv, d): centroid, a rank-8
    basis from two rounds of subspace iteration, coefficients; quantised."""
    parts = []
    step = max(1, (1 << 25) // (K.shape[1] * K.shape[2] * K.shape[3]))
    for lo in range(0, K.shape[0], step):
        x = K[lo:lo + step].float().permute(0, 2, 1, 3)                   # (n, kv, page, d)
        mu = x.mean(2)
        x = (x - mu[:, :, None]).contiguous()
        w = x[:, :, :RANK].contiguous()
        for it in range(3):
            for i in range(RANK):
                v = w[:, :, i]
                if i:
                    p = w[:, :, :i]
                    v = v - ((p * v[:, :, None]).sum(-1, keepdim=True) * p).sum(2)
                w[:, :, i] = v / v.norm(dim=-1, keepdim=True).clamp(min=1e-6)
            if it < 2:
                w = torch.matmul(torch.matmul(w, x.transpose(2, 3).contiguous()), x)
        c = torch.matmul(x, w.transpose(2, 3).contiguous())               # (n, kv, page, 8)
        ms = (mu.abs().amax(-1) / 127).clamp(min=1e-8)
        vs = (w.abs().amax(-1) / 7).clamp(min=1e-8)
        cs = (c.abs().amax(-1) / 127).clamp(min=1e-8)
        code = (w / vs[..., None]).round().clamp(-8, 7).to(torch.int32) & 15
        parts.append(((code[..., 0::2] | (code[..., 1::2] << 4)).to(torch.uint8), vs.to(torch.bfloat16),
                      (c / cs[..., None]).round().clamp(-127, 127).to(torch.int8), cs.to(torch.bfloat16),
                      (mu / ms[..., None]).round().clamp(-127, 127).to(torch.int8), ms.to(torch.bfloat16)))
    return [torch.cat(t) for t in zip(*parts)]


SLABS = ("pp_v4", "pp_vs", "pp_c8", "pp_cs", "pp_mu8", "pp_mus")


def _fill(st, layer, slabs):
    for name, t in zip(SLABS, slabs):
        getattr(st, name)[layer].copy_(t)


def _decode_layer(case, inp):
    n_kv, d = case["n_kv"], case["d"]
    kv = torch.stack([inp["keys"](n_kv, d), inp["keys"](n_kv, d)], dim=1)
    return kv, inp["normal"](len(inp["lens"]), n_kv * case["group"], d)


def _mla_layer(inp):
    return inp["latents"](), inp["normal"](len(inp["lens"]), 16, LATENT + ROPE)


def _mla_scale():
    return 1.0 / math.sqrt(128 + ROPE)


def _step(forward, graph):
    """A decode step as a program runs it: called, or captured once and replayed."""
    if not graph:
        return forward
    forward()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        forward()
    torch.cuda.synchronize()
    return g.replay


def prepare(case, seed):
    return {"decode": _prepare_decode, "mla": _prepare_mla, "build": _prepare_build, "tail": _prepare_build}[
        case["kind"]](case, seed)


def _prepare_decode(case, seed):
    from locks import LocksConfig
    from locks.backend.engine import LocksEngine
    from locks.selection import derive_page_params

    inp = _inputs(case, seed)
    n, L, n_kv, d = len(inp["lens"]), case["layers"], case["n_kv"], case["d"]
    layers = [_decode_layer(case, inp) for _ in range(L)]
    cfg = LocksConfig(budget_pages=case["budget_pages"] or None, quad_combine=case["combine"],
                      variant=case["variant"])
    eng = LocksEngine(cfg, [kv for kv, _ in layers], num_heads_q=n_kv * case["group"], num_heads_kv=n_kv,
                      head_dim=d, block_size=case["page"], max_num_seqs=n,
                      max_model_len=inp["MP"] * case["page"], max_num_batched_tokens=1024)
    for i, (kv, _) in enumerate(layers):
        _fill(eng.st, i, _summaries(kv[:, 0]))
        if eng.tier is not None:
            eng.tier.offload(i, kv, list(range(inp["NB"])))
    out = [torch.zeros(n, n_kv * case["group"], d, dtype=torch.bfloat16, device="cuda") for _ in layers]
    scale = 1.0 / math.sqrt(d)

    def forward():
        for (kv, q), o in zip(layers, out):
            eng.forward(q, kv, inp["bt"], inp["sl"], n, scale, o)

    derive_page_params(eng.st, inp["sl"], n)
    return dict(step=_step(forward, case["graph"]), hold=(eng, layers, inp),
                outputs=dict(out=out, page_table=eng.st.page_table, page_cnt=eng.st.page_cnt))


def _prepare_mla(case, seed):
    from locks.backend.mla_attn import mla_forward_mqa
    from locks.selection import MlaState

    inp = _inputs(case, seed)
    n, L = len(inp["lens"]), case["layers"]
    layers = [_mla_layer(inp) for _ in range(L)]
    st = MlaState("cuda", num_layers=L, num_blocks=inp["NB"], n_heads=16, max_reqs=n, max_pages=inp["MP"],
                  budget_pages=case["budget_pages"], sink_pages=1, window_pages=10)
    for i, (c, _) in enumerate(layers):
        _fill(st, i, _summaries(c[:, :, None, :LATENT]))
    out = [torch.zeros(n, 16, LATENT, dtype=torch.bfloat16, device="cuda") for _ in layers]
    lse = [torch.zeros(n, 16, device="cuda") for _ in layers]

    def forward():
        for i, (c, q) in enumerate(layers):
            mla_forward_mqa(q, c, inp["bt"], inp["sl"], st, _mla_scale(), out=out[i], lse=lse[i], layer=i,
                            derive=i == 0)

    return dict(step=_step(forward, True), hold=(st, layers, inp),
                outputs=dict(out=out, lse=lse, page_table=st.page_table, page_cnt=st.page_cnt))


def _build_layer(case, inp):
    """One layer's K pages as the builder takes them: a view into the cache."""
    if case["d"] == LATENT:
        return inp["latents"]()[:, :, None, :LATENT]
    return inp["keys"](case["n_kv"], case["d"])


def _prepare_build(case, seed):
    from locks.selection import MlaState, Rki4State, rki4_build_bulk, rki4_build_tail

    inp = _inputs(case, seed)
    n, L, page = len(inp["lens"]), case["layers"], case["page"]
    K = [_build_layer(case, inp) for _ in range(L)]
    if case["d"] == LATENT:
        st = MlaState("cuda", num_layers=L, num_blocks=inp["NB"], n_heads=16, max_reqs=n, max_pages=inp["MP"])
    else:
        st = Rki4State("cuda", num_layers=L, num_blocks=inp["NB"], n_kv=case["n_kv"], G=4, head_dim=case["d"],
                       page=page, max_reqs=n, max_pages=inp["MP"])

    def step():
        if case["kind"] == "tail":
            rki4_build_tail(st, K, inp["bt"], inp["sl"], n)
        else:
            rki4_build_bulk(st, K, inp["bt"], inp["sl"], n, max(inp["lens"]) // page)

    return dict(step=step, hold=inp, outputs={k: getattr(st, k) for k in SLABS + ("pp_tag",)})


def run(state):
    state["step"]()
    return state["outputs"]


# ---- what a pass cannot do without --------------------------------------------
def _budget(case, npg, window, sink):
    """Selected pages of a row of npg pages, the forced ones among them."""
    lo, hi = min(sink, npg), max(npg - window, min(sink, npg))
    if hi - lo <= 1:
        return npg
    if case["kind"] == "mla":
        b = max(case["budget_pages"] - sink - window, 1)
    else:
        b = case["budget_pages"] or max(1, math.ceil((hi - lo) * 0.1))
    return lo + min(b, hi - lo) + npg - hi


def _record(d, page):
    return 5 * d + 10 * page + 18


def work(case):
    page, lens = _page(case), _lens(case)
    if case["kind"] in ("build", "tail"):
        d = case["d"]
        pages = sum(s // page for s in lens) if case["kind"] == "build" else len(lens)
        grams = pages * case["n_kv"] * case["layers"]
        # K in, record and tag out; the gram, a symmetric eigensolve (about 9 n^3) and the basis
        return dict(bytes=grams * (2 * page * d + _record(d, page) + 16),
                    flops=grams * (2 * page * page * d + 9 * page ** 3 + 2 * page * d * RANK))
    mla = case["kind"] == "mla"
    n_kv, G, d, window = (1, 16, LATENT, 10) if mla else (case["n_kv"], case["group"], case["d"], 1)
    summary = _record(d, page) + (2 * page * ROPE if mla else 0)
    row = (LATENT + ROPE) if mla else 2 * d
    total = flops = 0
    for s in lens:
        npg = -(-s // page)
        cnt = _budget(case, npg, window, 1)
        total += n_kv * (max(npg - window, 0) * summary + cnt * page * row * 2 + 4 * G * d) + 4 * npg
        flops += n_kv * G * (max(npg - window, 0) * 2 * (9 * d + page * (RANK + (ROPE if mla else 0)))
                             + cnt * page * 2 * (d + (d + ROPE if mla else d)))
    return dict(bytes=total * case["layers"], flops=flops * case["layers"])


def tolerance(case):
    if case["kind"] in ("build", "tail"):
        # scales are bf16 (half an ulp is 0.4 %); a code may fall on the other side of a rounding
        # boundary, and a pair of near-equal eigenvalues may turn by any angle in its plane
        return {"rel": 5e-3, "max": 0.6, "differ": 2e-3}
    # bf16 outputs over fp16 probabilities; a page at the budget's edge may change places with a near-equal one
    return {"rel": 1e-2, "max": 0.4, "differ": 5e-3}


# ---- the same in 64 bits --------------------------------------------------------
def _q8(q):
    """int8 rounding of q per head, as whole numbers and their scale, in 64 bits."""
    qf = q.float()
    s = qf.abs().amax(-1, keepdim=True).clamp(min=1e-8) / 127
    return torch.round(qf / s).double(), s.double()


def _unpack(v4):
    lo, hi = (v4 & 15).to(torch.int32), (v4 >> 4).to(torch.int32)
    c = torch.stack([lo, hi], -1).flatten(-2)
    return torch.where(c > 7, c - 16, c).double()


def _tokens(slabs, blk, q8, qs):
    """Estimated q.k of every token (pages, kv, G, page): q8 (kv, G, d), qs (kv, G, 1)."""
    v4, vs, c8, cs, mu8, mus = (t[blk] for t in slabs)
    qt = torch.matmul(q8, _unpack(v4).transpose(-1, -2).contiguous()) * vs.double()[:, :, None]   # (P, kv, G, 8)
    mud = torch.matmul(q8, mu8.double()[..., None])[..., 0] * mus.double()[..., None]             # (P, kv, G)
    tok = torch.matmul(qt, c8.double().transpose(-1, -2).contiguous()) * cs.double()[:, :, None]
    return (tok + mud[..., None]) * qs


def _keep(score, npg, b, window, sink):
    """Kept logical pages of one row: sink and window, and the b best others."""
    lo, hi = min(sink, npg), max(npg - window, min(sink, npg))
    if hi - lo <= b or hi - lo <= 1:
        return torch.arange(npg, device=score.device)
    top = torch.topk(score[lo:hi], b).indices + lo
    forced = torch.cat([torch.arange(lo), torch.arange(hi, npg)]).to(score.device)
    return torch.cat([forced, top]).sort().values


def _attend(q, K, V, pages, page, s, scale):
    """Attention of heads q (G, d) over the tokens K, V (n, page, .) of the kept pages."""
    pos = (pages[:, None] * page + torch.arange(page, device=q.device)).reshape(-1)
    x = torch.matmul(q.double(), K.double().flatten(0, 1).t().contiguous()) * scale
    x = x.masked_fill(pos >= s, -math.inf)
    return torch.matmul(torch.softmax(x, -1), V.double().flatten(0, 1)), torch.logsumexp(x, -1)


def exact(case, seed):
    return {"decode": _exact_decode, "mla": _exact_mla, "build": _exact_build, "tail": _exact_build}[
        case["kind"]](case, seed)


def _exact_decode(case, seed):
    inp = _inputs(case, seed)
    n_kv, G, d, page = case["n_kv"], case["group"], case["d"], case["page"]
    scale, outs = 1.0 / math.sqrt(d), []
    for kv, q in [_decode_layer(case, inp) for _ in range(case["layers"])]:
        slabs, rows = _summaries(kv[:, 0]), []
        for r, (s, npg) in enumerate(zip(inp["lens"], inp["npg"])):
            q8, qs = _q8(q[r].view(n_kv, G, d))
            blk, score = inp["bt"][r, :npg].long(), []
            for lo in range(0, npg, 8192):
                score.append(torch.logsumexp(_tokens(slabs, blk[lo:min(lo + 8192, npg)], q8, qs) * scale, -1))
            score = torch.cat(score)[:max(npg - 1, 0)]                     # (P, kv, G), the window's page apart
            if case["combine"] == "nrm":
                score = torch.exp(score - score.amax(0, keepdim=True)).sum(-1) if npg > 1 else score.sum(-1)
            else:
                score = score.amax(-1)
            heads = []
            for h in range(n_kv):
                pages = _keep(score[:, h], npg, _budget(case, npg, 1, 1) - 2, 1, 1)
                t = kv[blk[pages], :, :, h]
                heads.append(_attend(q[r, h * G:(h + 1) * G], t[:, 0], t[:, 1], pages, page, s, scale)[0])
            rows.append(torch.cat(heads))
        outs.append(torch.stack(rows))
    return dict(out=outs, page_table=None, page_cnt=None)


def _exact_mla(case, seed):
    inp = _inputs(case, seed)
    page, scale, outs, lses = _page(case), _mla_scale(), [], []
    for c, q in [_mla_layer(inp) for _ in range(case["layers"])]:
        slabs, rows = _summaries(c[:, :, None, :LATENT]), []
        for r, (s, npg) in enumerate(zip(inp["lens"], inp["npg"])):
            q8, qs = _q8(q[r:r + 1, :, :LATENT])
            blk, score = inp["bt"][r, :npg].long(), []
            for lo in range(0, npg, 4096):
                b = blk[lo:lo + 4096]
                rope = torch.matmul(q[r, :, LATENT:].double(), c[b][:, :, LATENT:].double().transpose(1, 2).contiguous())
                score.append((_tokens(slabs, b, q8, qs)[:, 0] + rope).amax((1, 2)) * scale)
            pages = _keep(torch.cat(score), npg, max(case["budget_pages"] - 11, 1), 10, 1)
            t = c[blk[pages]]
            rows.append(_attend(q[r], t, t[:, :, :LATENT], pages, page, s, scale))
        outs.append(torch.stack([o for o, _ in rows]))
        lses.append(torch.stack([x for _, x in rows]))
    return dict(out=outs, lse=lses, page_table=None, page_cnt=None)


def _exact_build(case, seed):
    """The scales (the codes are whole numbers, and an eigenvector's sign is free)."""
    inp = _inputs(case, seed)
    page, n_kv, NB = case["page"], case["n_kv"], inp["NB"]
    if case["kind"] == "tail":
        done = torch.stack([inp["bt"][r, max(s // page - 1, 0)] for r, s in enumerate(inp["lens"])])
    else:
        done = torch.cat([inp["bt"][r, :s // page] for r, s in enumerate(inp["lens"])])
    done = done.long().unique()
    all_vs, all_cs, all_ms = [], [], []
    for K in [_build_layer(case, inp) for _ in range(case["layers"])]:
        x = K[done].double().permute(0, 2, 1, 3)                           # (n, kv, page, d)
        mu = x.mean(2)
        x = (x - mu[:, :, None]).contiguous()
        w, U = np.linalg.eigh(torch.matmul(x, x.transpose(2, 3).contiguous()).cpu().numpy())
        S = torch.from_numpy(w[..., -RANK:]).cuda().clamp(min=1e-10).sqrt()
        U = torch.from_numpy(np.ascontiguousarray(U[..., -RANK:])).cuda()  # (n, kv, page, 8)
        V = torch.matmul(x.transpose(2, 3).contiguous(), U) / S[:, :, None]
        for into, shape, v in ((all_vs, (RANK,), V.abs().amax(2) / 7), (all_cs, (page,), (U * S[:, :, None]).abs().amax(-1) / 127),
                               (all_ms, (), mu.abs().amax(-1) / 127)):
            t = torch.zeros(NB, n_kv, *shape, dtype=torch.float64, device="cuda")
            t[done] = v
            into.append(t)
    return dict(pp_v4=None, pp_vs=torch.stack(all_vs), pp_c8=None, pp_cs=torch.stack(all_cs), pp_mu8=None,
                pp_mus=torch.stack(all_ms), pp_tag=None)
