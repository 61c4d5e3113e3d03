"""Stage B: split-K sparse paged decode + LSE merge on the MI355X kernels.

Call contract of the reference (src/locks/attention/decode.py:130-156,
:328-387): partials m/l (R, n_kv, split, G) and acc (R, n_kv, split, G, D)
fp32 live on the state; pps = max(cdiv(page_cnt, split), pps_min) is derived
on device; ``out`` (T, H, d) rows [0, n_req) are written in place; no host
sync, no allocation.  K comes from the resident paged cache; V through the
V-source seam: the cache's V half or the DRAM tier (``locks.tier``).
"""
from __future__ import annotations

import ctypes

import math

import torch

from .. import _lib

MAX_SPLIT = 512


def _split_kv(kv_cache: torch.Tensor):
    """(K, V) views (num_blocks, page, n_kv, d) for either vLLM cache layout
    ((NB, 2, page, n_kv, d) or (2, NB, page, n_kv, d)); decode.py:64-73."""
    if kv_cache.shape[0] == 2 and kv_cache.shape[1] != 2:
        return kv_cache[0], kv_cache[1]
    if kv_cache.shape[1] == 1:
        return kv_cache.select(1, 0), None
    return kv_cache.select(1, 0), kv_cache.select(1, 1)


def _kv_args(kv_cache: torch.Tensor):
    """What a kernel call takes of _split_kv's views, without making them:
    (K address, V address or None, (block, token, head) element strides,
    (num_blocks, page, n_kv, d))."""
    n0, n1, page, n_kv, d = kv_cache.shape
    s0, s1, st, sh, _ = kv_cache.stride()
    k = kv_cache.data_ptr()
    if n0 == 2 and n1 != 2:
        return k, k + s0 * kv_cache.element_size(), (s1, st, sh), (n1, page, n_kv, d)
    v = None if n1 == 1 else k + s1 * kv_cache.element_size()
    return k, v, (s0, st, sh), (n0, page, n_kv, d)


_NO_V = ("ResidentVSource requires a resident V half; this cache is K-only: decode it with the DRAM "
         "tier's source (locks.tier.TierVSource, mem variants)")


class ResidentVSource:
    """V = the resident engine V half of kv_cache (V_SRC=0, decode.py:76-101)."""

    SRC_ID = 0

    def __init__(self, kv_cache: torch.Tensor):
        _, v = _split_kv(kv_cache)
        if v is None:
            raise ValueError(_NO_V)
        self._v = v

    def args(self):
        v = self._v
        return v, v.stride(0), v.stride(1), v.stride(2)


COUNTER_STRIDE = 64          # ints between rows' arrival counters (LOCKS_DECODE_COUNTER_STRIDE)
# False (default): the split kernel, then one merge workgroup per query head
# (measured faster per step: 1.306 vs 1.321 ms Llama 128K, 2.529 vs 2.612 ms
# GLM 1M -- the fused form merges a whole row's partials through one CU);
# True: one launch whose last split per row merges the row
FUSED_MERGE = False
PPS_MIN_OVERRIDE = None        # set by bench sweeps; None = the table below


def _pps_min(n_req: int, n_kv: int = 8) -> int:
    """Minimum pages per split workgroup (4 waves, 1-2 pages each at bs=1):
    amortises the q load, the 4-wave LDS merge and the partial store.
    Measured on MI355X at 128 attended pages per row: the best keeps ~256
    split workgroups, i.e. rows / 2 pages per split (at least 4) for rows =
    n_req x n_kv.  Steps at pps_min 16 / 8 / 4: GLM ragged batch of 4 (8
    rows) 1.907 / 1.853 / 1.846 ms, GLM 8 x 64K (16 rows) 1.765 / 1.733 /
    1.801, Llama 4 requests (32 rows) 2.108 / 2.168 / 2.268; bs = 1: Llama
    (8 rows) 4, GLM 1M (2 rows) at 8 / 4 / 2: 2.089-2.093 / 2.048-2.073 /
    2.071-2.084.  From 16 requests 32 (Llama 16 x 32K: 2.88-2.90 ms against
    2.89-2.99 at 16)."""
    if PPS_MIN_OVERRIDE:
        return int(PPS_MIN_OVERRIDE)
    if n_req >= 16:
        return 32
    half = max(1, -(-int(n_req) * int(n_kv) // 2))
    return min(16, max(4, 1 << (half - 1).bit_length()))


def _adaptive_split(max_reqs: int, max_pages: int, budget: float, hard_cap: int) -> int:
    """Allocation-time split count: about the number of active splits the
    expected selection needs at low batch (decode.py:103-127), capped."""
    if int(max_reqs) > 4:
        return min(hard_cap, MAX_SPLIT)
    pps = _pps_min(int(max_reqs))
    est = math.ceil(1.5 * float(budget) * int(max_pages) / max(1, pps))
    p2 = 1 << max(0, (max(1, est) - 1).bit_length())
    return int(min(hard_cap, MAX_SPLIT, max(16, p2)))


def ensure_stage_b_buffers(st, device, split: int) -> None:
    """Allocate the split-K partials on the state once (outside any graph)."""
    if getattr(st, "m_part", None) is not None:
        return
    split = int(min(split, MAX_SPLIT))
    R, n_kv, G, D = st.max_reqs, st.n_kv, st.G, st.D
    st.split = split
    st.m_part = torch.empty(R, n_kv, split, G, device=device, dtype=torch.float32)
    st.l_part = torch.empty(R, n_kv, split, G, device=device, dtype=torch.float32)
    st.acc_part = torch.empty(R, n_kv, split, G, D, device=device, dtype=torch.float32)
    # arrival counts of the fused decode; every call leaves them at zero
    st.dec_counters = torch.zeros(R, n_kv, COUNTER_STRIDE, device=device, dtype=torch.int32)


def _launch_split(stream, q, kv, block_table, seq_lens, page_table, cnt, parts, n_req: int, G: int, split: int,
                  pps_min: int, max_cnt: int, scale: float, tier_src=None) -> None:
    """The split kernel from addresses and strides alone.  kv: (K address, V
    address, K strides, V strides, (num_blocks, page, n_kv, d)); cnt: (page_cnt
    address, request stride); parts: the addresses of m, l and acc; tier_src:
    the DRAM tier's source select, or None."""
    kp, vp, ks, vs, (NB, page, n_kv, d) = kv
    q_sr, q_sh = q.stride()[:2]
    pt_sr, pt_sh, _ = page_table.stride()
    lib = _lib.load()
    fn, tail = (lib.locks_decode_splitk, (stream,)) if tier_src is None else \
        (lib.locks_decode_splitk_tier, (ctypes.addressof(tier_src), stream))
    _lib.check(fn(
        q.data_ptr(), q_sr, q_sh, kp, *ks, vp, *vs, NB, block_table.data_ptr(), block_table.stride(0),
        block_table.shape[1], page_table.data_ptr(), pt_sr, pt_sh, page_table.shape[2], *cnt, seq_lens.data_ptr(),
        *parts, n_req, n_kv, G, d, page, split, pps_min, max_cnt, scale, *tail), "decode_splitk")


def _launch_merge(stream, parts, cnt, pt_cols: int, out, n_req: int, n_kv: int, G: int, d: int, split: int,
                  pps_min: int, max_cnt: int) -> None:
    """The merge of _launch_split's partials."""
    o_sr, o_sh, _ = out.stride()
    _lib.check(_lib.load().locks_decode_merge(
        *parts, *cnt, pt_cols, out.data_ptr(), o_sr, o_sh, 1 if out.dtype == torch.float32 else 0, n_req, n_kv, G, d,
        split, pps_min, max_cnt, stream), "decode_merge")


def _view_args(k, v):
    """_launch_split's kv of explicit (num_blocks, page, n_kv, d) views."""
    return k.data_ptr(), v.data_ptr(), k.stride()[:3], v.stride()[:3], tuple(k.shape)


def _ptrs(*tensors):
    return tuple(t.data_ptr() for t in tensors)


def _check_tier(ts, dims) -> None:
    NB, page, n_kv, d = dims
    if (ts.n_kv, ts.page, ts.head_dim, ts.num_blocks) != (n_kv, page, d, NB) \
            or not 0 <= ts.layer < ts.num_layers:
        raise ValueError(f"tier laid out for n_kv {ts.n_kv} / page {ts.page} / head_dim {ts.head_dim} / "
                         f"{ts.num_blocks} blocks, layer {ts.layer} of {ts.num_layers}; the cache is "
                         f"n_kv {n_kv} / page {page} / head_dim {d} / {NB} blocks")


def decode_splitk(q, k, v, block_table, seq_lens, page_table, page_cnt, m_part, l_part,
                  acc_part, *, n_req: int, G: int, split: int, pps_min: int,
                  scale: float, max_cnt: int = 0) -> None:
    """Launch the split kernel on explicit tensors.  k, v: (NB, page, n_kv, d)
    views; page_table (R, n_kv, MP) i32; page_cnt (R, n_kv) i32."""
    _launch_split(_lib.stream_ptr(q.device), q, _view_args(k, v), block_table, seq_lens, page_table,
                  (page_cnt.data_ptr(), page_cnt.stride(0)), _ptrs(m_part, l_part, acc_part), int(n_req), int(G),
                  int(split), int(pps_min), int(max_cnt), float(scale))


def decode_splitk_tier(q, k, v, block_table, seq_lens, page_table, page_cnt, m_part, l_part,
                       acc_part, tier_src, *, n_req: int, G: int, split: int, pps_min: int,
                       scale: float, max_cnt: int = 0) -> None:
    """The split kernel with V (and, for mem-kv, K) from the DRAM tier
    (``locks.tier.TierVSource.tier_src()``; attention/decode_cuda.py:178-222).
    k, v: (NB, page, n_kv, d) views of the paged cache; v is never read and
    may be any view of k's shape when the cache holds no V half."""
    _check_tier(tier_src, k.shape)
    _launch_split(_lib.stream_ptr(q.device), q, _view_args(k, v), block_table, seq_lens, page_table,
                  (page_cnt.data_ptr(), page_cnt.stride(0)), _ptrs(m_part, l_part, acc_part), int(n_req), int(G),
                  int(split), int(pps_min), int(max_cnt), float(scale), tier_src)


def _check_out(out) -> None:
    """The kernels write 4-element runs along the last dim of ``out``."""
    if out.dtype not in (torch.bfloat16, torch.float32):
        raise TypeError(f"out must be bf16 or fp32, got {out.dtype}")
    if out.dim() != 3 or out.stride(-1) != 1:
        raise TypeError(f"out must be (n_req, heads, d) with a contiguous last dim, got shape "
                        f"{tuple(out.shape)} strides {tuple(out.stride())}")


def decode_fused(q, k, v, block_table, seq_lens, page_table, page_cnt, m_part, l_part,
                 acc_part, counters, out, *, n_req: int, G: int, split: int, pps_min: int,
                 scale: float, max_cnt: int = 0) -> None:
    """Split kernel whose last-arriving split of each (request, kv head) row
    merges the row into ``out`` (one launch).  ``counters`` (R, n_kv,
    COUNTER_STRIDE) i32 must be zero on the first call; each call leaves it
    zero."""
    if counters.numel() < int(n_req) * k.shape[2] * COUNTER_STRIDE:
        raise ValueError(f"counters needs n_req * n_kv * {COUNTER_STRIDE} int32 entries")
    _check_out(out)
    NB, page, n_kv, d = k.shape
    lib = _lib.load()
    _lib.check(lib.locks_decode_fused(
        _lib.ptr(q), q.stride(0), q.stride(1),
        _lib.ptr(k), k.stride(0), k.stride(1), k.stride(2),
        _lib.ptr(v), v.stride(0), v.stride(1), v.stride(2), int(NB),
        _lib.ptr(block_table), block_table.stride(0), int(block_table.shape[1]),
        _lib.ptr(page_table), page_table.stride(0), page_table.stride(1),
        int(page_table.shape[2]), _lib.ptr(page_cnt), page_cnt.stride(0), _lib.ptr(seq_lens),
        _lib.ptr(m_part), _lib.ptr(l_part), _lib.ptr(acc_part), _lib.ptr(counters),
        _lib.ptr(out), out.stride(0), out.stride(1), 1 if out.dtype == torch.float32 else 0,
        int(n_req), int(n_kv), int(G), int(d), int(page), int(split), int(pps_min),
        int(max_cnt), float(scale), _lib.stream_ptr(q.device)), "decode_fused")


def decode_fused_noalloc(q, k, v, block_table, seq_lens, page_table, page_cnt, out, *,
                         n_req: int, G: int, split: int, pps_min: int, scale: float,
                         max_cnt: int = 0) -> None:
    """decode_fused with its split partials and arrival counters in the
    library's fixed per-GPU scratch (LOCKS_NOALLOC_SCRATCH_BYTES): no buffer
    arguments, nothing allocated.  Calls overlapping on one GPU race."""
    _check_out(out)
    NB, page, n_kv, d = k.shape
    lib = _lib.load()
    _lib.check(lib.locks_decode_fused_noalloc(
        _lib.ptr(q), q.stride(0), q.stride(1),
        _lib.ptr(k), k.stride(0), k.stride(1), k.stride(2),
        _lib.ptr(v), v.stride(0), v.stride(1), v.stride(2), int(NB),
        _lib.ptr(block_table), block_table.stride(0), int(block_table.shape[1]),
        _lib.ptr(page_table), page_table.stride(0), page_table.stride(1),
        int(page_table.shape[2]), _lib.ptr(page_cnt), page_cnt.stride(0), _lib.ptr(seq_lens),
        _lib.ptr(out), out.stride(0), out.stride(1), 1 if out.dtype == torch.float32 else 0,
        int(n_req), int(n_kv), int(G), int(d), int(page), int(split), int(pps_min),
        int(max_cnt), float(scale), _lib.stream_ptr(q.device)), "decode_fused_noalloc")


def decode_merge(m_part, l_part, acc_part, page_cnt, out, *, n_req: int, n_kv: int, G: int,
                 split: int, pps_min: int, pt_cols: int, max_cnt: int = 0) -> None:
    """LSE merge of the split partials into ``out``; ``pt_cols`` is the page
    table width the split kernel was given (page_cnt is clamped to it)."""
    _check_out(out)
    _launch_merge(_lib.stream_ptr(out.device), _ptrs(m_part, l_part, acc_part),
                  (page_cnt.data_ptr(), page_cnt.stride(0)), int(pt_cols), out, int(n_req), int(n_kv), int(G),
                  acc_part.shape[-1], int(split), int(pps_min), int(max_cnt))


def decode_dense(q, k, v, block_table, seq_lens, m_part, l_part, acc_part, out, *, n_req: int,
                 G: int, split: int, scale: float) -> None:
    """Dense full-KV decode over every page of each row (the comparator of
    the sparse step): split partials in (R, n_kv, split, G[, d]) buffers,
    then a per-head merge into ``out``."""
    _check_out(out)
    NB, page, n_kv, d = k.shape
    lib = _lib.load()
    _lib.check(lib.locks_decode_dense(
        _lib.ptr(q), q.stride(0), q.stride(1),
        _lib.ptr(k), k.stride(0), k.stride(1), k.stride(2),
        _lib.ptr(v), v.stride(0), v.stride(1), v.stride(2), int(NB),
        _lib.ptr(block_table), block_table.stride(0), int(block_table.shape[1]),
        _lib.ptr(seq_lens), _lib.ptr(m_part), _lib.ptr(l_part), _lib.ptr(acc_part),
        _lib.ptr(out), out.stride(0), out.stride(1), 1 if out.dtype == torch.float32 else 0,
        int(n_req), int(n_kv), int(G), int(d), int(page), int(split), float(scale),
        _lib.stream_ptr(q.device)), "decode_dense")


def sparse_paged_decode_batched(q, kv_cache, block_table, seq_lens, st, out,
                                vsource=None, *, scale: float = None) -> None:
    """Batched Stage B (decode.py:328-387): the split kernel + the
    head-parallel merge, or (FUSED_MERGE) one launch whose last split per row
    merges it."""
    if scale is None:
        scale = st.scale
    n_req = seq_lens.shape[0]
    pps = _pps_min(n_req, st.n_kv)
    mc = page_cnt_bound(st)
    source = 0 if vsource is None else vsource.SRC_ID
    if source not in (0, 1):
        raise NotImplementedError(f"V source {source} is not built (0 = resident, 1 = DRAM tier)")
    if FUSED_MERGE and source == 0:
        k, _ = _split_kv(kv_cache)
        v = (ResidentVSource(kv_cache) if vsource is None else vsource).args()[0]
        decode_fused(q, k, v, block_table, seq_lens, st.page_table, st.page_cnt, st.m_part,
                     st.l_part, st.acc_part, st.dec_counters, out, n_req=n_req, G=st.G,
                     split=st.split, pps_min=pps, scale=scale, max_cnt=mc)
        return
    # two launches, from addresses and strides alone (with views and per-stage
    # argument lists 24 -> 13.5 us of host time a layer)
    _check_out(out)
    kp, vp, ks, dims = _kv_args(kv_cache)
    vs, tier_src = ks, None
    if source == 1:
        # DRAM tier (decode_cuda.py:1301-1314): the tier's source select; V is
        # not read from the cache
        tier_src = vsource.tier_src()
        _check_tier(tier_src, dims)
        vp = kp if vp is None else vp
    elif vsource is not None:
        v = vsource.args()[0]
        vp, vs = v.data_ptr(), v.stride()[:3]
    elif vp is None:
        raise ValueError(_NO_V)
    stream, pt, G, split = _lib.stream_ptr(q.device), st.page_table, int(st.G), int(st.split)
    cnt = (st.page_cnt.data_ptr(), st.page_cnt.stride(0))
    acc = st.acc_part
    parts = (st.m_part.data_ptr(), st.l_part.data_ptr(), acc.data_ptr())
    _launch_split(stream, q, (kp, vp, ks, vs, dims), block_table, seq_lens, pt, cnt, parts, n_req, G, split, pps, mc,
                  float(scale), tier_src)
    _launch_merge(stream, parts, cnt, pt.shape[2], out, n_req, int(st.n_kv), G, acc.shape[-1], split, pps, mc)


def page_cnt_bound(st) -> int:
    """Upper bound of any row's page_cnt under the state's budget: b_max
    selected pages plus the sink and window pages (a keep-all row has at most
    sink + 1 + window pages, and b >= 1).  Sizes the decode grid."""
    return int(st.b_max) + int(st.sink_pages) + int(st.window_pages)
