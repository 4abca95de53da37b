"""Tensor-level wrappers over the C ABI: allocate outputs with torch, pass raw pointers.

Everything here runs on the GPU through libhqmq_amd.so; there is no CPU path.
"""
from __future__ import annotations

import ctypes as C
from typing import Optional

import torch

from . import _lib as L


def _dt(t: torch.Tensor) -> int:
    try:
        return L.DT_CODE[t.dtype]
    except KeyError:
        raise L.HqmqError(f"unsupported dtype {t.dtype}; expected float32, float16 or bfloat16") from None


def build_joint(raw_hs4: torch.Tensor, dtype: torch.dtype):
    """(H, S, 4) fp32 raw secondaries on the GPU -> (joint (H, 24S, 4) in dtype, slack (H,) fp32).
    The table's cell lists for the quantize kernels (see include/hqmq_amd.h) are built along and travel as an attribute
    of `slack`; a slack tensor without it quantizes through the scan over the secondaries, with the same results."""
    L.require_gpu(raw_hs4, "raw")
    raw = raw_hs4.detach().to(torch.float32).contiguous()
    H, S, _ = raw.shape
    joint = torch.empty(H, 24 * S, 4, dtype=dtype, device=raw.device)
    slack = torch.empty(H, dtype=torch.float32, device=raw.device)
    with torch.cuda.device(raw.device):
        L.check(L.lib().hqmq_build_joint(L.ptr(raw), C.c_int(H), C.c_int(S), C.c_int(L.DT_CODE[dtype]), L.ptr(joint),
                                         L.ptr(slack), L.stream_ptr(raw.device)), "hqmq_build_joint")
        nbytes, kept = (int(f(C.c_int(H), C.c_int(S), C.c_int(L.DT_CODE[dtype])))
                        for f in (L.lib().hqmq_search_grid_bytes, L.lib().hqmq_search_grid_kept_bytes))
        if nbytes:
            grid = torch.empty(nbytes, dtype=torch.uint8, device=raw.device)
            L.check(L.lib().hqmq_build_search_grid(L.ptr(joint), C.c_int(H), C.c_int(S), C.c_int(L.DT_CODE[dtype]),
                                                   L.ptr(grid), L.i64(nbytes), L.stream_ptr(raw.device)), "hqmq_build_search_grid")
            slack.hqmq_grid = grid[:kept].clone()            # behind it: scratch memory of the build
    return joint, slack


def _book(joint: torch.Tensor, slack: Optional[torch.Tensor], radius_bits: int, n: int):
    """A QuantizeArgs with everything a codebook fixes, kept with `slack` from call to call, and the address of the cell
    lists."""
    book = getattr(getattr(slack, "hqmq_book", None), "value", None)
    if book is not None and book[0] is joint and book[1] == joint.data_ptr() and book[2] == (radius_bits, n):
        return book[3], book[4]
    a = L.QuantizeArgs()
    a.dtype, a.H, a.n_chunks = _dt(joint), joint.shape[0], n
    a.joint, a.slack = L.addr(joint), L.addr(slack)
    a.secondary_size, a.radius_bits = joint.shape[1] // 24, radius_bits
    grid = getattr(slack, "hqmq_grid", None)
    if grid is not None and grid.numel() != L.lib().hqmq_search_grid_kept_bytes(C.c_int(a.H), C.c_int(a.secondary_size), C.c_int(a.dtype)):
        grid = None                 # lists of another library version (loaded from a file): the scan gives the same codes
    grid = L.addr(grid)
    if slack is not None:
        slack.hqmq_book = L.Kept((joint, joint.data_ptr(), (radius_bits, n), a, grid))
    a.address = C.addressof(a)
    return a, grid


def _check_joint(x: torch.Tensor, joint: torch.Tensor) -> None:
    if joint.dtype != x.dtype or joint.shape[0] != x.shape[1] or not joint.is_contiguous():
        raise ValueError("joint must be a contiguous (H, 24S, 4) table in the dtype of x")


def _strided_x(x: torch.Tensor):
    if x.dim() != 4:
        raise ValueError(f"expected (B, H, T, d_head), got {tuple(x.shape)}")
    if x.shape[-1] > 1 and x.stride(-1) != 1:
        x = x.contiguous()
    return x


def quantize(x: torch.Tensor, joint: torch.Tensor, slack: Optional[torch.Tensor], radius_bits: int, *,
             want_codes: bool = True, want_dense: bool = False, thr: Optional[torch.Tensor] = None,
             want_mask: bool = False, cache=None, t_off: int = 0, pos: Optional[torch.Tensor] = None,
             algo: int = 0, stats: Optional[torch.Tensor] = None) -> dict:
    """Run the quantize kernel on x (B, H, T, d_h).

    Returns a dict with the requested outputs: idx/rq (int32), r_max (dtype of x),
    out (fake-quant tensor), mask (bool).  `cache` is a PackedTensor whose rows
    [t_off, t_off + T) (shifted by pos[b] per sequence) receive the packed codes.
    """
    L.require_gpu(x, "x")
    d_h = x.shape[-1]
    if d_h % 4 != 0:
        raise ValueError(f"d_head={d_h} not divisible by 4")
    n = d_h // 4
    tmpl, grid = _book(joint, slack, radius_bits, n)
    if want_codes and not want_dense and cache is None and stats is None and algo == 0:
        idx, rq, r_max, mask = L.tensors(L.native().codes(x, joint, tmpl.address, grid, thr, want_mask), "hqmq_quantize_grid")
        out = {"idx": idx, "rq": rq, "r_max": r_max}
        if mask is not None:
            out["mask"] = mask
        return out
    x = _strided_x(x)
    B, H, T, _ = x.shape
    _check_joint(x, joint)
    dev = x.device
    a = L.QuantizeArgs.from_buffer_copy(tmpl)
    a.x = x.data_ptr()
    a.x_stride_b, a.x_stride_h, a.x_stride_t, _ = x.stride()
    a.B, a.T, a.algo = B, T, algo
    out = {}
    if want_codes:
        out["idx"], out["rq"] = x.new_empty((B, H, T, n), dtype=torch.int32), x.new_empty((B, H, T, n), dtype=torch.int32)
        out["r_max"] = x.new_empty((B, H, T))
        a.idx_out, a.rq_out, a.rmax_out = out["idx"].data_ptr(), out["rq"].data_ptr(), out["r_max"].data_ptr()
    if want_dense:
        out["out"] = x.new_empty((B, H, T, d_h))
        a.dense_out = out["out"].data_ptr()
    if thr is not None:
        thr = thr.to(x.dtype).contiguous()
        a.thr = thr.data_ptr()
        if want_mask:
            out["mask"] = x.new_empty((B, H, T, n), dtype=torch.bool)        # one byte per chunk, 0 or 1
            a.mask_out = out["mask"].data_ptr()
    if cache is not None:
        a.main_plane, a.aux_plane = L.addr(cache.main), L.addr(cache.aux)
        a.scale_plane = L.addr(cache.scale)
        a.flag_plane = L.addr(cache.flags) if thr is not None else 0
        a.t_cap, a.t_off = cache.t_cap, t_off
        a.main_bits, a.aux_bits = cache.main_bits, cache.aux_bits
        a.scale_max_bits = L.addr(cache.scale_max)
        if pos is not None:
            pos = pos.to(device=dev, dtype=torch.int32).contiguous()
            a.pos = pos.data_ptr()
    a.stats = L.addr(stats)
    if T > 0:
        L.call(L.lib().hqmq_quantize_grid, "hqmq_quantize_grid", dev.index, C.addressof(a), grid)
    return out


_WS = {}
_WS_MOST = 256

# torch.quantile refuses more than 2^24 elements along the reduced dimension ("quantile() input tensor is too large"),
# which bounds the chunks per head of one Med-C call of the reference (src/quantizers/outlier_aware.py:68).  The
# radix select here has no such bound; check_quantile_limit(..., strict=True) mirrors the reference's refusal.
QUANTILE_LIMIT = 1 << 24


def check_quantile_limit(chunks_per_head: int, strict: bool) -> bool:
    """True when a Med-C call of this size is within torch.quantile's limit.  Beyond it the reference raises; with
    strict=True so does this function (same exception type and message), otherwise the call is an extension."""
    ok = chunks_per_head <= QUANTILE_LIMIT
    if not ok and strict:
        raise RuntimeError("quantile() input tensor is too large")
    return ok


def _workspace(nbytes: int, device, tag: str) -> torch.Tensor:
    """A cached scratch buffer of at least nbytes (grown on demand, reused across calls on the same stream; any content).
    Under stream capture a buffer of the call's own: torch takes it from the graph's memory, which later calls of the capture
    use again in stream order, no call outside it does, and the graph gives back when it goes."""
    if torch.cuda.is_current_stream_capturing():
        return torch.empty(nbytes, dtype=torch.uint8, device=device)
    index = device.index
    key = (tag, index, L.raw_stream(index))                          # calls on different streams may overlap
    buf = _WS.get(key)
    if buf is None or buf.numel() < nbytes:
        if len(_WS) >= _WS_MOST:                                     # streams that are gone: their buffers go back to torch
            _WS.clear()
        buf = torch.empty(max(nbytes, 1 << 16), dtype=torch.uint8, device=device)
        _WS[key] = buf
    return buf


def med3x_threshold(x: torch.Tensor, mult: float = 3.0, want_count: bool = True, strict_quantile_limit: bool = False):
    """Per-head (median fp32, threshold in x.dtype, #chunks above threshold int32) over the whole call.
    strict_quantile_limit: raise as the reference does when a head has more than 2^24 chunks in this call."""
    L.require_gpu(x, "x")
    if x.dim() != 4:
        raise ValueError(f"expected (B, H, T, d_head), got {tuple(x.shape)}")
    if strict_quantile_limit:
        check_quantile_limit(x.shape[0] * x.shape[2] * (x.shape[3] // 4), True)
    return L.tensors(L.native().med3x(x, mult, _med_workspace(x, "med3x"), want_count), "hqmq_med3x_threshold")


def _med_workspace(x: torch.Tensor, tag: str) -> torch.Tensor:
    H, f32 = x.shape[1], x.dtype == torch.float32
    key = (H, f32)
    nbytes = _MED_BYTES.get(key)
    if nbytes is None:
        nbytes = _MED_BYTES[key] = int(L.lib().hqmq_med3x_workspace_best_bytes(C.c_int(H), C.c_int(_dt(x))))
    return _workspace(nbytes + 12 * H + 16, x.device, tag)        # behind it: room for a median and a threshold nobody asked for


_MED_BYTES = {}


def fake_quant(x: torch.Tensor, joint: torch.Tensor, slack: torch.Tensor, radius_bits: int, median_mult: Optional[float] = None):
    """The fake-quant tensor of x (B, H, T, d_h), with Med-C extraction when median_mult is given: what med3x_threshold
    and quantize(want_dense=True) give, without tensors for the statistics in between.  Returns (out, flagged chunks
    per head or None)."""
    L.require_gpu(x, "x")
    if x.dim() != 4:
        raise ValueError(f"expected (B, H, T, d_head), got {tuple(x.shape)}")
    tmpl, grid = _book(joint, slack, radius_bits, x.shape[3] // 4)
    ws = None if median_mult is None else _med_workspace(x, "med3x")
    return L.tensors(L.native().fake(x, joint, tmpl.address, grid, median_mult, ws),
                     "hqmq_quantize_grid" if median_mult is None else "hqmq_quantize_med3x_grid")


def outlier_mask(x: torch.Tensor, thr: torch.Tensor) -> torch.Tensor:
    """Boolean (B, H, T, n) mask of chunks whose norm exceeds the per-head threshold."""
    L.require_gpu(x, "x")
    x = _strided_x(x)
    B, H, T, d_h = x.shape
    thr = thr.to(x.dtype).contiguous()
    mask = torch.empty(B, H, T, d_h // 4, dtype=torch.uint8, device=x.device)
    with torch.cuda.device(x.device):
        L.check(L.lib().hqmq_outlier_mask(
            L.ptr(x), L.i64(x.stride(0)), L.i64(x.stride(1)), L.i64(x.stride(2)), C.c_int(_dt(x)), C.c_int(B), C.c_int(H),
            C.c_int(T), C.c_int(d_h // 4), L.ptr(thr), L.ptr(mask), L.stream_ptr(x.device)), "hqmq_outlier_mask")
    return mask.bool()


def outlier_compact(x: torch.Tensor, cache, t_off: int = 0, pos: Optional[torch.Tensor] = None) -> None:
    """Append the flagged chunks of x (rows t_off.. of the cache) to the cache's sideband."""
    x = _strided_x(x)
    B, H, T, d_h = x.shape
    dev = x.device
    if pos is not None:
        pos = pos.to(device=dev, dtype=torch.int32).contiguous()
    rows = L.PackedRows()      # the planes of the same rows: a chunk that finds the sideband full goes back to a plain chunk
    rows.main_plane, rows.aux_plane, rows.scale_plane = L.ptr(cache.main), L.ptr(cache.aux), L.ptr(cache.scale)
    rows.idx_bits, rows.main_bits, rows.aux_bits, rows.qmax = cache.idx_bits, cache.main_bits, cache.aux_bits, cache.qmax
    with torch.cuda.device(dev):
        L.check(L.lib().hqmq_outlier_compact(
            L.ptr(x), L.i64(x.stride(0)), L.i64(x.stride(1)), L.i64(x.stride(2)), C.c_int(_dt(x)), C.c_int(B), C.c_int(H),
            C.c_int(T), C.c_int(d_h // 4), L.ptr(cache.flags), L.i64(cache.t_cap), C.c_int(t_off), L.ptr(pos),
            L.ptr(cache.sideband), L.i64(cache.sb_cap), L.ptr(cache.sb_tile_off), L.ptr(cache.sb_count),
            L.ptr(cache.sb_overflow), L.ptr(cache.sb_coord), C.byref(rows), L.stream_ptr(dev)), "hqmq_outlier_compact")


def crop(caches, lengths) -> None:
    """Outlier lists, tile offsets and flags of the PackedTensors (one, or K and V of equal shape) back to the state after
    the first `lengths` rows: an int for all sequences or an int32 tensor [B] on the caches' device."""
    c = caches[0]
    a = L.CropArgs()
    for i, t in enumerate(caches):
        a.flag_plane[i], a.sb_tile_off[i], a.sb_count[i] = t.flags.data_ptr(), t.sb_tile_off.data_ptr(), t.sb_count.data_ptr()
    a.count, a.B, a.H, a.t_cap, a.n_chunks = len(caches), c.B, c.H, c.t_cap, c.n
    if isinstance(lengths, int):
        a.length = max(0, min(lengths, c.t_cap))
    else:
        if lengths.numel() != c.B or lengths.dtype is not torch.int32 or lengths.device != c.flags.device or not lengths.is_contiguous():
            raise L.HqmqError(f"lengths must be {c.B} contiguous int32 on the caches' device")       # the kernel reads all B of them
        a.lengths = lengths.data_ptr()
    L.call(L.lib().hqmq_crop, "hqmq_crop", c.flags.device.index, C.addressof(a))


def append_kv(k: torch.Tensor, v: torch.Tensor, k_cache, v_cache, k_joint, k_slack, v_joint, v_slack, radius_bits: int, *,
              t_off: int = 0, pos: Optional[torch.Tensor] = None, median_mult: Optional[float] = None):
    """Quantize the new rows k, v (B, H, T, d_h) into rows t_off.. of the two PackedTensors (shifted by pos[b]),
    with Med-C extraction into their sidebands when median_mult is given.  Same results as med3x_threshold,
    quantize and outlier_compact for K and then for V; K and V of equal shape share every launch.
    Returns (k_count, v_count), the flagged chunks per head (int32 [H]) or (None, None)."""
    L.require_gpu(k, "k")
    L.require_gpu(v, "v")
    if k.shape[2] == 0 and v.shape[2] == 0:        # an empty tensor has no address to pass
        return None, None
    ak, grid_k, ws_k = _append_block(k, k_cache, k_joint, k_slack, radius_bits, median_mult, "med3x_k")
    av, grid_v, ws_v = _append_block(v, v_cache, v_joint, v_slack, radius_bits, median_mult, "med3x_v")
    return L.tensors(L.native().append(k, v, ak.address, av.address, grid_k, grid_v, t_off, pos, median_mult, ws_k, ws_v), "hqmq_append_kv_grid")


def _append_block(x, cache, joint, slack, radius_bits, median_mult, tag):
    """What a cache and its codebook fix of one tensor's append, filled in once (the library's caller copies it: several threads may
    append to one cache on streams of their own), the cell lists, the workspace of the call's median."""
    if x.dim() != 4:
        raise ValueError(f"expected (B, H, T, d_head), got {tuple(x.shape)}")
    _, H, T, d_h = x.shape
    med = median_mult is not None and T > 0
    tmpl = cache._append_template
    if tmpl is None or tmpl[0] is not joint or tmpl[1] is not slack or tmpl[2] != (joint.data_ptr(), cache.main.data_ptr(), radius_bits, d_h, med):
        if d_h % 4 != 0:
            raise ValueError(f"d_head={d_h} not divisible by 4")
        _check_joint(x, joint)
        book, grid = _book(joint, slack, radius_bits, d_h // 4)
        a = L.AppendArgs()
        C.memmove(C.addressof(a), C.addressof(book), C.sizeof(book))       # q is the first member
        q = a.q
        q.main_plane, q.aux_plane, q.scale_plane = L.addr(cache.main), L.addr(cache.aux), L.addr(cache.scale)
        q.t_cap, q.main_bits, q.aux_bits = cache.t_cap, cache.main_bits, cache.aux_bits
        q.scale_max_bits = L.addr(cache.scale_max)
        if med:
            q.flag_plane = L.addr(cache.flags)
            a.sideband, a.sb_cap = L.addr(cache.sideband), cache.sb_cap
            a.sb_tile_off, a.sb_count = L.addr(cache.sb_tile_off), L.addr(cache.sb_count)
            a.overflow, a.sb_coord = L.addr(cache.sb_overflow), L.addr(cache.sb_coord)
        a.address = C.addressof(a)
        tmpl = cache._append_template = (joint, slack, (joint.data_ptr(), cache.main.data_ptr(), radius_bits, d_h, med), a, grid)
    elif joint.dtype != x.dtype or joint.shape[0] != H:
        _check_joint(x, joint)
    return tmpl[3], tmpl[4], _med_workspace(x, tag) if med else None


def _i32(t: torch.Tensor) -> torch.Tensor:
    t = t if t.dtype == torch.int32 else t.to(torch.int32)
    return t if t.stride(-1) == 1 else t.contiguous()


def dequant(idx, radius_q, radius_scale, joint, r_qmax: int) -> torch.Tensor:
    """Unpacked codes -> dense (B, H, T, 4n) in joint.dtype (rounding of the reference's torch decode)."""
    L.require_gpu(idx, "idx")
    _dt(joint)
    return L.tensors(L.native().dequant(idx, radius_q, radius_scale, joint, r_qmax), "hqmq_dequant")


def pack_codes(idx, radius_q, cache, T: Optional[int] = None) -> None:
    """Write unpacked int codes into rows [0, T) of a PackedTensor's code planes."""
    idx, rq = _i32(idx), _i32(radius_q)
    B, H, Ti, n = idx.shape
    T = Ti if T is None else T
    with torch.cuda.device(idx.device):
        L.check(L.lib().hqmq_pack_codes(
            L.ptr(idx), L.i64(idx.stride(0)), L.i64(idx.stride(1)), L.i64(idx.stride(2)),
            L.ptr(rq), L.i64(rq.stride(0)), L.i64(rq.stride(1)), L.i64(rq.stride(2)),
            C.c_int(B), C.c_int(H), C.c_int(T), C.c_int(n), C.c_int(cache.idx_bits), C.c_int(cache.main_bits),
            C.c_int(cache.aux_bits), L.ptr(cache.main), L.ptr(cache.aux), L.i64(cache.t_cap), L.stream_ptr(idx.device)),
            "hqmq_pack_codes")


def dequant_packed(cache, T: Optional[int] = None, mode: int = 0) -> torch.Tensor:
    """Packed cache -> dense (B, H, T, d_h); mode 0 = attention rounding, 1 = quantizer fake-quant rounding."""
    T = cache.length if T is None else T
    out = torch.empty(cache.B, cache.H, T, cache.d_head, dtype=cache.dtype, device=cache.device)
    s = cache.c_struct()
    with torch.cuda.device(cache.device):
        L.check(L.lib().hqmq_dequant_packed(
            C.byref(s), C.c_int(L.DT_CODE[cache.dtype]), C.c_int(cache.B), C.c_int(cache.H), C.c_int(T), C.c_int(cache.n),
            L.i64(cache.t_cap), C.c_int(cache.idx_bits), C.c_int(cache.main_bits), C.c_int(cache.aux_bits),
            C.c_int(cache.qmax), C.c_int(mode), L.ptr(out), L.stream_ptr(cache.device)), "hqmq_dequant_packed")
    return out


def pick_splits(B: int, H_q: int, H_kv: int, T_q: int, T_kv: int, ragged: bool = False) -> int:
    key = (B, H_q, H_kv, T_q, (T_kv + 63) // 64, ragged)               # the library's choice changes at multiples of 64 tokens only
    n = _SPLITS.get(key)
    if n is None:
        if len(_SPLITS) >= 4096:
            _SPLITS.clear()
        n = _SPLITS[key] = int(L.lib().hqmq_attn_pick_splits(C.c_int(B), C.c_int(H_q), C.c_int(H_kv), C.c_int(T_q), C.c_int(T_kv),
                                                             C.c_int(1 if ragged else 0)))
    return n


_SPLITS = {}


def longest_first(kv_lens: torch.Tensor) -> torch.Tensor:
    """The batch_order for a ragged batch: sequences sorted by length, longest first (int32, on kv_lens' device).
    It stays valid while all sequences grow in step, so a decode loop computes it once."""
    return torch.argsort(kv_lens, descending=True, stable=True).to(torch.int32)


def attn_fwd(Q: torch.Tensor, Kc, Vc, T_kv: int, *, kv_lens: Optional[torch.Tensor] = None,
             kv_starts: Optional[torch.Tensor] = None, batch_order: Optional[torch.Tensor] = None, causal: bool = False,
             causal_offset: int = 0, softmax_scale: Optional[float] = None, n_splits: int = 0,
             out: Optional[torch.Tensor] = None, skip_combine: bool = False,
             force_generic: bool = False, kernel_events: Optional[tuple] = None,
             static_scratch: bool = False, workspace: Optional[torch.Tensor] = None, fp8_table_storage: bool = False):
    """Fused attention of Q (B, H_q, T_q, d_h) over packed K/V (PackedTensor each).
    kernel_events: two raw hipEvent_t handles (ints) that receive the GPU timestamps of the begin and the end of
    the main attention kernel (profiling).
    static_scratch: call hqmq_attn_fwd_static, which keeps the split partials in the library's own device array
    instead of a torch workspace (pass `out` as well and the call allocates nothing on the device).
    fp8_table_storage: both joint tables hold float8 e4m3 numbers (PackedTensor.with_fp8_table) and the kernel may keep
    them as float8 in LDS; same results, see include/hqmq_amd.h.
    skip_combine: leave the split partials unmerged and return (O, partials, n_splits): the partials are in `workspace`
    if given, else in a buffer of their own (never the cached scratch that the next call on the stream overwrites);
    attn_combine(partials, O, n_splits) merges them."""
    if not Q.is_cuda:
        L.require_gpu(Q, "Q")
    shape, stride = Q.shape, Q.stride()
    if stride[-1] != 1:
        Q = Q.contiguous()
        stride = Q.stride()
    ks, vs = Kc.c_struct(), Vc.c_struct()
    plan = Kc._attn_plans.get((shape, stride))
    if plan is None or plan[0] is not ks or plan[1] is not vs or plan[2] is not Q.dtype:
        plan = _attn_plan(Q, Kc, Vc, ks, vs)
    for t, what in ((kv_starts, "kv_starts must hold one entry per sequence"), (batch_order, "batch_order must be a permutation of the sequences")):
        if t is not None and t.numel() != shape[0]:
            raise L.HqmqError(f"{what} ({shape[0]})")
    options = None
    if skip_combine or static_scratch or kernel_events or workspace is not None:
        start, stop = kernel_events or (0, 0)
        options = (skip_combine, static_scratch, workspace, start or 0, stop or 0)
    # (wide_range: V scales outside [2^-8, 2^15), the generic kernel guards the range)
    return L.tensors(L.native().attn(Q, plan[3].address, out, T_kv, kv_lens, kv_starts, batch_order, causal, causal_offset, softmax_scale, n_splits,
                                     force_generic, fp8_table_storage, Vc.wide_range, _workspace, options),
                     "hqmq_attn_fwd_static" if static_scratch else "hqmq_attn_fwd")


_FUSED = {}


def fused_unpacked(Q: torch.Tensor, k: tuple, v: tuple, r_qmax: int, *, kv_lens: Optional[torch.Tensor] = None, causal: bool = True,
                   causal_offset: int = 0, softmax_scale: Optional[float] = None, n_splits: int = 0) -> torch.Tensor:
    """Attention of Q over unpacked codes: k and v are (idx, radius_q, radius_scale, joint).  One launch packs both tensors into
    planes of this call, then the packed attention runs over them."""
    dt = Q.dtype
    idx, rq, _, joint = k
    idx_v, rq_v, _, joint_v = v
    for i, r in ((idx, rq), (idx_v, rq_v)):
        if r.shape != i.shape:
            raise L.HqmqError(f"radius codes {tuple(r.shape)} and indices {tuple(i.shape)} differ in shape")
    if idx_v.shape[0] != idx.shape[0] or idx_v.shape[1] != idx.shape[1] or idx_v.shape[3] != idx.shape[3] or Q.shape[0] != idx.shape[0]:
        raise L.HqmqError("K and V codes must have equal batch, head and chunk counts, Q the same batch")
    if Q.stride(-1) != 1:
        Q = Q.contiguous()
    key = (Q.shape, Q.stride(), idx.shape, idx_v.shape[2], joint.shape[1], joint_v.shape[1], r_qmax, dt)
    plan = _FUSED.get(key)
    if plan is None:
        if len(_FUSED) >= 256:                     # shapes that no longer come
            _FUSED.clear()
        plan = _FUSED[key] = _fused_plan(Q, idx, idx_v.shape[2], joint.shape[1], joint_v.shape[1], r_qmax)
    pack, a, nbytes = plan
    return L.tensors(L.native().fused(Q, *k, *v, pack.address, a.address, nbytes, kv_lens, causal, causal_offset, softmax_scale, n_splits),
                     "hqmq_attn_fwd")


def _fused_plan(Q: torch.Tensor, idx: torch.Tensor, T_v: int, K: int, K_v: int, r_qmax: int):
    """What the shapes fix of a fused_unpacked call: both argument blocks, with the planes' offsets in its buffer, and the bytes of
    the buffer."""
    B, H, T, n = idx.shape
    Hq, Tq = Q.shape[1], Q.shape[2]
    radius_bits = max(1, int(r_qmax).bit_length())
    if radius_bits > 8:
        raise L.HqmqError(f"r_qmax={r_qmax} needs more than 8 radius bits")
    # a table of K rows is addressed like one of ceil(K/24) secondaries; the radius field holds r_qmax
    ib, mb, ab = L.layout_bits(max(1, -(-max(K, K_v) // 24)), radius_bits)
    if mb == 12 and (n // 4) % 2:      # a lane's share of a 12-bit row must be whole bytes: use 16-bit codes
        mb, ab = 16, max(0, ib + radius_bits - 16)
    cap = (max(T, T_v, 1) + 63) // 64 * 64         # whole attention super-tiles
    sizes = [cap * B * H * ((n * mb + 7) // 8)] * 2 + [cap * B * H * Q.element_size()] * 2 + [cap * B * H * ((n * ab + 7) // 8)] * 2
    offsets, at = [], 0
    for size in sizes:
        offsets.append(at)
        at += (size + 255) // 256 * 256
    pack, a = L.PackArgs(), L.AttnArgs()
    for i, t in enumerate((T, T_v)):
        p = pack.side[i]
        p.T, p.main_plane, p.scale_plane, p.aux_plane = t, offsets[i], offsets[2 + i], offsets[4 + i]
    code = L.DT_CODE[Q.dtype]
    pack.dtype, pack.B, pack.H, pack.n_chunks, pack.t_cap = code, B, H, n, cap
    pack.idx_bits, pack.main_bits, pack.aux_bits = ib, mb, ab
    a.q_sb, a.q_sh, a.q_st = Q.stride(0), Q.stride(1), Q.stride(2)
    for t, rows in ((a.K, K), (a.V, K_v)):
        t.scale_sb, t.scale_sh, t.scale_st, t.K = H * cap, cap, 1, rows
    a.dtype, a.B, a.H_q, a.H_kv, a.T_q, a.T_kv, a.n_chunks, a.t_cap = code, B, Hq, H, Tq, T, n, cap
    a.idx_bits, a.main_bits, a.aux_bits, a.qmax = ib, mb, ab, int(r_qmax)
    a.softmax_scale = Q.shape[3] ** -0.5
    pack.address, a.address = C.addressof(pack), C.addressof(a)
    return pack, a, max(at, 256)


def _attn_plan(Q: torch.Tensor, Kc, Vc, ks, vs):
    """What a shape of Q and a pair of packed tensors fix of an attention call, kept with the K cache."""
    B, Hq, Tq, d_h = Q.shape
    if d_h != Kc.d_head or d_h != Vc.d_head:
        raise AssertionError(f"d_h={d_h} != n_chunks*4={Kc.d_head}")
    if Hq % Kc.H:
        raise AssertionError(f"H_q={Hq} must be divisible by H_kv={Kc.H}")
    if Q.dtype != Kc.dtype:
        raise L.HqmqError(f"Q dtype {Q.dtype} differs from the cache dtype {Kc.dtype}")
    a = L.AttnArgs()
    a.q_sb, a.q_sh, a.q_st = Q.stride(0), Q.stride(1), Q.stride(2)
    a.K, a.V = ks, vs
    a.dtype = L.DT_CODE[Q.dtype]
    a.B, a.H_q, a.H_kv, a.T_q, a.n_chunks = B, Hq, Kc.H, Tq, Kc.n
    a.t_cap = Kc.t_cap
    a.idx_bits, a.main_bits, a.aux_bits, a.qmax = Kc.idx_bits, Kc.main_bits, Kc.aux_bits, Kc.qmax
    a.softmax_scale = d_h ** -0.5
    plan = (ks, vs, Q.dtype, a)
    if len(Kc._attn_plans) >= 64:                  # shapes that no longer come
        Kc._attn_plans.clear()
    a.address = C.addressof(a)
    Kc._attn_plans[(Q.shape, Q.stride())] = plan
    return plan


def attn_combine(partials: Optional[torch.Tensor], O: torch.Tensor, n_splits: int) -> torch.Tensor:
    """Merge the split partials a skip_combine call left behind into O (B, H_q, T_q, d_h)."""
    if n_splits <= 1 or partials is None:
        return O
    B, Hq, Tq, d_h = O.shape
    with torch.cuda.device(O.device):
        L.check(L.lib().hqmq_attn_combine(L.ptr(partials), L.ptr(O), C.c_int(L.DT_CODE[O.dtype]), C.c_int(B), C.c_int(Hq),
                                          C.c_int(Tq), C.c_int(d_h), C.c_int(n_splits), L.i64(O.stride(0)), L.i64(O.stride(1)),
                                          L.i64(O.stride(2)), L.stream_ptr(O.device)), "hqmq_attn_combine")
    return O
