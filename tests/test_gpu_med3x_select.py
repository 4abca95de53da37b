"""Calls whose quantize launch works the Med3x threshold out for itself (16-bit types, more than 16384 chunks and up to 128 parts per head), against the
threshold's own calls, which take a launch for it: the same flags, counts and rows.  Packed rows in the same launch, at the edges of their
forms."""
import pytest
import torch

from tests.helpers import DT, kv_input

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _two_groups(x):
    """Half of the chunks a thousand times smaller: the two middle norms lie far apart, in different groups of bins."""
    x = x.reshape(-1, 4).clone()
    x[::2] *= 1e-3
    return x


@pytest.mark.parametrize("dn,S,b_r,shape,what", [
    ("fp16", 96, 4, (1, 2, 513, 128), "plain"), ("bf16", 24, 3, (3, 2, 700, 128), "plain"), ("fp16", 192, 6, (2, 1, 2100, 64), "two groups"),
    ("bf16", 192, 4, (1, 3, 1200, 64), "two groups"), ("bf16", 341, 4, (1, 1, 600, 128), "plain"), ("fp16", 341, 4, (1, 1, 600, 128), "two groups"),
    ("fp16", 24, 3, (1, 2, 520, 128), "nan"), ("bf16", 96, 4, (1, 2, 4100, 20), "plain"), ("fp16", 96, 4, (1, 1, 9000, 128), "equal"),
    ("bf16", 24, 3, (1, 9, 530, 128), "zero"),
    # parts per head around the lines of the selection: 32 and 33, 128 and 129
    ("fp16", 24, 3, (1, 3, 4096, 128), "plain"), ("bf16", 96, 4, (1, 3, 4100, 128), "two groups"),
    ("bf16", 24, 3, (1, 1, 16384, 128), "two groups"), ("fp16", 96, 4, (1, 1, 16400, 128), "two groups"), ("fp16", 24, 3, (1, 2, 16384, 128), "nan")])
def test_quantize_launch_selects_the_threshold(dn, S, b_r, shape, what):
    import hqmq
    from hqmq_amd import ops
    dt = DT[dn]
    B, H, T, d_h = shape
    assert B * T * (d_h // 4) > 16384
    x = kv_input(shape, torch.float32, seed=T, outlier_p=0.02)
    if what == "two groups":
        x = _two_groups(x).reshape(shape)
    elif what == "equal":
        x = torch.full(shape, 0.75)
        x[:, :, ::50] = 4.0
    elif what == "zero":
        x[:, 1:] = 0.0
    x = x.to(dt)
    if what == "nan":
        x[0, 1, 7, 5] = float("nan")
    x = x.to(DEV)
    q = hqmq.HQMQ(n_layers=1, n_heads=H, secondary_size=S, radius_bits=b_r, device=DEV)
    w = hqmq.with_outlier_extraction(q, C=3.0)
    for view in (x, x.transpose(1, 2).contiguous().transpose(1, 2)):
        med, thr, count = ops.med3x_threshold(view, 3.0)
        mask = ops.outlier_mask(view, thr).bool()
        assert torch.equal(count.long(), mask.sum(dim=(0, 2, 3)))
        plain = q.quantize_K(view, 0)
        want = torch.where(mask.repeat_interleave(4, -1), view, plain)
        joint, slack = q._joint_and_slack(0, 0, view)
        got, flagged = ops.fake_quant(view, joint, slack, b_r, 3.0)
        assert torch.equal(flagged, count) and torch.equal(got.view(torch.int16), want.view(torch.int16))
        assert torch.equal(w.quantize_K(view, 0).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("dn", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", [
    (4400, 2, 1, 16), (300, 2, 3, 76),          # a block's step goes over many sequences, not a whole number of them
    (1, 3, 4097, 20), (2, 1, 601, 120),         # rows that do not divide a block's lanes
    (3, 2, 11, 4400),                           # rows of more chunks than a block has lanes
    (1, 1, 129, 512), (1, 5, 513, 128),         # last blocks of a single step
    (1, 2, 4096, 128), (1, 2, 4100, 128), (1, 1, 16400, 128)])      # 32, 33 and 129 parts per head
def test_histograms_count_every_chunk_once(dn, shape):
    """Calls that count in one histogram per block (16-bit types, more than 16384 chunks per head), contiguous and with strides."""
    from hqmq_amd import ops
    from oracle import c_oracle as CO
    B, H, T, d_h = shape
    assert B * T * (d_h // 4) > 16384
    x = kv_input(shape, DT[dn], seed=T + d_h, outlier_p=0.03)
    want = CO.med3x(x, 3.0)
    for view in (x.to(DEV), x.transpose(1, 2).contiguous().to(DEV).transpose(1, 2)):
        med, thr, count = ops.med3x_threshold(view, 3.0)
        assert torch.equal(med.cpu(), want["median"]) and torch.equal(thr.cpu().view(torch.int16), want["threshold"].view(torch.int16))
        assert torch.equal(count.cpu().long(), want["mask"].sum(dim=(0, 2, 3)))


@pytest.mark.parametrize("dn,S,b_r,d_h,med", [
    ("fp16", 96, 4, 128, True), ("bf16", 24, 3, 128, True), ("bf16", 24, 3, 64, True), ("fp16", 192, 6, 128, True), ("fp16", 192, 6, 64, False),
    ("bf16", 192, 5, 128, True), ("fp16", 192, 4, 64, True), ("bf16", 24, 5, 128, False), ("fp16", 24, 4, 64, True)])
@pytest.mark.parametrize("T,t_off", [(33, 0), (515, 0), (600, 7), (1100, 64)])
def test_long_appends_write_the_rows_of_short_ones(dn, S, b_r, d_h, med, T, t_off):
    """Rows that neighbouring lanes put together (16 and 32 codes, 12 and 16 bits, one to three bits aside), with rows before and behind that
    must stay as they are, against the unpacked codes read back from the planes."""
    import hqmq
    from tests.helpers import unpack_planes
    dt = DT[dn]
    B, H, cap = 2, 3, T + t_off + 9
    q = hqmq.HQMQ(n_layers=1, n_heads=H, secondary_size=S, radius_bits=b_r, device=DEV)
    w = hqmq.with_outlier_extraction(q, C=3.0) if med else q
    k, v = (kv_input((B, H, T, d_h), dt, seed=T + i, outlier_p=0.02).to(DEV) for i in (0, 1))
    cache = w.new_cache(B, cap, d_h, dt, 0)
    planes = {(n, p): getattr(t, p) for n, t in (("K", cache.K), ("V", cache.V)) for p in ("main", "aux", "scale") if getattr(t, p) is not None}
    for p in planes.values():
        p.view(torch.uint8).fill_(0xA5)
    if t_off:
        w.append(cache, k[:, :, :t_off], v[:, :, :t_off], 0)
    before = {key: p.clone() for key, p in planes.items()}
    w.append(cache, k, v, 0)
    for t, x, encode in ((cache.K, k, w.encode_K), (cache.V, v, w.encode_V)):
        c = encode(x, 0)
        mask = c["mask"].bool() if med else torch.zeros_like(c["idx"]).bool()
        for b in range(B):
            idx, rq, flags = unpack_planes(t, b, t_off + T)
            assert torch.equal(idx[:, t_off:], c["idx"][b].long()) and torch.equal(rq[:, t_off:], c["rq"][b].long() * ~mask[b])
            assert not med or torch.equal(flags[:, t_off:], mask[b])
        assert torch.equal(t.scale[:, :, t_off:t_off + T].view(torch.int16), c["r_max"].reshape(B, H, T).view(torch.int16))
    for key, p in planes.items():
        assert torch.equal(p[:, :, :t_off], before[key][:, :, :t_off]) and torch.equal(p[:, :, t_off + T:], before[key][:, :, t_off + T:]), key


def _appended_through_the_c_abi(case, ks, vs, med, layout, dt, S, b_r, d_h, H):
    """hqmq_append_kv_grid with the workspaces laid out as `layout` says; [(x, quantizer, PackedTensor, median, thr, count or None)]."""
    import ctypes as C

    import hqmq
    from hqmq_amd import _lib as L, ops
    q = hqmq.with_outlier_extraction(hqmq.HQMQ(n_layers=1, n_heads=H, secondary_size=S, radius_bits=b_r, device=DEV), C=3.0)
    lib, code = L.lib(), ops._dt(ks)
    best = int(lib.hqmq_med3x_workspace_best_bytes(C.c_int(H), C.c_int(code)))
    least = int(lib.hqmq_med3x_workspace_bytes(C.c_int(H), C.c_int(code)))
    # (offset, bytes) of K's and V's workspace in one buffer
    spans = {"apart": ((0, best), (best, best)), "same": ((0, best), (0, best)), "overlap": ((0, best), (65536, best)),
             "overlap below": ((65536, best), (0, best)), "V's is small": ((0, best), (4096, least)), "K's is small": ((4096, least), (0, best)),
             "both small": ((0, least), (0, least))}[layout]
    room = torch.full((2 * best,), 0x5A, dtype=torch.uint8, device=DEV)
    cache = q.new_cache(ks.shape[0], max(ks.shape[2], vs.shape[2]), d_h, dt, 0)
    args, keep = [], []
    for i, (x, t) in enumerate(((ks, cache.K), (vs, cache.V))):
        joint, slack = q.inner._joint_and_slack(0, i, x)
        tmpl, grid, _ = ops._append_block(x, t, joint, slack, b_r, 3.0 if i in med else None, "c abi %d" % i)
        assert grid
        a = L.AppendArgs.from_buffer_copy(tmpl)
        a.q.x, a.q.B, a.q.T = x.data_ptr(), x.shape[0], x.shape[2]
        a.q.x_stride_b, a.q.x_stride_h, a.q.x_stride_t, _ = x.stride()
        median, thr, count = (torch.full((H,), -1, dtype=d, device=DEV) for d in (torch.float32, dt, torch.int32))
        if i in med:
            a.median_mult, a.med_workspace, a.med_workspace_bytes = 3.0, room.data_ptr() + spans[i][0], spans[i][1]
            a.median, a.thr, a.n_out = median.data_ptr(), thr.data_ptr(), count.data_ptr()
        args.append((a, grid))
        keep.append((x, joint, slack, t, median, thr, count))
    (ak, gk), (av, gv) = args
    L.call(lib.hqmq_append_kv_grid, case, torch.cuda.current_device(), C.addressof(ak), C.addressof(av), gk, gv)
    torch.cuda.synchronize()
    return q, keep


@pytest.mark.parametrize("layout", ["apart", "same", "overlap", "overlap below", "V's is small", "K's is small", "both small"])
@pytest.mark.parametrize("dn,S,b_r,d_h,T_k,T_v,med", [
    ("fp16", 96, 4, 128, 700, 700, (0, 1)), ("bf16", 24, 3, 128, 650, 650, (0, 1)), ("fp16", 192, 6, 64, 1100, 2300, (0, 1)),
    ("bf16", 96, 4, 128, 2200, 600, (0, 1)), ("fp16", 24, 3, 128, 600, 300, (0, 1)), ("fp16", 96, 4, 128, 620, 620, (0,)), ("bf16", 24, 3, 128, 620, 700, (1,))])
def test_appends_whatever_the_workspaces(layout, dn, S, b_r, d_h, T_k, T_v, med):
    """K and V of one append are the threshold's, the quantizer's and the compaction's calls for K and then for V, also where the two share
    a workspace or a part of one, differ in length, or only one of them extracts outliers.  V's norms are a hundred times K's."""
    from hqmq_amd import ops
    from hqmq_amd.packed import PackedTensor
    dt, B, H = DT[dn], 1, 3
    ks = kv_input((B, H, T_k, d_h), dt, seed=T_k, outlier_p=0.02).to(DEV)
    vs = (kv_input((B, H, T_v, d_h), torch.float32, seed=T_v + 1, outlier_p=0.03, outlier_gain=(5.0, 9.0)) * 100).to(dt).to(DEV)
    q, got = _appended_through_the_c_abi("append", ks, vs, med, layout, dt, S, b_r, d_h, H)
    for i, (x, joint, slack, t, median, thr, count) in enumerate(got):
        want = PackedTensor(B, H, t.t_cap, d_h, S, b_r, dt, DEV, joint, outliers=True, layout=(t.idx_bits, t.main_bits, t.aux_bits))
        if i in med:
            m, th, n = ops.med3x_threshold(x, 3.0)
            assert torch.equal(median, m) and torch.equal(thr.view(torch.int16), th.view(torch.int16)) and torch.equal(count, n) and int(n.min()) > 0
        ops.quantize(x, joint, slack, b_r, want_codes=False, thr=th if i in med else None, cache=want)
        if i in med:
            ops.outlier_compact(x, want)
        for name in ("main", "aux", "scale", "flags", "sb_tile_off", "sb_count", "sb_overflow"):
            a, b = getattr(t, name), getattr(want, name)
            assert (a is None) == (b is None) and (a is None or torch.equal(a.view(torch.uint8), b.view(torch.uint8))), (name, "KV"[i])
        for b in range(B):
            for h in range(H):
                n = int(want.sb_count[b, h])
                assert torch.equal(t.sideband[b, h, :n].view(torch.int16), want.sideband[b, h, :n].view(torch.int16)) and torch.equal(t.sb_coord[b, h, :n], want.sb_coord[b, h, :n])
