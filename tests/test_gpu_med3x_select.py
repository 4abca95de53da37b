"""Calls whose quantize launch works the Med3x threshold out for itself (16-bit types, more than 16384 chunks per head), against the
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
    ("bf16", 24, 3, (1, 9, 530, 128), "zero")])
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
    (1, 1, 129, 512), (1, 5, 513, 128)])        # last blocks of a single step
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
