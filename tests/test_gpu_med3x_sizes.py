"""Med3x statistics, compaction and cropping at the sizes where a launch changes its kind: keys in registers of one
wavefront (512 chunks per head) and of a block (8192), histograms with packed and with 32-bit counters, appends on both
sides of the bulk compaction (512 rows), cuts on and off a tile."""
import pytest
import torch

from oracle import c_oracle as CO
from tests.helpers import DT, bit_equal, kv_input

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dn", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("shape", [(1, 2, 16, 128), (1, 2, 17, 128), (3, 2, 1, 80), (2, 1, 128, 128), (1, 1, 257, 128), (1, 2, 2049, 20),
                                   (1, 1, 3000, 128), (2, 1, 5, 4200)])
def test_threshold_at_the_edges(dn, shape):
    from hqmq_amd import ops
    dt = DT[dn]
    x = kv_input(shape, dt, seed=sum(shape), outlier_p=0.05)
    want = CO.med3x(x, 3.0)
    for view in (x.to(DEV), torch.nn.functional.pad(x, (1, 1)).to(DEV)[..., 1:1 + shape[-1]], x.to(DEV).transpose(1, 2).contiguous().transpose(1, 2)):
        med, thr, cnt = ops.med3x_threshold(view, 3.0)
        assert torch.equal(med.cpu(), want["median"]) and bit_equal(thr, want["threshold"])
        assert torch.equal(cnt.cpu().long(), want["mask"].sum(dim=(0, 2, 3)))


@pytest.mark.parametrize("dn", ["fp16", "bf16"])
def test_wide_and_packed_counters_agree(dn):
    """6.3 M chunks of one head (512 blocks, packed counters) and the same five times over (31 M: 256 blocks of 122880, beyond what
    16 bits count).  The two middle norms are equal, which the counts on either side show, so whatever the interpolation the
    median is that norm in both calls, the threshold is equal and the count five times."""
    from hqmq_amd import ops
    dt = DT[dn]
    x = torch.randn(1, 1, 49152, 512, generator=torch.Generator(device=DEV).manual_seed(3), device=DEV).to(dt)
    five = x.expand(5, -1, -1, -1).contiguous()
    n = x.numel() // 4
    assert n * 5 / 512 > 60000 and n / 512 < 60000               # the launch's rule for the counters
    (med, thr, cnt), (med5, thr5, cnt5) = ops.med3x_threshold(x, 1.5), ops.med3x_threshold(five, 1.5)
    m = med.to(dt)
    assert torch.equal(m.float(), med.float())                   # a norm of the call
    above, from_it = int(ops.outlier_mask(x, m).sum()), int(ops.outlier_mask(x, (m.view(torch.int16) - 1).view(dt)).sum())
    assert above < n // 2 < from_it                              # norms > median, norms >= median
    assert torch.equal(med, med5) and bit_equal(thr, thr5)
    assert int(ops.outlier_mask(x, thr).sum()) == int(cnt[0]) > 0 and int(cnt5[0]) == 5 * int(cnt[0])


@pytest.mark.parametrize("dn,d_h", [("fp16", 128), ("bf16", 64), ("fp32", 48), ("fp16", 16)])
@pytest.mark.parametrize("T", [33, 64, 65, 511, 512, 513, 2100])
def test_append_lists_and_crop(dn, d_h, T):
    """Sideband entries in (token, chunk) order, tile offsets and counts equal what the mask says, before and after a cut."""
    import hqmq
    dt = DT[dn]
    B, H, n = 2, 2, d_h // 4
    w = hqmq.with_outlier_extraction(hqmq.HQMQ(n_layers=1, n_heads=H, secondary_size=24, radius_bits=3, device=DEV), C=3.0)
    k, v = kv_input((B, H, T, d_h), dt, seed=T, outlier_p=0.1).to(DEV), kv_input((B, H, T, d_h), dt, seed=T + 1, outlier_p=0.02).to(DEV)
    cache = w.new_cache(B, T, d_h, dt, 0, sideband_frac=0.5)
    w.append(cache, k, v, 0)

    def check(lens):
        for pt, x in ((cache.K, k), (cache.V, v)):
            mask = w.encode(x, 0, 0)["mask"]
            for b in range(B):
                m = mask[b].clone()
                m[:, lens[b]:] = False
                assert torch.equal(pt.sb_count[b].long(), m.sum(dim=(1, 2)))
                for h in range(H):
                    tok, chunk = m[h].nonzero(as_tuple=True)
                    assert torch.equal(pt.sideband[b, h, :len(tok)], x[b, h].view(T, n, 4)[tok, chunk])
                    assert torch.equal(pt.sb_coord[b, h, :len(tok)].long(), (tok % 16) << 8 | chunk)
                    tiles = (lens[b] + 15) // 16
                    before = torch.tensor([int((tok < 16 * i).sum()) for i in range(tiles)])
                    assert torch.equal(pt.sb_tile_off[b, h, :tiles].long().cpu(), before)
                    assert bool((pt.sb_tile_off[b, h, (pt.t_cap if lens[b] == T else lens[b] + 15) // 16:] == 0x7fffffff).all())
                    flags = torch.stack([(pt.flags[b, h] >> i) & 1 for i in range(8)], -1).reshape(pt.t_cap, -1)[:, :n].bool()
                    assert torch.equal(flags[:T], m[h]) and not bool(flags[T:].any())

    check([T, T])
    cut = torch.tensor([T // 2, (T // 3) // 16 * 16], dtype=torch.int32, device=DEV)
    cache.crop_(cut)
    check(cut.tolist())
    cache.crop_(5)
    check([min(5, c) for c in cut.tolist()])
    cache.crop_(0)
    check([0, 0])


def test_crop_of_a_cache_made_for_cuda_without_an_index():
    """device="cuda" names no GPU index: the call goes to the device the planes are on.  Lengths on the host are accepted, K and V
    of different capacity are cropped one after the other."""
    from hqmq_amd.packed import PackedKV, PackedTensor
    K, V = (PackedTensor(2, 1, cap, 64, 24, 3, torch.float16, "cuda", outliers=True) for cap in (128, 192))
    for t in (K, V):
        t.flags.fill_(1)                # two flagged chunks in every row
        t.sb_tile_off.copy_(32 * torch.arange(t.t_cap // 16, dtype=torch.int32).expand(2, 1, -1))
        t.sb_count.fill_(2 * t.t_cap)
    PackedKV(K, V).crop_(torch.tensor([40, 128]))
    assert K.sb_count.flatten().tolist() == [2 * 40, 2 * 128] and V.sb_count.flatten().tolist() == [2 * 40, 2 * 128]
    K.crop_(16)
    assert K.sb_count.flatten().tolist() == [2 * 16, 2 * 16] and not bool(K.flags[:, :, 16:].any())


@pytest.mark.parametrize("dn", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", [(1, 3, 2, 128), (1, 3, 3, 128), (2, 2, 16, 128), (1, 2, 33, 124), (5, 1, 13, 64), (1, 2, 65, 128), (2, 2, 64, 128), (1, 1, 129, 128),
                                   (1, 2, 511, 128), (4, 1, 128, 128), (1, 2, 513, 128), (1, 2, 3, 4000), (1, 1, 16, 4096), (1, 1, 17, 4096), (3, 1, 20, 12)])
def test_histogram_of_a_block(dn, shape):
    """65 to 16384 chunks per head, on both sides of 1, 2, 4, 8 and 16 keys per lane and with rows that do not fill the lanes; ordinary
    norms, all equal, two values of which the middle ranks take one each, zeros, infinities, a NaN."""
    from hqmq_amd import ops
    dt = DT[dn]
    x = kv_input(shape, dt, seed=sum(shape) + 1, outlier_p=0.05)
    n = shape[0] * shape[2] * shape[3] // 4
    flat = torch.arange(n).view(1, n, 1).expand(shape[1], n, 4)
    two = torch.where(flat < n // 2, 0.25, 2.0).reshape(shape[1], shape[0], shape[2], shape[3]).transpose(0, 1)
    inf = x.clone()
    inf[:, :, ::2, 0] = float("inf")
    nan = x.clone()
    nan[-1, -1, -1, -1] = float("nan")
    for y in (x, torch.full(shape, 0.5).to(dt), two.to(dt), torch.zeros(shape).to(dt), inf, nan):
        want = CO.med3x(y, 3.0)
        med, thr, cnt = ops.med3x_threshold(y.to(DEV), 3.0)
        same = (med.cpu() == want["median"]) | (med.cpu().isnan() & want["median"].isnan())
        assert same.all() and (bit_equal(thr, want["threshold"]) or thr.isnan().any())
        assert torch.equal(cnt.cpu().long(), want["mask"].sum(dim=(0, 2, 3)))


@pytest.mark.parametrize("dn", ["fp16", "bf16"])
@pytest.mark.parametrize("H,rows,mult", [(1, 4100, 3.0), (7, 600, 100.0), (300, 257, 0.01), (2, 4097, 0.0), (3, 5000, 1e5)])
def test_histograms_of_blocks(dn, H, rows, mult):
    """16-bit types beyond 8192 chunks per head: one part of the workspace per block, from one part for a head to as many as a
    launch may have; thresholds in the median's group of bins, next to it and far from it; the two middle norms in different
    groups; a head of equal norms; infinite norms, NaN and zeros."""
    from hqmq_amd import _lib, ops
    dt = DT[dn]
    x = kv_input((1, H, rows, 128), dt, seed=H + rows, outlier_p=0.03)
    if H >= 3:
        half = rows * 16                                    # of rows * 32 chunks
        x[0, 1] = 0.25
        x[0, 1].view(-1, 4)[half:] *= 4096.0                # the middle two: 0.5 and 2048
        x[0, 2] = 1.5
    if H >= 7:
        x[0, 3].view(-1, 4)[:40] = float("inf")
        x[0, 4, 5, 7] = float("nan")
        x[0, 5].view(-1, 4)[: half + 9] = 0
        x[0, 6].view(-1, 4)[:] = 6e-5 * (1 + torch.arange(rows * 32) % 9).to(dt).view(-1, 1)
    want = CO.med3x(x, mult)
    med, thr, cnt = ops.med3x_threshold(x.to(DEV), mult)
    assert bit_equal(med, want["median"]) and bit_equal(thr, want["threshold"])
    assert torch.equal(cnt.cpu().long(), want["mask"].sum(dim=(0, 2, 3)))
    again = ops.med3x_threshold(x.to(DEV), mult)            # over what the first call left in the workspace
    assert bit_equal(again[0], med) and bit_equal(again[1], thr) and torch.equal(again[2], cnt)
    # the smaller workspace: one histogram per head
    xg, med2, thr2, cnt2 = x.to(DEV), torch.empty_like(med), torch.empty_like(thr), torch.empty_like(cnt)
    ws = torch.full((_lib.lib().hqmq_med3x_workspace_bytes(H, _lib.DT_CODE[dt]),), 255, dtype=torch.uint8, device=DEV)
    _lib.call(_lib.lib().hqmq_med3x_threshold, "hqmq_med3x_threshold", 0, xg.data_ptr(), *xg.stride()[:3], _lib.DT_CODE[dt], 1, H, rows, 32, mult,
              ws.data_ptr(), ws.numel(), med2.data_ptr(), thr2.data_ptr(), cnt2.data_ptr())
    assert bit_equal(med2, med) and bit_equal(thr2, thr) and torch.equal(cnt2, cnt)
