"""V's codewords and radius codes through transposing LDS reads: every code layout, all radius codes, ragged ends of tiles and ranges."""
import pytest
import torch

from tests.helpers import unpack_planes
from tests.test_gpu_attn_rounding import merged

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


# 16+0 (index widths 12, 11 and 8), 12+1 (10: tables multiplied out, 9, 6), 16+3 (13, 12, 11), 16+1, 16+2, 12+2, 12+3; up to 8 radius bits; tables of odd sizes
@pytest.mark.parametrize("S,b_r", [(96, 4), (64, 5), (24, 3), (21, 4), (192, 6), (192, 4), (96, 6), (24, 4), (24, 5), (96, 7), (10, 8), (48, 8), (2, 8), (90, 4), (171, 6)])
@pytest.mark.parametrize("d", [64, 128])
def test_every_token_chunk_and_radius(S, b_r, d):
    import hqmq
    from hqmq_amd import ops
    B, Hkv, G, n = 3, 2, 4, d // 4
    q = hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=S, radius_bits=b_r, device="cuda")
    for T, Tq, ns, med, dt in ((1, 1, 1, False, torch.float16), (77, 1, 1, False, torch.bfloat16), (333, 5, 2, True, torch.float16), (1100, 1, 1, True, torch.bfloat16), (4600, 1, 1, False, torch.float16), (5003, 1, 1, False, torch.bfloat16)):
        g = torch.Generator().manual_seed(S + d + T)
        # norms spread over the whole range of a token's radius codes
        x = torch.nn.functional.normalize(torch.randn(2, B, Hkv, T, n, 4, generator=g), dim=-1) * torch.rand(2, B, Hkv, T, n, 1, generator=g)
        if med:
            x = torch.where(torch.rand(2, B, Hkv, T, n, 1, generator=g) < 0.03, 40 * x, x)
        k, v = (y.reshape(B, Hkv, T, d).to(dt).cuda() for y in x)
        w = hqmq.with_outlier_extraction(q, C=3.0) if med else q
        cache = w.new_cache(B, T, d, dt, 0)
        w.append(cache, k, v, 0)
        Q = torch.randn(B, Hkv * G, Tq, d, generator=g).to(dt).cuda()

        def decoded(t, b, raw):         # as the kernels decode: codeword * radius code in fp16, scale and 1 / qmax behind it
            idx, rq, flags = unpack_planes(t, b, T)
            cw = torch.stack([t.joint[h].half()[idx[h]] for h in range(Hkv)])
            y = (cw * rq.unsqueeze(-1).half()).double() * (t.scale[b, :, :T].double() / t.qmax).view(Hkv, T, 1, 1)
            if flags is not None:
                y = torch.where(flags.unsqueeze(-1), raw.double().view(Hkv, T, n, 4), y)
            assert T < 300 or int(rq.max()) == t.qmax and int(rq.unique().numel()) == t.qmax + 1
            return y.view(Hkv, T, d)

        ref, size = [], []
        for b in range(B):
            K, V = decoded(cache.K, b, k[b]), decoded(cache.V, b, v[b])
            P = torch.softmax(Q[b].double().view(Hkv, G * Tq, d) @ K.transpose(1, 2).contiguous() * d ** -0.5, -1)
            ref.append((P @ V).view(Hkv * G, Tq, d))
            size.append((P @ V.abs()).view(Hkv * G, Tq, d))
        ref, size = torch.stack(ref), torch.stack(size)
        # one rounding of the weight, 2^-11; fp32 scores below 64 and their exponential, 6e-5 of a weight; fp32 sums
        bound = (2.0 ** -11 + 1e-4) * size + 1e-6
        for form in (0, 2):
            if ns > 1:
                O, parts, splits = ops.attn_fwd(Q, cache.K, cache.V, T, n_splits=ns, skip_combine=True, force_generic=form)
                assert bool(((merged(O, parts, splits) - ref).abs() <= bound).all()), (T, form)
            else:                       # (stored in the cache dtype)
                O = ops.attn_fwd(Q, cache.K, cache.V, T, n_splits=1, force_generic=form)
                eps = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
                assert bool(((O.double() - ref).abs() <= bound + eps * ref.abs() + 2.0 ** -24).all()), (T, form)


# (index bits, main bits, aux bits) of radius fields with more than 8 bits, and of an index field with less than 3: the table of radius codes
# ends at 256, so the layout-generic kernel has these calls
@pytest.mark.parametrize("layout,b_r", [((7, 16, 0), 9), ((6, 16, 0), 10), ((2, 16, 0), 9), ((1, 16, 0), 4), ((6, 12, 3), 9), ((5, 12, 2), 8), ((8, 16, 1), 9)])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_radius_fields_wider_than_the_table(layout, b_r, d, dt):
    from hqmq_amd import ops
    from hqmq_amd.packed import PackedTensor
    B, H, G, T, n, K = 2, 2, 4, 333, d // 4, min(120, 1 << layout[0])
    g = torch.Generator().manual_seed(d + b_r + layout[0])
    most = min((1 << b_r) - 1, 1023)
    sides, dense = [], []
    for _ in range(2):
        idx = torch.randint(0, K, (B, H, T, n), generator=g, dtype=torch.int32)
        rq = torch.randint(0, most + 1, (B, H, T, n), generator=g, dtype=torch.int32)
        rq[:, :, 0, :2] = torch.tensor([0, most], dtype=torch.int32)
        joint = torch.nn.functional.normalize(torch.randn(H, K, 4, generator=g), dim=-1).to(dt)
        t = PackedTensor(B, H, T, d, 1, b_r, dt, "cuda", joint=joint.cuda(), layout=layout)
        t.scale[:, :, :T] = (0.5 + torch.rand(B, H, T, generator=g)).to(dt).cuda()
        ops.pack_codes(idx.cuda(), rq.cuda(), t)
        sides.append(t)
        cw = torch.stack([joint[h].half()[idx[:, h].long()] for h in range(H)], 1)
        y = (cw * rq.unsqueeze(-1).half()).double() * (t.scale[:, :, :T].cpu().double() / t.qmax).view(B, H, T, 1, 1)
        dense.append(y.view(B, H, T, d))
    Q = torch.randn(B, H * G, 1, d, generator=g).to(dt).cuda()
    P = torch.softmax(Q.cpu().double().view(B, H, G, d) @ dense[0].transpose(2, 3).contiguous() * d ** -0.5, -1)
    ref, size = (P @ dense[1]).view(B, H * G, 1, d), (P @ dense[1].abs()).view(B, H * G, 1, d)
    eps = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    for ns in (1, 2):
        for form in (0, 1, 2):
            O = ops.attn_fwd(Q, sides[0], sides[1], T, n_splits=ns, force_generic=form).cpu().double()
            # two roundings of the weight, 2^-11 each, fp32 scores and exponential as above, and the output's own rounding
            assert bool(((O - ref).abs() <= (2.0 ** -10 + 1e-4) * size + eps * ref.abs() + 1e-6).all()), (ns, form)


# 264 blocks of heads of 64, whole sequences: started longest first each has a compute unit of its own, else two share one
@pytest.mark.parametrize("S,b_r,dt", [(192, 4, torch.bfloat16), (192, 6, torch.float16), (24, 5, torch.bfloat16)])
@pytest.mark.parametrize("T", [3900, 4000, 4200])
def test_the_order_of_the_sequences_changes_nothing(S, b_r, dt, T):
    import hqmq
    from hqmq_amd import ops
    B, H = 33, 8
    q = hqmq.HQMQ(n_layers=1, n_heads=H, secondary_size=S, radius_bits=b_r, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(T)
    k, v = (torch.randn(B, H, T, 64, generator=g, device="cuda", dtype=dt) for _ in range(2))
    cache = q.new_cache(B, T, 64, dt, 0)
    q.append(cache, k, v, 0)
    lens = torch.randint(1, T + 1, (B,), generator=g, device="cuda", dtype=torch.int32)
    lens[3] = T
    Q = torch.randn(B, 2 * H, 1, 64, generator=g, device="cuda", dtype=dt)
    plain, ordered = (ops.attn_fwd(Q, cache.K, cache.V, T, kv_lens=lens, batch_order=o, n_splits=1) for o in (None, ops.longest_first(lens)))
    assert torch.equal(plain, ordered)
    assert bool(((plain - ops.attn_fwd(Q, cache.K, cache.V, T, kv_lens=lens, force_generic=1)).abs() <= (2e-3 if dt == torch.float16 else 1e-2)).all())


# 248 and 256 blocks of whole sequences around the lines between the kernel whose loads land in LDS and twelve wavefronts
@pytest.mark.parametrize("S,b_r,dt", [(96, 4, torch.float16), (12, 7, torch.bfloat16)])
@pytest.mark.parametrize("B", [31, 32])
def test_lines_of_the_twelve_wavefront_form(S, b_r, dt, B):
    import hqmq
    from hqmq_amd import ops
    H, T = 8, 5010
    q = hqmq.HQMQ(n_layers=1, n_heads=H, secondary_size=S, radius_bits=b_r, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(B)
    k, v = (torch.randn(B, H, T, 128, generator=g, device="cuda", dtype=dt) for _ in range(2))
    cache = q.new_cache(B, T, 128, dt, 0)
    q.append(cache, k, v, 0)
    Q = torch.randn(B, 2 * H, 1, 128, generator=g, device="cuda", dtype=dt)
    for t in (4095, 4096, 4999, 5000):
        O, plain = (ops.attn_fwd(Q, cache.K, cache.V, t, n_splits=1, force_generic=form) for form in (0, 1))
        # each weight rounded to fp16 twice at most, outputs (means of 4000 values and more: below 0.5) once: 2^-10 and the type's epsilon, on both sides
        assert float((O.float() - plain.float()).abs().max()) <= 2 * (2.0 ** -10 + 0.5 * (2.0 ** -11 if dt == torch.float16 else 2.0 ** -8)), t


# 12 + 1 bits, around the most codewords that tables multiplied out have room for: 1022, and 1016 over an outlier cache's values
@pytest.mark.parametrize("K", [1014, 1016, 1018, 1022, 1024])
@pytest.mark.parametrize("med", [False, True])
@pytest.mark.parametrize("d,dt", [(64, torch.bfloat16), (128, torch.float16)])
def test_largest_tables_of_ten_index_bits(K, med, d, dt):
    import hqmq
    from hqmq_amd import ops
    B, H, G, T, n = 2, 2, 4, 700, d // 4
    q = hqmq.HQMQ(n_layers=1, n_heads=H, secondary_size=42, radius_bits=3, device="cuda")
    w = hqmq.with_outlier_extraction(q, C=3.0) if med else q
    g = torch.Generator().manual_seed(K + d)
    x = torch.randn(2, B, H, T, n, 4, generator=g)
    if med:
        x = torch.where(torch.rand(2, B, H, T, n, 1, generator=g) < 0.03, 20 * x, x)
    k, v = (y.reshape(B, H, T, d).to(dt).cuda() for y in x)
    cache = w.new_cache(B, T, d, dt, 0)
    w.append(cache, k, v, 0)
    assert (cache.K.idx_bits, cache.K.main_bits, cache.K.aux_bits) == (10, 12, 1)
    dense = []
    for t, raw in ((cache.K, k), (cache.V, v)):     # the codebook's 1008 codewords counted from the end of a table of K
        codes = [unpack_planes(t, b, T) for b in range(B)]
        idx, rq = (torch.stack([c[i].cpu() for c in codes]).int() for i in (0, 1))
        table = torch.nn.functional.normalize(torch.randn(H, K, 4, generator=g), dim=-1).to(dt)
        table[:, K - 1008:] = t.joint.cpu().flip(1)
        third = (torch.arange(T) % 3 == 0).view(T, 1)
        idx = torch.where(third, torch.randint(0, K, idx.shape, generator=g, dtype=torch.int32), K - 1 - idx)    # and every codeword of the table
        t.joint = table.cuda()
        ops.pack_codes(idx.cuda(), rq.cuda(), t)
        cw = torch.stack([table[h].half()[idx[:, h].long()] for h in range(H)], 1)
        y = (cw * rq.unsqueeze(-1).half()).double() * (t.scale[:, :, :T].cpu().double() / t.qmax).view(B, H, T, 1, 1)
        if med:
            flags = torch.stack([c[2].cpu() for c in codes])
            assert int(flags.sum()) > 0 and int(rq[flags].max()) == 0
            y = torch.where(flags.unsqueeze(-1), raw.cpu().double().view(B, H, T, n, 4), y)
        dense.append(y.view(B, H, T, d))
    Q = torch.randn(B, H * G, 1, d, generator=g).to(dt).cuda()
    P = torch.softmax(Q.cpu().double().view(B, H, G, d) @ dense[0].transpose(2, 3).contiguous() * d ** -0.5, -1)
    ref, size = (P @ dense[1]).view(B, H * G, 1, d), (P @ dense[1].abs()).view(B, H * G, 1, d)
    # what weights below fp16's normal numbers lose: 2^-25 of weight * scale and weight * qmax, layout-generic of weight * scale / qmax and weight
    small = 2.0 ** -25 / min(float(cache.V.scale[:, :, :T].min()), cache.V.qmax) * dense[1].abs().sum(2, keepdim=True).expand(B, H, G, d).reshape(B, H * G, 1, d)
    eps = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    for ns in (1, 3):
        for form in (0, 1):
            O = ops.attn_fwd(Q, cache.K, cache.V, T, n_splits=ns, force_generic=form).cpu().double()
            # two roundings of the weight, 2^-11 each, fp32 scores and exponential (6e-5 of a weight), and the output's own rounding
            bound = (2.0 ** -10 + 1e-4) * size + eps * ref.abs() + (small * cache.V.qmax if form else small) + 2.0 ** -24
            assert bool(((O - ref).abs() <= bound).all()), (ns, form)
