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
