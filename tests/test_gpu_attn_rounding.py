"""How often the attention kernels round on the way from a softmax weight to the product with V: once, to fp16.  The split partials
leave the kernel in fp32, so that with every weight of a row alike, and V alike in every weighted token, the relative error of an
output is that of one weight."""
import pytest
import torch

from tests.helpers import unpack_planes

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def merged(O, partials, n_splits):
    """Split partials (m, l, two unused, acc) -> outputs in float64."""
    B, H, Tq, d = O.shape
    r = partials[:B * H * Tq * n_splits * (d + 4) * 4].view(torch.float32).view(B, H, Tq, n_splits, d + 4).double()
    w = torch.exp2(r[..., :1] - r[..., :1].amax(3, keepdim=True))
    return (r[..., 4:] * w).sum(3) / (r[..., 1:2] * w).sum(3)


@pytest.mark.parametrize("med", [False, True])
@pytest.mark.parametrize("dn", ["fp16", "bf16"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("S,b_r", [(96, 4), (24, 3), (192, 6), (192, 4)])
def test_weights_are_rounded_once(S, b_r, d, dn, med):
    import hqmq
    from hqmq_amd import ops
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dn]
    Hkv, G, T, ns, n = 4, 4, 160, 2, d // 4
    for B, Tq in ((8, 1), (16, 9)):       # one column group; three, two of them in one wavefront where the layout has that form
        g = torch.Generator().manual_seed(S + d + Tq)
        # every 16th token has the largest score and V = 0; the others are alike, so their weights are too, in every wavefront
        peak = torch.arange(T) % 16 == 0
        k, v = (torch.nn.functional.normalize(torch.randn(B, Hkv, 1, n, 4, generator=g), dim=-1) for _ in range(2))
        k = k.reshape(B, Hkv, 1, d).expand(B, Hkv, T, d).clone()
        k[:, :, ~peak] *= 0.5
        v = v * (0.7 + 0.6 * torch.rand(B, Hkv, 1, n, 1, generator=g)) * (0.7 + 1.3 * torch.rand(B, Hkv, 1, 1, 1, generator=g))
        v = v.reshape(B, Hkv, 1, d) * ~peak.view(T, 1)
        if med:                           # two chunks of every token verbatim, in different lanes and positions
            v[..., 4:8] = v[..., 4:8].sign() * (v[..., 4:8].abs() + 20)
            v[..., d - 8:d - 4] = v[..., d - 8:d - 4].sign() * (v[..., d - 8:d - 4].abs() + 20)
            v[:, :, peak] = 0
        q = hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=S, radius_bits=b_r, device="cuda")
        if med:
            q = hqmq.with_outlier_extraction(q, C=3.0)
        cache = q.new_cache(B, T, d, dt, 0)
        q.append(cache, k.to(dt).cuda(), v.to(dt).cuda(), 0)
        # queries along K, so that the peaks win, by 0.3 to 3 units of the exponent
        gap = (0.3 + 2.7 * torch.rand(B, Hkv, G, Tq, 1, generator=g)) / (d ** -0.5 * 0.5 * (k[:, :, :1].unsqueeze(2) ** 2).sum(-1, keepdim=True))
        Q = (gap * k[:, :, :1].unsqueeze(2)).to(dt).reshape(B, Hkv * G, Tq, d).cuda()

        # both tensors as the kernels decode them: codeword * radius code in fp16, scales and 1 / qmax behind it
        def decoded(t, b, x):
            idx, rq, flags = unpack_planes(t, b, T)
            cw = torch.stack([t.joint[h].half()[idx[h]] for h in range(Hkv)])
            y = (cw * rq.unsqueeze(-1).half()).double() * (t.scale[b, :, :T].double() / t.qmax).view(Hkv, T, 1, 1)
            if flags is not None:
                y = torch.where(flags.unsqueeze(-1), x.double().view(Hkv, T, n, 4), y)
            return y.view(Hkv, T, d), flags

        ref = []
        for b in range(B):
            K, kf = decoded(cache.K, b, k[b].to(dt).cuda())
            V, vf = decoded(cache.V, b, v[b].to(dt).cuda())
            assert not med or (int(vf.sum()) == 2 * Hkv * int((~peak).sum()) and int(kf.sum()) == 0)
            s = Q[b].double().view(Hkv, G * Tq, d) @ K.transpose(1, 2).contiguous() * d ** -0.5
            assert float(s.abs().max()) < 16
            ref.append((torch.softmax(s, -1) @ V).view(Hkv * G, Tq, d))
        ref = torch.stack(ref)
        assert bool((ref.abs().amax(-1) > 0.01).all())
        # 2^-11 for the weight; scores up to 16 from fp32 sums of d products and the exponential, 4e-5 of a weight
        bound = (2.0 ** -11 + 4e-5) * ref.abs() + 1e-6
        for generic in (0, 1, 2):
            O, parts, splits = ops.attn_fwd(Q, cache.K, cache.V, T, n_splits=ns, skip_combine=True, force_generic=generic)
            err = (merged(O, parts, splits) - ref).abs()
            assert bool((err <= bound).all()), (B, Tq, generic, float((err / bound).max()))
