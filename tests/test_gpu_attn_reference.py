"""The reference of a column's softmax in the prefill kernels moves when a score exceeds it by more than six powers of two, with V scales
above 512 by anything: weights times V scales have to stay fp16 numbers either way, and as exact as they were."""
import pytest
import torch

from tests.helpers import exact_dense, unpack_planes

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("rise", [0.0, 5.0, 5.9, 40.0])         # of the scores over the sequence, in powers of two
@pytest.mark.parametrize("large_from", [None, 0, 100, 191, 192])   # first token whose V scale is far above 512
@pytest.mark.parametrize("d,med,dn", [(128, False, "fp16"), (64, False, "bf16"), (128, True, "fp16"), (64, True, "fp16")])
def test_rising_scores_and_large_values(d, med, dn, large_from, rise):
    import hqmq
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dn]
    Hkv, G, T, Tq, n = 2, 4, 333, 40, d // 4
    g = torch.Generator().manual_seed(d + int(rise))
    k = 0.05 * torch.randn(1, Hkv, T, d, generator=g)
    k[..., :4] += torch.linspace(0.05, 1, T).view(T, 1) * torch.tensor([0.5, 0.5, 0.5, 0.5])
    v = torch.randn(1, Hkv, T, n, 4, generator=g)
    v = torch.nn.functional.normalize(v, dim=-1).reshape(1, Hkv, T, d)
    if large_from is not None:
        v[:, :, large_from:] *= 25000.0
    if med:
        v[:, :, ::7, 8:12] *= 2.0                               # (of two verbatim fp16 chunks, none overflows)
    Q = torch.zeros(1, Hkv * G, Tq, d)
    Q[..., :4] = rise / 1.4427 * d ** 0.5 * 0.5
    Q += 0.3 * torch.randn(Q.shape, generator=g)
    q = hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=96, radius_bits=4, device="cuda")
    w = hqmq.with_outlier_extraction(q, C=1.5) if med else q
    cache = w.new_cache(1, T, d, dt, 0)
    k, v, Q = k.to(dt).cuda(), v.to(dt).cuda(), Q.to(dt).cuda()
    w.append(cache, k, v, 0)
    # K as the kernel multiplies it, codeword * radius code in fp16 and the scale behind it (half a unit of that, in a score of 28, is
    # 0.7 % of a weight)
    idx, rq, flags = unpack_planes(cache.K, 0, T)
    K = (torch.stack([cache.K.joint[h].half()[idx[h]] for h in range(Hkv)]) * rq.unsqueeze(-1).half()).double()
    K = K * (cache.K.scale[0, :, :T].double() / cache.K.qmax).view(Hkv, T, 1, 1)
    if med:
        K = torch.where(flags.unsqueeze(-1), k[0].double().view(Hkv, T, n, 4), K)
    K, V = K.view(Hkv, T, d), exact_dense(cache.V, 0, T, v[0]).double()
    s = Q[0].double().view(Hkv, G * Tq, d) @ K.transpose(1, 2).contiguous() * d ** -0.5
    p = torch.softmax(s, -1)
    ref, mass = (p @ V).view(1, Hkv * G, Tq, d), (p @ V.abs()).view(1, Hkv * G, Tq, d)
    # a weight and a value rounded to fp16 once each, scores of up to 64 in fp32, the output rounded to its type
    bound = (2 * 2.0 ** -11 + 2e-4) * mass + (2.0 ** -11 if dn == "fp16" else 2.0 ** -8) * ref.abs() + 1e-6
    for ns in (1, 3):
        O = hqmq.fused_attention_packed(Q, cache, n_splits=ns, force_generic=3)
        err = (O.double() - ref).abs()
        assert bool(torch.isfinite(O).all()) and bool((err <= bound).all()), (ns, float((err / bound).max()))
