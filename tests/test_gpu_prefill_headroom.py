"""The prefill kernel lets weights grow to 2^4 before it takes a new reference, but not where their products with V's scales could leave
fp16: scores that climb a little from tile to tile, V scales on both sides of the line (2048), and beyond it in one late token only."""
import pytest
import torch

from tests.helpers import unpack_planes

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("top", [1.0, 2000.0, 2100.0, 3e4, 6e4])
@pytest.mark.parametrize("late", [False, True])
@pytest.mark.parametrize("dn", ["fp16", "bf16"])
def test_climbing_scores_and_large_scales(dn, late, top):
    import hqmq
    from hqmq_amd import ops
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dn]
    if dn == "bf16" and top > 32767:
        top = 3e4                       # (beyond 2^15 the layout-generic kernel takes bf16 caches)
    B, Hkv, G, d, T, Tq = 1, 2, 4, 128, 700, 40
    g = torch.Generator().manual_seed(7)
    q = hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=96, radius_bits=4, device="cuda")
    # every key points the same way and is longer than the one before it: the maximum moves in every tile, by a power of two or two
    way = torch.randn(1, 1, 1, d, generator=g)
    k = way * (0.5 + torch.arange(T).view(T, 1) / T) * torch.ones(B, Hkv, 1, 1)
    v = torch.nn.functional.normalize(torch.randn(B, Hkv, T, d // 4, 4, generator=g), dim=-1).reshape(B, Hkv, T, d)
    size = torch.full((T, 1), top)
    if late:                            # ordinary tokens in front of the large one, whose score is below the maximum by then
        size = torch.ones(T, 1)
        size[620] = top
        k[:, :, 620] *= 0.97
    v = v * size
    cache = q.new_cache(B, T, d, dt, 0)
    q.append(cache, k.to(dt).cuda(), v.to(dt).cuda(), 0)
    Q = (way * (0.8 + 0.4 * torch.rand(B, Hkv * G, Tq, 1, generator=g)) * 2.5).to(dt).cuda()
    O = ops.attn_fwd(Q, cache.K, cache.V, T, causal=True, causal_offset=T - Tq, n_splits=1, force_generic=3)
    limit = torch.arange(Tq, device="cuda").view(1, Tq, 1) + T - Tq + 1
    for h in range(Hkv):
        def decoded(t):
            idx, rq, _ = unpack_planes(t, 0, T)
            cw = t.joint[h].half()[idx[h]]
            return ((cw * rq[h].unsqueeze(-1).half()).double() * (t.scale[0, h, :T].double() / t.qmax).view(T, 1, 1)).view(T, d)
        K, V = decoded(cache.K), decoded(cache.V)
        s = Q[0, h * G:(h + 1) * G].double().reshape(G * Tq, d) @ K.t().contiguous() * d ** -0.5
        s = s.view(G, Tq, T).masked_fill(torch.arange(T, device="cuda").view(1, 1, T) >= limit, -torch.inf)
        P = torch.softmax(s, -1).view(G * Tq, T)
        ref, mass = P @ V, P @ V.abs()
        # one rounding of the product of weight and scale; fp32 scores below 128; the output's own rounding
        eps = 2.0 ** -11 if dn == "fp16" else 2.0 ** -8
        bound = (2.0 ** -11 + 2e-4) * mass + eps * ref.abs() + 1e-6
        err = (O[0, h * G:(h + 1) * G].double().reshape(G * Tq, d) - ref).abs()
        assert bool(torch.isfinite(O).all()) and bool((err <= bound).all()), float((err / bound).max())
