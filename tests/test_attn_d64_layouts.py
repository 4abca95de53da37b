"""Attention over packed caches of 64-wide heads whose codes do not fill 16 bits each (12-bit main rows, radius bits in rows of 2, 4
or 6 bytes): every layout and both kernels' forms of it, against dense attention over the codes and the layout-generic kernel."""
import pytest
import torch

from tests.helpers import assert_attention_close, masked_two_refs

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

LAYOUTS = {(24, 3): (12, 1), (48, 2): (12, 1), (24, 4): (12, 2), (96, 3): (12, 3), (24, 5): (12, 3), (192, 4): (16, 1), (192, 5): (16, 2),
           (96, 6): (16, 2), (192, 6): (16, 3), (96, 7): (16, 3)}


@pytest.mark.parametrize("med", [False, True])
@pytest.mark.parametrize("dn", ["fp16", "bf16"])
@pytest.mark.parametrize("S,b_r", list(LAYOUTS))
def test_split_layouts_of_64_wide_heads(S, b_r, dn, med):
    import hqmq
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dn]
    # tokens: part of a tile, edges of half-steps and tiles, ranges of twelve wavefronts; columns: one, a group of 16 and a part of the
    # next, two groups per wavefront (a block per compute unit is left: 16 sequences x 8 heads x 2 pairs of groups)
    for B, Hq, Hkv, T, Tq, ns in ((2, 6, 2, 5, 1, 0), (3, 8, 4, 129, 1, 0), (2, 4, 2, 700, 5, 3), (2, 8, 2, 1601, 9, 1), (1, 8, 2, 4170, 1, 1), (16, 64, 8, 130, 7, 1)):
        g = torch.Generator().manual_seed(S + T)
        k, v = (torch.randn(B, Hkv, T, 64, generator=g) for _ in range(2))
        if med:
            k[:, :, ::3, 20] = 40.0
            v[:, :, 1::5, 47] = -25.0
        q = hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=S, radius_bits=b_r, device="cuda")
        if med:
            q = hqmq.with_outlier_extraction(q, C=3.0)
        cache = q.new_cache(B, T, 64, dt, 0)
        assert (cache.K.main_bits, cache.K.aux_bits) == LAYOUTS[S, b_r]
        q.append(cache, k.to(dt).cuda(), v.to(dt).cuda(), 0)
        Q = torch.randn(B, Hq, Tq, 64, generator=g).to(dt).cuda()
        lens = torch.randint(1, T + 1, (B,), generator=g)
        lens[0] = T
        row = torch.arange(T).view(1, 1, 1, T)
        causal = (row <= torch.arange(T - Tq, T).view(1, 1, Tq, 1)).cuda()
        ragged = (row < lens.view(B, 1, 1, 1)).cuda()
        for kw, vis in (({"causal": True, "causal_offset": T - Tq}, causal), ({"kv_lens": lens.int().cuda()}, ragged)):
            refs = masked_two_refs(cache, Q, T, vis)
            for generic in (0, 1):
                O = hqmq.fused_attention_packed(Q, cache, T_kv=T, n_splits=ns, force_generic=generic, **kw)
                assert_attention_close(O, *refs, base=2e-3, what=f"T={T} Tq={Tq} {list(kw)} generic={generic}")
