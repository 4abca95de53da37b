"""The number of blocks that share one sequence: what the choice promises to its callers (CPU) and, on the GPU, attention over
contexts and batches on both sides of where it changes, against dense attention over the dequantized cache."""
import ctypes as C

import pytest
import torch

from tests.helpers import assert_attention_close, masked_two_refs


def _args(B, Hq, Hkv, Tq, T, n, flags, dtype, kv_len=False, generic=0):
    from hqmq_amd import _lib as L
    a = L.AttnArgs()
    a.B, a.H_q, a.H_kv, a.T_q, a.T_kv, a.t_cap, a.n_chunks, a.dtype, a.qmax, a.idx_bits, a.force_generic = B, Hq, Hkv, Tq, T, T, n, dtype, 15, 12, generic
    a.K.flag_plane = 16 if flags else None
    a.kv_len = 16 if kv_len else None
    return a


def test_splits_keep_to_rounds_of_blocks_and_to_earlier_workspaces():
    from hqmq_amd import _lib as L
    lib = L.lib()
    for ragged in (0, 1):
        for n, flags, dtype, generic in ((32, 0, L.DT_CODE[torch.float16], 0), (32, 1, L.DT_CODE[torch.bfloat16], 0), (16, 1, L.DT_CODE[torch.float16], 0),
                                         (16, 0, L.DT_CODE[torch.bfloat16], 1), (20, 0, L.DT_CODE[torch.float32], 0)):
            for B in (1, 2, 3, 5, 31, 32, 33, 64, 127, 128, 129, 130, 1000):
                for T in (1, 63, 64, 65, 127, 128, 129, 300, 511, 513, 1025, 4096, 6145, 20001, 1 << 20):
                    base = B * 8
                    old = max(1, min(((512 if ragged else 256) + base - 1) // base, (T + 127) // 128, 512))
                    assert 1 <= lib.hqmq_attn_pick_splits(B, 32, 8, 1, T, ragged) <= old
                    a = _args(B, 32, 8, 1, T, n, flags, dtype, ragged, generic)
                    s = lib.hqmq_attn_splits(C.addressof(a))
                    assert 1 <= s <= max(1, (T + 127) // 128) and (s == 1 or base * s <= (640 if ragged else 1024)), (B, T, s)
                    a.T_kv = a.t_cap = (T + 63) // 64 * 64
                    assert lib.hqmq_attn_splits(C.addressof(a)) == s                    # the key under which callers keep it
    assert lib.hqmq_attn_pick_splits(1, 32, 8, 1, 0, 0) == 1 and lib.hqmq_attn_pick_splits(1, 4, 8, 1, 500, 0) == 1
    for T, s in ((300, 1), (4096, 32), (32768, 32)):       # one block, whole rounds of 256
        assert lib.hqmq_attn_pick_splits(1, 32, 8, 1, T, 0) == s
    assert lib.hqmq_attn_pick_splits(12, 32, 8, 1, 4096, 0) == 2                        # 192 blocks, not 288


def test_any_wide_range_is_the_generic_kernel():
    from hqmq_amd import _lib as L
    lib, word = L.lib(), C.c_uint32()
    a = _args(4, 32, 8, 1, 700, 32, False, L.DT_CODE[torch.bfloat16])
    a.V.scale_max_bits = C.addressof(word)
    few = lib.hqmq_attn_splits(C.addressof(a))
    for w in (1, 2, 3, -1):
        a.wide_range = w
        assert lib.hqmq_attn_splits(C.addressof(a)) > few, w
    assert lib.hqmq_attn_fwd_guarded(C.byref(a), None) != 0             # either the caller knows or the GPU decides
    a.wide_range, a.V.scale_max_bits = 0, None
    assert lib.hqmq_attn_fwd_guarded(C.byref(a), None) != 0
    assert lib.hqmq_attn_fwd_guarded(None, None) != 0


def test_ragged_batches_beyond_one_round():
    from hqmq_amd import _lib as L
    f16 = L.DT_CODE[torch.float16]
    for n, flags, counts in ((32, False, {41: 2, 48: 2, 56: 2, 62: 2, 63: 1, 64: 1, 80: 1}), (32, True, {41: 2, 48: 2, 56: 2, 62: 2, 63: 1, 64: 1}),
                             (16, True, {41: 2, 62: 2, 64: 1}), (16, False, {41: 3, 48: 2, 64: 2, 65: 1})):
        for B, splits in counts.items():      # 328 to 1024 pairs of up to 16384 tokens; whole sequences of few tokens
            a = _args(B, 32, 8, 1, 16384, n, flags, f16, True)
            assert L.lib().hqmq_attn_splits(C.addressof(a)) == splits, (n, flags, B)
            a.T_kv = a.t_cap = 1024
            assert L.lib().hqmq_attn_splits(C.addressof(a)) == 1, (n, flags, B)


@pytest.mark.parametrize("B,Hq,Hkv,d_h,T,Tq,S,b_r,dn,splits", [
    # us measured with the decode kernels and with the prefill kernel; the two would run with different numbers of splits
    (1, 32, 8, 128, 19403, 33, 24, 3, "fp16", 6),       # 37.8, 47.2 with 16
    (1, 32, 8, 128, 21640, 43, 24, 3, "fp16", 5),       # 45.3, 52.1 with 16
    (1, 32, 8, 128, 9170, 127, 24, 3, "bf16", 2),       # 46.6, 51.2 with 8
    (10, 64, 8, 64, 2717, 16, 192, 4, "bf16", 3),       # 46.5 with 1, 34.4
    (2, 64, 8, 64, 2070, 76, 24, 3, "fp16", 3),         # 36.7 with 1, 29.4
    (3, 28, 4, 128, 5811, 70, 192, 4, "bf16", 5),       # 62.9 with 1, 50.8
    (7, 28, 4, 128, 2990, 73, 192, 6, "fp16", 2)])      # 70.9 with 1, 60.5
def test_prefill_chunks_take_the_faster_kernel(B, Hq, Hkv, d_h, T, Tq, S, b_r, dn, splits):
    from hqmq_amd import _lib as L
    a = _args(B, Hq, Hkv, Tq, T, d_h // 4, False, L.DT_CODE[{"fp16": torch.float16, "bf16": torch.bfloat16}[dn]])
    a.idx_bits, a.main_bits, a.aux_bits = L.layout_bits(S, b_r)
    a.K.K = a.V.K = 24 * S
    a.t_cap, a.qmax, a.softmax_scale, a.causal, a.causal_offset = (T + 63) // 64 * 64, (1 << b_r) - 1, d_h ** -0.5, 1, T - Tq
    assert L.lib().hqmq_attn_splits(C.addressof(a)) == splits
    a.force_generic = 2           # never the prefill kernel
    assert (L.lib().hqmq_attn_splits(C.addressof(a)) == splits) == (S == 24 and T > 9000)


@pytest.mark.parametrize("med,B,Hq,Hkv,d_h,T,Tq,S,b_r", [
    # over outlier caches: with the prefill kernel, whose error is 0.82 of the decode kernels' where K's verbatim chunks are large
    (True, 8, 32, 8, 128, 341, 17, 96, 4), (True, 7, 28, 4, 128, 909, 21, 192, 6), (True, 1, 28, 4, 128, 8299, 43, 96, 4),
    (True, 1, 32, 8, 128, 4393, 101, 192, 6), (True, 5, 28, 4, 128, 215, 29, 192, 4),
    # over plain fp16 caches: with the decode kernels, up to 2 % nearer to 64-bit results
    (False, 8, 64, 8, 64, 3109, 31, 192, 4), (False, 6, 32, 8, 128, 1024, 45, 96, 4), (False, 8, 32, 8, 128, 1382, 46, 24, 3),
    (False, 1, 64, 8, 64, 5289, 79, 192, 4), (False, 3, 32, 8, 128, 1121, 87, 192, 6)])
def test_fp16_chunks_keep_to_the_kernel_of_smaller_error(med, B, Hq, Hkv, d_h, T, Tq, S, b_r):
    """Calls near the line between the two kernels, for which the times alone would name the other one (with its own number of splits)."""
    from hqmq_amd import _lib as L
    a = _args(B, Hq, Hkv, Tq, T, d_h // 4, False, L.DT_CODE[torch.float16])
    a.idx_bits, a.main_bits, a.aux_bits = L.layout_bits(S, b_r)
    a.t_cap, a.qmax, a.softmax_scale, a.causal, a.causal_offset = (T + 63) // 64 * 64, (1 << b_r) - 1, d_h ** -0.5, 1, T - Tq
    for t in (a.K, a.V):
        t.K = 24 * S
        if med:
            t.flag_plane = t.sideband = t.sb_coord = t.sb_count = t.sb_tile_off = 16
            t.sb_cap = 64
    splits = {}
    for a.force_generic in (0, 2, 3):           # the call's own choice, the decode kernels, the prefill kernel
        splits[a.force_generic] = L.lib().hqmq_attn_splits(C.addressof(a))
    assert splits[2] != splits[3] and splits[0] == splits[3 if med else 2]


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("B,Hq,Hkv,T,Tq,S,b_r", [(8, 32, 8, 341, 17, 96, 4), (5, 28, 4, 215, 29, 192, 4), (7, 28, 4, 909, 21, 192, 6)])
def test_chunks_over_large_verbatim_keys(B, Hq, Hkv, T, Tq, S, b_r):
    """fp16 outlier caches with 2 % of K's chunks 50 to 200 times the others: a chunk of few queries takes the prefill kernel, with an error of
    0.82 to 0.84 of the decode kernels' (38 calls measured)."""
    import hqmq
    from tests.helpers import exact_dense, kv_input
    dt, d_h = torch.float16, 128
    k = kv_input((B, Hkv, T, d_h), dt, 71, lognormal=False, outlier_p=0.02).cuda()
    v = kv_input((B, Hkv, T, d_h), dt, 72, lognormal=False).cuda()
    Q = torch.randn(B, Hq, Tq, d_h, generator=torch.Generator().manual_seed(73)).to(dt).cuda()
    w = hqmq.with_outlier_extraction(hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=S, radius_bits=b_r, device="cuda"), C=3.0)
    cache = w.new_cache(B, T, d_h, dt, 0)
    w.append(cache, k, v, 0)
    out = {f: hqmq.fused_attention_packed(Q, cache, causal=True, causal_offset=T - Tq, force_generic=f) for f in (0, 2, 3)}
    seen = torch.arange(T, device="cuda").view(1, T) <= torch.arange(Tq, device="cuda").view(Tq, 1) + T - Tq
    err = {f: 0.0 for f in out}
    for b in range(B):
        K, V = (exact_dense(t, b, T, x[b]).double().repeat_interleave(Hq // Hkv, 0) for t, x in ((cache.K, k), (cache.V, v)))
        s = torch.matmul(Q[b].double(), K.transpose(1, 2).contiguous()) * d_h ** -0.5
        ref = torch.matmul(torch.softmax(s.masked_fill(~seen, float("-inf")), -1), V)
        for f in out:
            err[f] += float((out[f][b].double() - ref).square().sum())
    assert torch.equal(out[0].view(torch.int16), out[3].view(torch.int16))
    assert err[0] < 0.9 ** 2 * err[2], err


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("S,b_r,dn,d_h,med,B,contexts", [
    (96, 4, "fp16", 128, False, 1, (1, 64, 300, 640, 704, 768, 1025)), (192, 4, "fp16", 128, False, 33, (257, 1100)),
    (24, 3, "bf16", 128, True, 1, (255, 384, 385, 450)), (96, 4, "bf16", 64, True, 5, (300, 640, 1024, 1025)),
    (96, 4, "fp16", 64, False, 12, (500, 1500, 2100)), (24, 3, "fp32", 128, False, 3, (129, 600))])
def test_attention_on_both_sides_of_the_choice(S, b_r, dn, d_h, med, B, contexts):
    import hqmq
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}[dn]
    Hq, Hkv, T = 32, 8, max(contexts)
    g = torch.Generator().manual_seed(S + d_h)
    k, v = (torch.randn(B, Hkv, T, d_h, generator=g) for _ in range(2))
    if med:
        k[..., ::37, 3] = 30.0
    q = hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=S, radius_bits=b_r, device="cuda")
    if med:
        q = hqmq.with_outlier_extraction(q, C=3.0)
    cache = q.new_cache(B, T, d_h, dt, 0)
    q.append(cache, k.to(dt).cuda(), v.to(dt).cuda(), 0)
    Q = torch.randn(B, Hq, 1, d_h, generator=g).to(dt).cuda()
    for t in contexts:
        lens = torch.randint(1, t + 1, (B,), generator=g).int()
        lens[0] = t
        for kw in ({}, {"kv_lens": lens.cuda()}):
            vis = torch.arange(t).view(1, 1, 1, t) < lens.view(B, 1, 1, 1) if kw else None
            refs = masked_two_refs(cache, Q, t, None if vis is None else vis.cuda())
            for ns in (0, 1, 5):
                O = hqmq.fused_attention_packed(Q, cache, T_kv=t, n_splits=ns, **kw)
                assert_attention_close(O, *refs, base=1e-3 if dn == "fp32" else 2e-3, what=f"T={t} {list(kw)} n_splits={ns}")


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("S,b_r,dn,d_h", [(96, 4, "fp16", 128), (96, 4, "bf16", 64), (192, 4, "bf16", 128), (24, 3, "fp16", 128)])
def test_column_groups_between_one_and_two_rounds(S, b_r, dn, d_h):
    """More than 256 blocks of one column group and fewer than 256 of two: 32 (sequence, head) pairs x 9 groups, the last block's second
    group past the end; 255 and 256 tokens where the choice looks at the length too."""
    import hqmq
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dn]
    B, Hq, Hkv, Tq = 4, 32, 8, 33
    g = torch.Generator().manual_seed(S + d_h)
    k, v = (torch.randn(B, Hkv, 300, d_h, generator=g).to(dt).cuda() for _ in range(2))
    q = hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=S, radius_bits=b_r, device="cuda")
    cache = q.new_cache(B, 300, d_h, dt, 0)
    q.append(cache, k, v, 0)
    Q = torch.randn(B, Hq, Tq, d_h, generator=g).to(dt).cuda()
    for t in (40, 255, 256, 300):
        vis = (torch.arange(t).view(1, 1, 1, t) <= torch.arange(t - Tq, t).view(1, 1, Tq, 1)).cuda()
        refs = masked_two_refs(cache, Q, t, vis)
        for ns in (0, 1):
            O = hqmq.fused_attention_packed(Q, cache, T_kv=t, causal=True, causal_offset=t - Tq, n_splits=ns)
            assert_attention_close(O, *refs, base=2e-3, what=f"T={t} n_splits={ns}")


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("dn,d_h", [("fp16", 64), ("bf16", 64), ("fp16", 128), ("bf16", 128), ("fp16", 32), ("fp32", 64)])
def test_merge_of_any_number_of_splits(dn, d_h):
    """The merge kernels at the edges of their record counts, with splits that hold no token and outputs of any alignment."""
    import hqmq
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}[dn]
    g = torch.Generator().manual_seed(d_h)
    k, v = (torch.randn(2, 2, 700, d_h, generator=g).to(dt).cuda() for _ in range(2))
    q = hqmq.HQMQ(n_layers=1, n_heads=2, secondary_size=96, radius_bits=4, device="cuda")
    cache = q.new_cache(2, 700, d_h, dt, 0)
    q.append(cache, k, v, 0)
    Q = torch.randn(2, 6, 3, d_h, generator=g).to(dt).cuda()
    lens = torch.tensor([700, 90], dtype=torch.int32)
    vis = torch.arange(700).view(1, 1, 1, 700) < lens.view(2, 1, 1, 1)
    refs = masked_two_refs(cache, Q, 700, vis.cuda())
    for ns in (1, 2, 4, 5, 8, 9, 11, 32, 33, 40):
        O = hqmq.fused_attention_packed(Q, cache, T_kv=700, kv_lens=lens.cuda(), n_splits=ns)
        assert_attention_close(O, *refs, base=1e-3 if dn == "fp32" else 2e-3, what=f"n_splits={ns}")
        for first in (1, 2):
            out = torch.full((2, 6, 3, d_h + 3), 7.0, dtype=dt, device="cuda")
            hqmq.fused_attention_packed(Q, cache, T_kv=700, kv_lens=lens.cuda(), n_splits=ns, out=out[..., first:first + d_h])
            assert_attention_close(out[..., first:first + d_h], *refs, base=1e-3 if dn == "fp32" else 2e-3, what=f"n_splits={ns} at {first}")
            assert bool((out[..., :first] == 7).all()) and bool((out[..., first + d_h:] == 7).all())
