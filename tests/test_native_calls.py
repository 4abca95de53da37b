"""The compiled host side of the calls: inputs as they come (strides, integer and float types, expanded scales) against the same values
laid out plainly, errors as exceptions, calls from several threads on streams of their own."""
import threading

import pytest
import torch

from tests.helpers import bit_equal

DEV = "cuda:0"


def test_refuses_what_is_not_a_call():
    from hqmq_amd import _lib as L
    n = L.native()
    for f in (n.codes, n.fake, n.med3x, n.append, n.dequant, n.attn, n.fused):
        with pytest.raises(TypeError):
            f()
    with pytest.raises(TypeError):
        n.dequant(1, 2, 3, 4, 5)
    with pytest.raises(ValueError):
        n.med3x(torch.zeros(3, 4), 3.0, torch.zeros(4), True)
    with pytest.raises(L.HqmqError):
        L.tensors(-2, "a call")


def _setup(dt, med, T=70):
    import hqmq
    q = hqmq.HQMQ(n_layers=1, n_heads=3, secondary_size=24, radius_bits=4, device=DEV)
    g = torch.Generator().manual_seed(7)
    k, v = (torch.randn(2, 3, T, 64, generator=g).to(dt).to(DEV) for _ in range(2))
    return (hqmq.with_outlier_extraction(q, C=2.0) if med else q), k, v


@pytest.mark.gpu
@pytest.mark.parametrize("dn", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("med", [False, True])
def test_inputs_as_they_come(dn, med):
    import hqmq
    from hqmq.kernels import decode_dequant
    dt = getattr(torch, dn)
    w, k, v = _setup(dt, med)
    plain = w.encode_K(k, 0)
    views = [k.transpose(1, 2).contiguous().transpose(1, 2), torch.nn.functional.pad(k, (3, 2))[..., 3:67], k.transpose(2, 3).contiguous().transpose(2, 3)]
    for view in views:
        assert view.stride() != k.stride()
        got = w.encode_K(view, 0)
        assert got.keys() == plain.keys()
        assert all(bit_equal(got[n], plain[n]) if plain[n].is_floating_point() else torch.equal(got[n], plain[n]) for n in plain)
        assert bit_equal(w.quantize_K(view, 0), w.quantize_K(k, 0))
        a, b = w.new_cache(2, 128, 64, dt, 0), w.new_cache(2, 128, 64, dt, 0)
        w.append(a, view, v, 0)
        w.append(b, k, v, 0)
        assert torch.equal(a.K.main, b.K.main) and torch.equal(a.V.main, b.V.main) and bit_equal(a.K.scale, b.K.scale)
    vc = w.encode_V(v, 0)
    qmax = 15
    dense = decode_dequant(plain["idx"], plain["rq"], plain["r_max"], plain["joint"], qmax)
    odd = (plain["idx"].long(), plain["rq"].to(torch.int16).transpose(0, 1).contiguous().transpose(0, 1), plain["r_max"].float(), plain["joint"])
    assert bit_equal(decode_dequant(*odd, qmax), dense)
    Q = torch.randn(2, 6, 1, 64, generator=torch.Generator().manual_seed(1)).to(dt).to(DEV)
    one = torch.ones_like(plain["r_max"][:, :, :1])
    V = (vc["idx"], vc["rq"], vc["r_max"], vc["joint"])
    want = hqmq.fused_attention(Q, plain["idx"], plain["rq"], one.expand(2, 3, 70).contiguous(), plain["joint"], *V, qmax, causal=False)
    got = hqmq.fused_attention(Q.expand(2, 6, 1, 64), odd[0], odd[1], one, plain["joint"], *V, qmax, causal=False)
    assert bit_equal(got, want)
    for lens in (torch.tensor([70, 9]), torch.tensor([70, 9], dtype=torch.int32, device=DEV)):
        O = hqmq.fused_attention_packed(Q, b, kv_lens=lens, T_kv=70)
        assert bit_equal(O, hqmq.fused_attention_packed(Q, b, kv_lens=lens.to(DEV).int(), T_kv=70, out=torch.empty_like(Q)))
        assert bit_equal(hqmq.fused_attention(Q, plain["idx"], plain["rq"], plain["r_max"], plain["joint"], *V, qmax, causal=False, kv_lens=lens),
                         hqmq.fused_attention(Q, plain["idx"], plain["rq"], plain["r_max"], plain["joint"], *V, qmax, causal=False, kv_lens=lens.to(DEV).int()))


@pytest.mark.gpu
def test_errors_are_exceptions():
    import hqmq
    from hqmq.kernels import decode_dequant
    from hqmq_amd import _lib as L, ops
    w, k, v = _setup(torch.float16, False)
    c = w.encode_K(k, 0)
    joint, slack = w._joint_and_slack(0, 0, k)
    for call in (lambda: ops.quantize(k.float(), joint, slack, 4), lambda: ops.quantize(k[:, :2], joint, slack, 4), lambda: ops.fake_quant(k[0], joint, slack, 4)):
        with pytest.raises(ValueError):
            call()
    for mult, name in ((None, "hqmq_quantize_grid"), (3.0, "hqmq_quantize_med3x_grid")):        # under the name of the call that was made
        with pytest.raises(L.HqmqError, match=name):
            ops.fake_quant(k, joint, slack, 99, mult)
    with pytest.raises(L.HqmqError):                        # a status of the library
        decode_dequant(c["idx"], c["rq"], c["r_max"], c["joint"], 0)
    with pytest.raises(L.HqmqError):
        decode_dequant(c["idx"], c["rq"], c["r_max"], c["joint"].double(), 15)
    with pytest.raises(L.HqmqError):
        ops.quantize(k.cpu(), joint, slack, 4)
    cache = w.new_cache(2, 128, 64, torch.float16, 0)
    w.append(cache, k, v, 0)
    Q = torch.zeros(2, 6, 1, 64, dtype=torch.float16, device=DEV)
    for kw in (dict(batch_order=torch.zeros(3, dtype=torch.int32, device=DEV)), dict(kv_starts=torch.zeros(1, dtype=torch.int32, device=DEV))):
        for _ in range(2):                                  # the first call works out the splits
            with pytest.raises(L.HqmqError):
                hqmq.fused_attention_packed(Q, cache, **kw)
            hqmq.fused_attention_packed(Q, cache)


@pytest.mark.gpu
def test_threads_on_streams_of_their_own():
    import hqmq
    w, k, v = _setup(torch.float16, True, T=300)
    Q = torch.randn(2, 6, 1, 64, generator=torch.Generator().manual_seed(1)).half().to(DEV)
    want = (w.encode_K(k, 0)["idx"], w.quantize_K(k, 0))
    cache = w.new_cache(2, 300, 64, torch.float16, 0)
    w.append(cache, k, v, 0)
    O = hqmq.fused_attention_packed(Q, cache, n_splits=2)
    torch.cuda.synchronize()
    bad = []

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                own = w.new_cache(2, 300, 64, torch.float16, 0)
                w.append(own, k, v, 0)
                got = w.encode_K(k, 0)["idx"], w.quantize_K(k, 0), hqmq.fused_attention_packed(Q, cache, n_splits=2), own.K.main
                torch.cuda.current_stream().synchronize()
                if not (torch.equal(got[0], want[0]) and bit_equal(got[1], want[1]) and bit_equal(got[2], O) and torch.equal(got[3], cache.K.main)):
                    bad.append(1)

    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.gpu
@pytest.mark.parametrize("S,b_r,d_h", [(96, 4, 128), (24, 3, 64), (192, 6, 64), (24, 3, 128)])
@pytest.mark.parametrize("B,T,Tq,n_splits", [(1, 70, 1, 0), (2, 700, 1, 5), (1, 300, 300, 0), (3, 200, 7, 1), (9, 65, 40, 2)])
def test_unpacked_bf16_scales_of_any_size(S, b_r, d_h, B, T, Tq, n_splits):
    """V scales times a power of two: the outputs times the same power, whichever kernel the GPU lets run.  Each kernel keeps
    to 2e-3 plus fp16 noise (8 * 2^-11 of the attention-weighted |V|, about 1 here) of exact arithmetic, and each output is rounded to
    bf16 once, by half a unit in the last place, which is 2^-8 of the value at most."""
    import hqmq
    dt = torch.bfloat16
    q = hqmq.HQMQ(n_layers=1, n_heads=2, secondary_size=S, radius_bits=b_r, device=DEV)
    g = torch.Generator().manual_seed(T)
    k, v = (torch.randn(B, 2, T, d_h, generator=g).to(dt).to(DEV) for _ in range(2))
    Q = torch.randn(B, 8, Tq, d_h, generator=g).to(dt).to(DEV)
    ck, cv = q.encode_K(k, 0), q.encode_V(v, 0)
    qmax = (1 << b_r) - 1

    def attend(power):
        return hqmq.fused_attention(Q, ck["idx"], ck["rq"], ck["r_max"], ck["joint"], cv["idx"], cv["rq"], cv["r_max"] * 2.0 ** power, cv["joint"], qmax,
                                    causal=Tq > 1, n_splits=n_splits)

    want = attend(0).float()
    for power in (20, -30, 13, -7, 60, -60):
        got = attend(power).float() * 2.0 ** -power
        assert bool(((got - want).abs() <= 1.2e-2 + 2.0 ** -7 * want.abs()).all()), (power, float((got - want).abs().max()))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = attend(20)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert bool(((out.float() * 2.0 ** -20 - want).abs() <= 1.2e-2 + 2.0 ** -7 * want.abs()).all())


@pytest.mark.gpu
@pytest.mark.parametrize("S", [24, 192, 213])
@pytest.mark.parametrize("dn", ["float16", "bfloat16"])
def test_prefill_over_tables_of_any_alignment(dn, S):
    """Tables read two codewords at a time, and tables that cannot be: an odd number of codewords, a base on 8 bytes."""
    import hqmq
    dt, T, qmax = getattr(torch, dn), 700, 15                # long enough for the prefill kernels
    g = torch.Generator().manual_seed(S)
    Q = torch.randn(4, 16, T, 128, generator=g).to(dt).to(DEV)
    joint = torch.nn.functional.normalize(torch.randn(2, 24 * S, 4, generator=g), dim=-1).to(dt).to(DEV)
    codes = [[torch.randint(1, hi, (4, 2, T, 32), generator=g).int().to(DEV) for hi in (24 * S, qmax + 1)] for _ in range(2)]
    rs = (torch.rand(4, 2, T, generator=g) + 0.5).to(dt).to(DEV)
    (ki, kr), (vi, vr) = codes

    def attend(table, first):
        return hqmq.fused_attention(Q, ki - first, kr, rs, table, vi - first, vr, rs, table, qmax)

    want = attend(joint, 0)
    assert bit_equal(attend(joint[:, 1:], 1), want) and bit_equal(attend(joint[:, 1:].contiguous(), 1), want)
    assert bit_equal(attend(torch.nn.functional.pad(joint, (0, 0, 1, 0))[:, 1:], 0), want)


@pytest.mark.gpu
@pytest.mark.parametrize("d_h", [64, 128])
@pytest.mark.parametrize("dn", ["float16", "bfloat16"])
def test_prefill_queries_and_outputs_of_any_alignment(dn, d_h):
    """Rows of Q and O aligned to 16 bytes and to 8: the same bits."""
    import hqmq
    dt = getattr(torch, dn)
    q = hqmq.HQMQ(n_layers=1, n_heads=2, secondary_size=96, radius_bits=4, device=DEV)
    g = torch.Generator().manual_seed(d_h)
    k, v = (torch.randn(2, 2, 150, d_h, generator=g).to(dt).to(DEV) for _ in range(2))
    cache = q.new_cache(2, 150, d_h, dt, 0)
    q.append(cache, k, v, 0)
    Q = torch.randn(2, 6, 90, d_h, generator=g).to(dt).to(DEV)
    kw = dict(causal=True, causal_offset=60, force_generic=3)
    for n_splits in (1, 2):
        want = hqmq.fused_attention_packed(Q, cache, n_splits=n_splits, **kw)
        odd_q = torch.nn.functional.pad(Q, (4, 0))[..., 4:]
        out = torch.full((2, 6, 90, d_h + 4), 7.0, dtype=dt, device=DEV)
        assert odd_q.data_ptr() % 16 == 8 and odd_q.stride(2) * 2 % 16 == 8
        assert bit_equal(hqmq.fused_attention_packed(odd_q, cache, n_splits=n_splits, **kw), want)
        hqmq.fused_attention_packed(Q, cache, n_splits=n_splits, out=out[..., :d_h], **kw)
        assert bit_equal(out[..., :d_h].contiguous(), want) and bool((out[..., d_h:] == 7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("generic", [0, 2])
@pytest.mark.parametrize("dn,d_h,med", [("float16", 64, False), ("bfloat16", 64, True), ("float16", 128, False), ("bfloat16", 128, True)])
def test_decode_queries_and_outputs_of_any_alignment(dn, d_h, med, generic):
    """The same of the kernels for few columns: 3 and 15 of them, a part of a second group, one and two splits."""
    import hqmq
    dt = getattr(torch, dn)
    q = hqmq.HQMQ(n_layers=1, n_heads=2, secondary_size=96, radius_bits=4, device=DEV)
    q = hqmq.with_outlier_extraction(q, C=2.0) if med else q
    g = torch.Generator().manual_seed(d_h)
    k, v = (torch.randn(2, 2, 150, d_h, generator=g).to(dt).to(DEV) for _ in range(2))
    cache = q.new_cache(2, 150, d_h, dt, 0)
    q.append(cache, k, v, 0)
    for Tq in (1, 5, 7):
        Q = torch.randn(2, 6, Tq, d_h, generator=g).to(dt).to(DEV)
        kw = dict(causal=True, causal_offset=150 - Tq, force_generic=generic)
        for n_splits in (1, 2):
            want = hqmq.fused_attention_packed(Q, cache, n_splits=n_splits, **kw)
            odd_q = torch.nn.functional.pad(Q, (4, 0))[..., 4:]
            assert odd_q.data_ptr() % 16 == 8
            assert bit_equal(hqmq.fused_attention_packed(odd_q, cache, n_splits=n_splits, **kw), want)
            for first in (0, 1, 4):
                out = torch.full((2, 6, Tq, d_h + 5), 7.0, dtype=dt, device=DEV)
                hqmq.fused_attention_packed(Q, cache, n_splits=n_splits, out=out[..., first:first + d_h], **kw)
                assert bit_equal(out[..., first:first + d_h].contiguous(), want)
                assert bool((out[..., :first] == 7).all()) and bool((out[..., first + d_h:] == 7).all())
