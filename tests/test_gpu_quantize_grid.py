"""The cell-list search against the exhaustive scan and the CPU oracle, at the sizes where it can go wrong: one secondary,
the largest codebook with lists (341) and the first without (342), codewords crowded round the Hurwitz units, call sizes
on both sides of a wavefront, a block of four and a round of the long kernel, rows that cannot be read as vectors."""
import pytest
import torch

from oracle import c_oracle as CO
from tests.helpers import bit_equal

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _raw(S, crowded, g):
    raw = torch.randn(2, S, 4, generator=g)
    if crowded:                       # every secondary next to a unit: one cell of the grid sees all of them
        raw = torch.eye(4)[torch.arange(S) % 4] + 0.05 * raw
    return raw


@pytest.mark.parametrize("dn", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("S,crowded", [(1, False), (24, True), (96, False), (341, False), (341, True), (342, False)])
def test_cell_lists_pick_what_the_scan_picks(S, crowded, dn):
    from hqmq_amd import _lib, ops
    dt = DT[dn]
    g = torch.Generator().manual_seed(S)
    raw = _raw(S, crowded, g)
    J, slack = ops.build_joint(raw.to(DEV), dt)
    assert hasattr(slack, "hqmq_grid") == (S <= 341)
    if S <= 341:                            # the lists alone are kept (2 heads): no memory of the build behind them
        kept = _lib.lib().hqmq_search_grid_kept_bytes(2, S, _lib.DT_CODE[dt])
        assert slack.hqmq_grid.numel() == slack.hqmq_grid.untyped_storage().nbytes() == kept
    for T, d_h in ((1, 128), (2, 128), (3, 80), (8, 128), (9, 128), (33, 128), (70, 64), (5, 1024), (300, 160)):
        x = torch.randn(1, 2, T, d_h, generator=g)
        x[:, :, T // 2, :4] = J[0, 0].float().cpu()          # a codeword, a zero chunk, a chunk on a unit, one between two units
        x[:, :, T // 2, 4:8] = 0
        x[:, :, T // 2, 8:12] = torch.tensor([0.0, -2.0, 0.0, 0.0])
        x[:, :, T // 2, 12:16] = torch.tensor([0.5, 0.5, 0.0, 0.0])
        x = x.to(dt)
        for view in (x.to(DEV), torch.nn.functional.pad(x, (1, 2)).to(DEV)[..., 1:1 + d_h]):
            a = ops.quantize(view, J, slack, 4, want_dense=True)
            b = ops.quantize(view, J, slack, 4, want_dense=True, algo=1)
            c = ops.quantize(view, J, slack.clone(), 4, want_dense=True)          # without lists: the scan over the secondaries
            for other in (b, c):
                assert torch.equal(a["idx"], other["idx"]) and torch.equal(a["rq"], other["rq"]), (T, d_h)
                assert bit_equal(a["out"], other["out"]) and bit_equal(a["r_max"], other["r_max"]), (T, d_h)
    want = CO.quantize(x, CO.joint_table(raw, dt), 4)
    assert torch.equal(a["idx"].cpu(), want["idx"]) and torch.equal(a["rq"].cpu(), want["rq"]) and bit_equal(a["out"], want["out"])


@pytest.mark.parametrize("dn", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("S", [192, 341])
def test_unordinary_chunks_in_boxes_without_a_list(S, dn):
    """Directions that do not have length 1 (norm below the clamp, 16-bit subnormal, infinite, NaN) score all rows, also where
    their box carries no list: codebooks crowded round the units leave the boxes at the cell's centre without one."""
    import hqmq
    from hqmq_amd import ops
    dt = DT[dn]
    if S == 192:
        raw = hqmq.HQMQ(n_layers=1, n_heads=2, secondary_size=S, init="hurwitz_perturbed", device="cpu").secondary_raw.detach()[0, :, 0]
    else:
        raw = _raw(S, True, torch.Generator().manual_seed(S))
    J, slack = ops.build_joint(raw.to(DEV), dt)
    units = hqmq.HQMQ(n_layers=1, n_heads=2, device="cpu")._primary.float()
    x = torch.randn(1, 2, 96, 128, generator=torch.Generator().manual_seed(S + 1))
    gains = (1e-9, 3e-9, 4e-9, 6e-8, 1.2e-7, 1e-30, float("inf"), float("nan"))
    for i, gain in enumerate(gains):
        rows = x[:, :, 8 * i:8 * i + 6]
        rows[..., :96] = (units * gain).nan_to_num(nan=float("nan") if gain != gain else 0.0, posinf=float("inf"), neginf=float("-inf")).reshape(-1)
        rows[..., 96:] = (torch.tensor([[1.2, 0.6, 0, 0]] * 8) * (gain if gain < 1 else 1e-7)).reshape(-1)      # subnormal ratios: between two units
    x = x.to(dt)
    want = CO.quantize(x, CO.joint_table(raw, dt), 4)
    assert not (want["idx"] == 24 * S - 1).all()
    for t in (96, 8, 1):                    # a block's copy of the table, a block of four wavefronts, one wavefront
        for t0 in range(0, 96, t if t > 1 else 8):
            part = x[:, :, t0:t0 + t].to(DEV)
            got = ops.quantize(part, J, slack, 4, want_dense=True)
            scan = ops.quantize(part, J, slack, 4, want_dense=True, algo=1)
            ref = {k: want[k][:, :, t0:t0 + t] for k in ("idx", "rq", "r_max", "out")}
            assert torch.equal(scan["idx"].cpu(), ref["idx"]), (t, t0)
            assert torch.equal(got["idx"].cpu(), ref["idx"]) and torch.equal(got["rq"].cpu(), ref["rq"]), (t, t0)
            assert bit_equal(got["out"], ref["out"]) and bit_equal(got["r_max"], ref["r_max"]), (t, t0)


def _border_directions(n, g):
    """Unit quaternions on and next to the borders of the search's boxes (27 per axis of the stereographic cube), turned by every
    axis unit, some with equal or vanishing components."""
    scale = (13.5 - 0.1) / 0.41422
    z = (torch.randint(-14, 14, (n, 3), generator=g) + 0.5) / scale + torch.randn(n, 3, generator=g) * 10.0 ** -torch.randint(2, 7, (n, 1), generator=g)
    z = torch.where(torch.rand(n, 3, generator=g) < 0.1, torch.zeros(()), z).clamp(-0.4142, 0.4142)
    z = torch.where(torch.rand(n, 1, generator=g) < 0.1, z[:, :1].expand(n, 3), z)
    s = (z * z).sum(1, keepdim=True)
    w = torch.cat([(1 - s) / (1 + s), 2 * z / (1 + s)], 1)
    turned = torch.stack([w, torch.stack([-w[:, 1], w[:, 0], -w[:, 3], w[:, 2]], 1), torch.stack([-w[:, 2], w[:, 3], w[:, 0], -w[:, 1]], 1),
                          torch.stack([-w[:, 3], -w[:, 2], w[:, 1], w[:, 0]], 1)])
    u = turned[torch.randint(0, 4, (n,), generator=g), torch.arange(n)]
    return u * (1 - 2 * torch.randint(0, 2, (n, 1), generator=g))


@pytest.mark.parametrize("dn", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("H,S,T,d_h", [(8, 96, 1100, 128), (3, 24, 2500, 64), (2, 341, 1500, 96)])
def test_box_borders_and_many_rounds(H, S, T, d_h, dn):
    """Long calls: blocks of several rounds, with heads that fill the XCDs evenly and heads that do not; norms from ordinary down to
    where a wavefront leaves the short forms (16-bit subnormals), mixed with whole wavefronts that take them."""
    from hqmq_amd import ops
    dt = DT[dn]
    g = torch.Generator().manual_seed(S + H)
    J, slack = ops.build_joint(torch.randn(H, S, 4, generator=g).to(DEV), dt)
    u = _border_directions(H * T * d_h // 4, g)
    gain = torch.where(torch.rand(H * T, 1, generator=g) < 0.05, 10.0 ** -(3 + 4 * torch.rand(H * T, 1, generator=g)), 0.2 + 4 * torch.rand(H * T, 1, generator=g))
    x = (u.view(H * T, -1) * gain).view(1, H, T, d_h).to(dt).to(DEV)
    got = ops.quantize(x, J, slack, 4, want_dense=True)
    scan = ops.quantize(x, J, slack.clone(), 4, want_dense=True)
    assert hasattr(slack, "hqmq_grid")
    assert torch.equal(got["idx"], scan["idx"]) and torch.equal(got["rq"], scan["rq"])
    assert bit_equal(got["out"], scan["out"]) and bit_equal(got["r_max"], scan["r_max"])
