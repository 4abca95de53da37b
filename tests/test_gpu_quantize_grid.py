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
    from hqmq_amd import ops
    dt = DT[dn]
    g = torch.Generator().manual_seed(S)
    raw = _raw(S, crowded, g)
    J, slack = ops.build_joint(raw.to(DEV), dt)
    assert hasattr(slack, "hqmq_grid") == (S <= 341)
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
