"""GPU: the row-grouped expert GEMMs at the edges of their tiles.

Expert row counts on both sides of the tile (256 rows) and of its half (a tile
of at most 128 rows runs half the matrix work), in sequences where both kinds
follow each other on one block; reductions of one k tile, of an odd number and
with a remainder; column counts that are not a multiple of the tile's. Gathered
input rows and routing weights, every output against fp64 on the same 16-bit
operands: an output is one rounding of an fp32 sum or of a short expression of
such sums, so its relative error is about 2^-9 / sqrt(3) in bf16 (2^-12 /
sqrt(3) in fp16), allowed three times over.
"""

from __future__ import annotations

import pytest
import torch

from tests._gpu_helpers import DEV, MAX_ABS_FRAC, check_close, gen, ref_grouped, say

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 4e-3, torch.float16: 5e-4}

ROWS = {
    "edges": [256, 257, 128, 129, 1, 0, 127, 64],
    "short": [33, 96, 40, 64, 128, 17, 100, 50, 128],
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H, I", [(64, 32), (136, 72), (712, 264)])
@pytest.mark.parametrize("rows", list(ROWS))
def test_row_grouped_tile_edges(rows, H, I, dtype):
    from pluggy_amd import ops

    n = ROWS[rows]
    E, P = len(n), sum(n)
    say(f"tile edges {n} H={H} I={I} {dtype}")
    g = gen(11)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(n))[torch.randperm(P, generator=g)].reshape(-1, 1)
    x = torch.randn(P, H, generator=g).to(dtype)
    gy = torch.randn(P, H, generator=g).to(dtype)
    w = (torch.rand(P, 1, generator=g) + 0.5).to(dtype)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.1).to(dtype)
    wdn = (torch.randn(E, H, I, generator=g) * 0.1).to(dtype)
    counts, offs, _, _, tok, sw = ops.permute_rows(ids.to(DEV), w.to(DEV), E)
    assert counts.cpu().tolist() == n
    o, t, ws = offs.cpu(), tok.cpu().long(), sw.cpu().double()[:, None]
    tol, mx = TOL[dtype], MAX_ABS_FRAC[dtype]

    gu, mid = ops.gate_up_swiglu(x.to(DEV), wgu.to(DEV), offs, tok, sw)
    check_close("gate_up", gu, ref_grouped(x[t], wgu, o, trans_w=True), tol, mx)
    gate, up = gu.cpu().double().chunk(2, dim=1)
    s = torch.sigmoid(gate)
    check_close("mid", mid, gate * s * up * ws, tol, mx)
    y = ops.down_proj(mid, wdn.to(DEV), offs)
    check_close("y", y, ref_grouped(mid.cpu(), wdn, o, trans_w=True), tol, mx)

    ggu, part = ops.down_proj_dgrad(gy.to(DEV), gu, wdn.to(DEV), offs, tok, sw, need_part=True)
    dm = ref_grouped(gy[t], wdn, o, trans_w=False)
    ref = torch.cat([dm * ws * up * s * (1 + gate * (1 - s)), dm * ws * gate * s], dim=1)
    check_close("dgate_up", ggu, ref, tol, mx)
    check_close("dw", part.sum(1, dtype=torch.float64), (dm * gate * s * up).sum(1), 1e-5, 1e-5)
    gx = ops.gate_up_dgrad(ggu, wgu.to(DEV), offs)
    check_close("dx_perm", gx, ref_grouped(ggu.cpu(), wgu, o, trans_w=False), tol, mx)
