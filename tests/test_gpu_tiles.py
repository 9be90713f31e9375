"""GPU: the row-grouped expert GEMMs at the edges of their tiles.

Expert row counts on both sides of the tile (256 rows) and of its half (a tile
of at most 128 rows runs half the matrix work); reductions of one k tile, of an
odd number and with a remainder; column counts that are not a multiple of the
tile's; and lists long enough that full and half tiles follow each other on a
block (one block per CU walks the tiles). Gathered input rows and routing
weights, every output against fp64 on the same 16-bit operands: an output is one
rounding of an fp32 sum or of a short expression of such sums, so its relative
error is about 2^-9 / sqrt(3) in bf16 (2^-12 / sqrt(3) in fp16), allowed three
times over.
"""

from __future__ import annotations

import pytest
import torch

from tests._gpu_helpers import DEV, MAX_ABS_FRAC, check_close, gen, ref_grouped, ref_wgrad, say

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 4e-3, torch.float16: 5e-4}

ROWS = {
    "edges": [256, 257, 128, 129, 1, 0, 127, 64],
    "short": [33, 96, 40, 64, 128, 17, 100, 50, 128],
}


# 11 tiles of both kinds (and an expert without rows) in eight experts
CHAIN = [300, 100, 140, 520, 128, 257, 0, 60]


def _check_rows(n, H, I, dtype):
    from pluggy_amd import ops

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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H, I", [(64, 32), (136, 72), (712, 264)])
@pytest.mark.parametrize("rows", list(ROWS))
def test_row_grouped_tile_edges(rows, H, I, dtype):
    _check_rows(ROWS[rows], H, I, dtype)


@pytest.mark.parametrize("H, I, dtype", [(1544, 1416, torch.bfloat16), (1544, 1416, torch.float16),
                                         (72, 1416, torch.bfloat16), (1544, 72, torch.bfloat16)])
def test_tiles_follow_each_other(H, I, dtype):
    """88 m-tiles: two to four tiles a block in the GEMMs with many columns, at
    23 to 45 k tiles, and at two (with and without gathered rows) and three."""
    _check_rows(CHAIN * 8, H, I, dtype)


def test_many_tiles_per_block():
    """66 tiles a block (at 256 blocks) wrap the 64-entry ring of tile places.
    Small integers: every output is exact."""
    from pluggy_amd import ops

    E, cols, K = 512, 8448, 8
    n = [30, 38, 34, 140] * (E // 4)
    P = sum(n)
    say(f"ring of tile places: {E} experts, {P} rows, {cols} columns")
    g = gen(3)
    ints = lambda *s: torch.randint(-4, 5, s, generator=g).bfloat16().to(DEV)  # noqa: E731
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(n))[torch.randperm(P, generator=g)].reshape(-1, 1)
    x, a, w = ints(P, K), ints(P, K), ints(E, cols, K)
    _, offs, _, _, tok, sw = ops.permute_rows(ids.to(DEV), torch.ones(P, 1, device=DEV, dtype=torch.bfloat16), E)
    y = ops.down_proj(a, w, offs)
    gu, _ = ops.gate_up_swiglu(x, w, offs, tok, sw)
    xs, lo = x[tok.long()], 0
    for e, rows in enumerate(n):
        we = w[e].float().t().contiguous()
        assert torch.equal(y[lo:lo + rows].float(), a[lo:lo + rows].float() @ we), f"down_proj, expert {e}"
        assert torch.equal(gu[lo:lo + rows].float(), xs[lo:lo + rows].float() @ we), f"gate_up, expert {e}"
        lo += rows


def _f32_case(rows, H, I, seed):
    from pluggy_amd import ops

    E, P = len(rows), sum(rows)
    g = gen(seed)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))[torch.randperm(P, generator=g)].reshape(-1, 1)
    x = torch.randn(P, H, generator=g)
    w = torch.rand(P, 1, generator=g) + 0.5
    wgu = torch.randn(E, 2 * I, H, generator=g) * 0.1
    wdn = torch.randn(E, H, I, generator=g) * 0.1
    _, offs, _, _, tok, sw = ops.permute_rows(ids.to(DEV), w.to(DEV), E)
    return ops, x, wgu, wdn, offs, tok, sw


@pytest.mark.parametrize("scale", [1.0, 1e-25, 1e25])
@pytest.mark.parametrize("H, I", [(40, 24), (512, 264)])
def test_fp32_gemms_are_fp32_exact(H, I, scale):
    """fp32 operands through their bf16 pieces: the error against fp64 is that of
    fp32 sums. A sum of n products accumulated in fp32 in any order is off by at
    most n 2^-24 of the sum of magnitudes; roundings of random sign give about
    sqrt(n) 2^-24 of the result's norm, allowed twice (the pieces left out, 2^-23
    of a product at worst, are inside that)."""
    ops, x, wgu, wdn, offs, tok, sw = _f32_case([64, 65, 1, 0, 200, 63], H, I, 5)
    x = x * scale
    say(f"fp32 GEMMs H={H} I={I} scale={scale}")
    bound = lambda n: 2.0 * max(n, 4) ** 0.5 * 2.0 ** -24  # noqa: E731
    o, t = offs.cpu(), tok.cpu().long()
    gu, _ = ops.gate_up_swiglu(x.to(DEV), wgu.to(DEV), offs, tok, sw)
    check_close("gate_up", gu, ref_grouped(x[t], wgu, o, trans_w=True), bound(H), 1e-5)
    a = x[:, :1].expand(-1, I).contiguous() * torch.linspace(0.5, 2.0, I)
    y = ops.down_proj(a.to(DEV), wdn.to(DEV), offs)
    check_close("y", y, ref_grouped(a, wdn, o, trans_w=True), bound(I), 1e-5)
    gg = torch.cat([a, -a], dim=1)
    gx = ops.gate_up_dgrad(gg.to(DEV), wgu.to(DEV), offs)
    check_close("dx_perm", gx, ref_grouped(gg, wgu, o, trans_w=False), bound(2 * I), 1e-5)
    gw = ops.gate_up_wgrad(gg.to(DEV), wgu[0, :1].expand(x.shape[0], -1).contiguous().to(DEV), offs, len(wgu))
    check_close("dgate_up", gw, ref_wgrad(gg, wgu[0, :1].expand(x.shape[0], -1).contiguous(), o), bound(200), 1e-5)


@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), float("nan")])
def test_fp32_gemms_keep_infinities(bad):
    """A row with an infinity or NaN gives the infinities and NaNs of fp32
    arithmetic, and the other rows of its tile their values."""
    H, I = 64, 40
    ops, x, wgu, wdn, offs, tok, sw = _f32_case([70, 30], H, I, 9)
    say(f"fp32 GEMMs with {bad}")
    x[17, 5] = bad
    t = tok.cpu().long()
    gu, _ = ops.gate_up_swiglu(x.to(DEV), wgu.to(DEV), offs, tok, sw)
    ref = ref_grouped(x[t], wgu, offs.cpu(), trans_w=True)
    got, fine = gu.cpu().double(), torch.isfinite(ref)
    assert torch.equal(fine, torch.isfinite(got)) and torch.equal(torch.isnan(ref), torch.isnan(got))
    assert torch.equal(ref[~fine].nan_to_num(nan=0.0), got[~fine].nan_to_num(nan=0.0))
    assert int((~fine).any(dim=1).sum()) == 1
    check_close("finite rows", got[fine], ref[fine], 1e-6, 1e-5)
