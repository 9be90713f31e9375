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

from tests._gpu_helpers import DEV, MAX_ABS_FRAC, check_close, gen, ref_grouped, ref_wgrad, rel, say

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
    23 to 45 k tiles, at two (of gathered rows) and at three."""
    _check_rows(CHAIN * 8, H, I, dtype)


def test_many_tiles_per_block():
    """66 tiles a block (at 256 blocks) wrap the 64-entry ring of tile places, without
    gathered rows at three k tiles and with them at two. Signs and zeros: every
    output is a whole number of at most 136, exact in bf16."""
    from pluggy_amd import ops

    E, cols = 512, 8448
    n = [30, 38, 34, 140] * (E // 4)
    P = sum(n)
    say(f"ring of tile places: {E} experts, {P} rows, {cols} columns")
    g, gd = gen(3), torch.Generator(device=DEV).manual_seed(3)
    signs = lambda *s: torch.randint(-1, 2, s, generator=gd, device=DEV).bfloat16()  # noqa: E731
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(n))[torch.randperm(P, generator=g)].reshape(-1, 1)
    _, offs, _, _, tok, sw = ops.permute_rows(ids.to(DEV), torch.ones(P, 1, device=DEV, dtype=torch.bfloat16), E)
    for name, K in (("down_proj", 136), ("gate_up", 8)):
        x, w = signs(P, K), signs(E, cols, K)
        if name == "down_proj":
            y, xs = ops.down_proj(x, w, offs), x
        else:
            y, xs = ops.gate_up_swiglu(x, w, offs, tok, sw)[0], x[tok.long()]
        lo = 0
        for e, rows in enumerate(n):
            ref = xs[lo:lo + rows].float() @ w[e].float().t().contiguous()
            assert torch.equal(y[lo:lo + rows].float(), ref), f"{name}, expert {e}"
            lo += rows


@pytest.mark.parametrize("I", [56, 64, 72, 128, 136])
def test_short_reductions_of_plain_gemms(I):
    """Both sides of the reduction of 128 up to which down's forward and gate_up's
    input gradient keep the persistent engine's loop: the same sums either way,
    over full and half tiles."""
    _check_rows(CHAIN, 264, I, torch.bfloat16)


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
    sqrt(n) 2^-24 of the result's norm, allowed twice (the products of pieces left
    out, 2^-24 of a product at worst and of random sign, are inside that)."""
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


def _fma_chain(a, b):
    """a^T b, (n, M) and (n, N), summed in fp32 one product after the other (each
    product exact, one rounding per sum); in fp64."""
    acc = torch.zeros(a.shape[1], b.shape[1], dtype=torch.float64)
    for k in range(a.shape[0]):
        acc = (acc + torch.outer(a[k].double(), b[k].double())).float().double()
    return acc


@pytest.mark.parametrize("same_sign", [False, True])
def test_fp32_short_reductions(same_sign):
    """Weight gradients of experts with few rows: no further from fp64 than a chain
    of fp32 additions, in the norm (the same roundings drawn otherwise: 5 % of room)
    and, where a single product is the sum, in every element (half an fp32 ulp)."""
    from pluggy_amd import ops

    rows = [1, 2, 3, 0, 4, 5, 8, 16, 31, 33, 64, 100]
    offs = torch.tensor(rows).cumsum(0).int()
    P, g = sum(rows), gen(21)
    gg, x = torch.randn(P, 128, generator=g), torch.randn(P, 192, generator=g)
    if same_sign:
        gg, x = gg.abs(), x.abs()
    say(f"fp32 short reductions, same sign: {same_sign}")
    gw = ops.gate_up_wgrad(gg.to(DEV), x.to(DEV), offs.to(DEV), len(rows)).cpu().double()
    ref = ref_wgrad(gg, x, offs)
    lo = 0
    for e, n in enumerate(rows):
        if n:
            chain = _fma_chain(gg[lo:lo + n], x[lo:lo + n])
            r, c = rel(gw[e], ref[e]), rel(chain, ref[e])
            say(f"  {n} rows: {r:.2e}, the chain's {c:.2e}")
            assert r <= 1.05 * c
        if n == 1:
            assert (((gw[e] - ref[e]) / ref[e]).abs() <= 2.0 ** -24).all()
        lo += n


@pytest.mark.parametrize("n", [1, 8, 16])
def test_fp32_products_of_full_pieces(n):
    """Operands whose pieces are as large as they get, all of one sign, so that
    whatever a product leaves out adds up. Up to 16 products are six MFMAs, of which
    the last alone adds at the sum's magnitude (the others at 2^-7 of it), in one
    step or in two of eight products: at most two fp32 ulps, 2^-22 (what products
    of truncated pieces leave out reaches 2^-21)."""
    from pluggy_amd import ops

    bits = torch.tensor([0x3F80FFFF, 0x3F807FFF, 0x3F817F7F, 0x3F80FF7F, 0x3FFF7F7F], dtype=torch.int32)
    v = bits.view(torch.float32).repeat(16)
    a = v.repeat(n, 1)
    say(f"fp32 products of full pieces, {n} rows")
    offs = torch.tensor([n], dtype=torch.int32)
    gw = ops.gate_up_wgrad(a.to(DEV), a.to(DEV), offs.to(DEV), 1).cpu().double()
    ref = ref_wgrad(a, a, offs)
    assert ((gw - ref).abs() <= 2.0 ** -22 * ref).all()


def _six_f32_gemms(ops, x, wgu, wdn, offs, tok, A, G):
    """name -> (output, fp64 reference) of the six GEMMs without routing weights: x (P, H) and
    G (P, H) gathered by tok, A (P, I) in sorted rows; the input gradient's SwiGLU sees A in both
    its halves."""
    o, t, E = offs.cpu(), tok.cpu().long(), len(wgu)
    d = lambda v: v.to(DEV)  # noqa: E731
    aa = torch.cat([A, A], dim=1)
    out = {"gate_up": (ops.gate_up_swiglu(d(x), d(wgu), offs, tok)[0], ref_grouped(x[t], wgu, o, trans_w=True)),
           "down": (ops.down_proj(d(A), d(wdn), offs), ref_grouped(A, wdn, o, trans_w=True)),
           "gate_up dgrad": (ops.gate_up_dgrad(d(aa), d(wgu), offs), ref_grouped(aa, wgu, o, trans_w=False)),
           "gate_up wgrad": (ops.gate_up_wgrad(d(aa), d(x), offs, E, row_index=tok), ref_wgrad(aa, x[t], o)),
           "down wgrad": (ops.down_proj_wgrad(d(G), d(A), offs, E, row_index=tok), ref_wgrad(G[t], A, o))}
    gate = torch.linspace(-2.0, 2.0, A.shape[1]).expand(A.shape[0], -1)
    dm, s = ref_grouped(G[t], wdn, o, trans_w=False), torch.sigmoid(gate.double())
    out["down dgrad"] = (ops.down_proj_dgrad(d(G), d(torch.cat([gate, gate + 3.0], dim=1)), d(wdn), offs, tok)[0],
                         torch.cat([dm * (gate + 3.0) * s * (1 + gate * (1 - s)), dm * gate * s], dim=1))
    return out


# of the operand rows and of the weights (and of the other operand of the weight
# gradients): below bf16's range in the last piece, below fp32's normal range,
# and where rounding to bf16 overflows
@pytest.mark.parametrize("e1, e2", [(-108, 0), (-112, 0), (-122, 10), (-126, 30), (-138, 60), (127, -40)])
def test_fp32_gemms_over_the_whole_range(e1, e2):
    """Operands near the ends of fp32's range: the error of fp32 sums, as in
    test_fp32_gemms_are_fp32_exact, in every GEMM."""
    ops, x, wgu, wdn, offs, tok, _ = _f32_case([70, 0, 5, 45], 64, 40, 13)
    g = gen(14)
    far = lambda *s: ((torch.rand(s, generator=g, dtype=torch.float64) + 0.999) * 2.0 ** e1 *  # noqa: E731
                      (torch.randint(0, 2, s, generator=g) * 2 - 1)).float()
    x, A = far(*x.shape), far(x.shape[0], 40)
    wgu, wdn = wgu * 2.0 ** e2, wdn * 2.0 ** e2
    G = (torch.randn(x.shape, generator=g) * 2.0 ** e2)
    say(f"fp32 GEMMs at 2^{e1} and 2^{e2}")
    t, o, E = tok.cpu().long(), offs.cpu(), len(wgu)
    aa = torch.cat([A, A], dim=1)
    pairs = [(ops.gate_up_swiglu(x.to(DEV), wgu.to(DEV), offs, tok)[0], ref_grouped(x[t], wgu, o, trans_w=True), 64),
             (ops.down_proj(A.to(DEV), wdn.to(DEV), offs), ref_grouped(A, wdn, o, trans_w=True), 40),
             (ops.gate_up_dgrad(aa.to(DEV), wgu.to(DEV), offs), ref_grouped(aa, wgu, o, trans_w=False), 80),
             (ops.gate_up_wgrad(torch.cat([G, G[:, :16]], 1).to(DEV), x.to(DEV), offs, E, row_index=tok),
              ref_wgrad(torch.cat([G, G[:, :16]], 1), x[t], o), 70),
             (ops.down_proj_wgrad(G.to(DEV), A.to(DEV), offs, E, row_index=tok), ref_wgrad(G[t], A, o), 70)]
    for i, (got, ref, n) in enumerate(pairs):
        check_close(f"{i}", got, ref, 2.0 * n ** 0.5 * 2.0 ** -24, 1e-5)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_fp32_gemms_confine_infinities(bad):
    """One operand value that is no finite number: every output that it enters is
    what fp32 arithmetic gives, every other one is itself, in all six GEMMs."""
    ops, x, wgu, wdn, offs, tok, _ = _f32_case([70, 30], 64, 40, 9)
    g = gen(10)
    A, G = torch.randn(100, 40, generator=g), torch.randn(100, 64, generator=g)
    x[17, 5], A[33, 7], G[61, 9] = bad, bad, bad
    say(f"fp32 GEMMs with {bad}")
    for name, (got, ref) in _six_f32_gemms(ops, x, wgu, wdn, offs, tok, A, G).items():
        got, fine = got.cpu().double(), torch.isfinite(ref)
        assert 0 < int((~fine).sum()) < ref.numel() // 4
        assert torch.equal(fine, torch.isfinite(got)), name
        if name != "down dgrad":  # (whose infinities meet the SwiGLU's factors)
            assert torch.equal(torch.isnan(ref), torch.isnan(got)), name
            assert torch.equal(ref[~fine].nan_to_num(nan=0.0), got[~fine].nan_to_num(nan=0.0)), name
        check_close(name, got[fine], ref[fine], 2e-6, 1e-5)


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
