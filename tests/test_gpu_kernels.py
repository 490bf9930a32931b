"""Each HIP kernel alone against its plain reference (the functions of
tests/plain/reference_model.py, or float64 library routines), at sizes other
than the engine's tiny models use: widths and vocabularies that are no powers
of two, head sizes in steps of 16, odd head counts and groups."""
import math

import numpy as np
import pytest
import torch

from plain import reference_model as R

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


def K():
    from yalm_amd.ops import kernels
    return kernels


def rnd(shape, seed, dtype=torch.float32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g, dtype=torch.float64) * scale).to(dtype)


def tol(dtype):
    return 2e-5 if dtype == torch.float32 else 1.2e-2


ACTS = ["silu", "gelu"]


def gate(act):
    """The plain activation and the epilogue code of a gated product."""
    k = K()
    return {"silu": (R.silu, k.EPI_GATED), "gelu": (R.gelu, k.EPI_GATED_GELU)}[act]


def close(got, want, dtype, what, factor=1.0):
    got = got.detach().to("cpu", torch.float64)
    want = want.to(torch.float64)
    assert torch.isfinite(got).all(), what
    err = (got - want).abs().max().item()
    lim = factor * tol(dtype) * max(1.0, want.abs().max().item())
    assert err <= lim, "%s: max error %.3e, allowed %.3e" % (what, err, lim)


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


# The cache's pages as the kernels store them.  Head sizes that are multiples of 32 are kept in blocks:
# keys [element // 32][place(row)][element % 32], values [row // 32][element][row % 32], where place(row) is
# the row's place in the order in which the matrix-core decode attention takes the rows of a page
# (16 rows an instruction: rows 8 a + b (+ 4) (+ 32) for a, b < 4).  Other head sizes: keys [row][element],
# values [element][row], which is also how the tests fill and read pages.
def row_place(r):
    return 16 * (2 * (r >> 5) + ((r >> 2) & 1)) + 4 * ((r >> 3) & 3) + (r & 3)


def pages_as_stored(kp, vp):
    """[pages, heads, 64, hd] keys and [pages, heads, hd, 64] values in rows -> the same shapes in storage order."""
    P, H, R, hd = kp.shape
    if hd % 32:
        return kp, vp
    place = torch.tensor([row_place(r) for r in range(R)], device=kp.device)
    ks = torch.empty_like(kp).view(P, H, hd // 32, R, 32)
    ks[:, :, :, place, :] = kp.view(P, H, R, hd // 32, 32).permute(0, 1, 3, 2, 4)
    vs = vp.view(P, H, hd, R // 32, 32).permute(0, 1, 3, 2, 4).contiguous()
    return ks.view(P, H, R, hd), vs.view(P, H, hd, R)


def pages_as_rows(kp, vp):
    """The inverse of pages_as_stored."""
    P, H, R, hd = kp.shape
    if hd % 32:
        return kp, vp
    place = torch.tensor([row_place(r) for r in range(R)], device=kp.device)
    kr = kp.view(P, H, hd // 32, R, 32)[:, :, :, place, :].permute(0, 1, 3, 2, 4).contiguous().view(P, H, R, hd)
    vr = vp.view(P, H, R // 32, hd, 32).permute(0, 1, 3, 2, 4).contiguous().view(P, H, hd, R)
    return kr, vr


def test_page_layout_helpers_invert_each_other():
    assert sorted(row_place(r) for r in range(64)) == list(range(64))
    assert [row_place(r) for r in (0, 1, 4, 8, 32, 63)] == [0, 1, 16, 4, 32, 63]
    for hd in (16, 64, 128):
        kp, vp = rnd((3, 2, 64, hd), 1), rnd((3, 2, hd, 64), 2)
        ks, vs = pages_as_stored(kp, vp)
        assert (hd % 32 != 0) == torch.equal(ks, kp)
        a, b = pages_as_rows(ks, vs)
        assert torch.equal(a, kp) and torch.equal(b, vp)
        if hd % 32 == 0:        # the formula of the layout, element by element
            for (r, e) in ((0, 0), (5, 33), (63, hd - 1), (36, 31)):
                assert ks[1, 1].reshape(-1)[((e // 32) * 64 + row_place(r)) * 32 + e % 32] == kp[1, 1, r, e]
                assert vs[1, 1].reshape(-1)[((r // 32) * hd + e) * 32 + r % 32] == vp[1, 1, e, r]


# ------------------------------------------------------------------ embedding, norm

@pytest.mark.parametrize("dtype", DTYPES)
def test_embed(dtype):
    V, D = 37, 50
    table = rnd((V, D), 1, dtype)
    tokens = [0, 36, 5, 5, -1, 12]
    out = torch.full((len(tokens), D), 7.0, device=DEV)
    K().embed(table.to(DEV), i32(tokens), out)
    want = R.embedding(table, torch.tensor([t if t >= 0 else 0 for t in tokens]))
    want[4] = 0
    assert torch.equal(out.cpu().double(), want)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D,T", [(1028, 1), (2052, 5), (4096, 7), (8192, 3), (1536, 300)])
def test_embed_and_norm_in_one(D, T, dtype):
    """The bits of the two kernels, in both outputs; tokens outside the table give zeros."""
    V = 37
    table, w = rnd((V, D), 1, dtype).to(DEV), (1 + 0.1 * rnd((D,), 3)).to(DEV)
    tokens = i32([(5 * t) % V if t % 4 != 1 else (-1, V)[t % 8 == 1] for t in range(T)])
    raw, want, x, kept, alone = (torch.full((T, D), 7.0, device=DEV) for _ in range(5))
    assert K().embed_norm_fits(table, w, x, kept)
    K().embed(table, tokens, raw)
    K().rmsnorm(raw, w, want, 1e-3)
    K().embed_norm(table, tokens, w, 1e-3, x, kept)
    K().embed_norm(table, tokens, w, 1e-3, alone)
    assert torch.equal(x, want) and torch.equal(kept, want) and torch.equal(alone, want)


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("N,Kd", [(16, 64), (40, 128), (1000, 576), (4096, 4096), (1024, 14336)])
def test_two_products_in_one_launch(M, N, Kd):
    """The bits of each product alone (up to 4,096 weight rows one kernel serves both), against 64 bits too: K products of bfloat16 are
    exact in float32, and a sum of K of them in any order is off by at most K units in the last place of the sum of their sizes."""
    a, a2, w, w2 = (rnd((r, Kd), s, torch.bfloat16) for r, s in ((M, 1), (M, 2), (N, 3), (N, 4)))
    dev = [t.to(DEV) for t in (a, w, a2, w2)]
    out, out2, alone, alone2 = (torch.full((M, N), float("nan"), device=DEV) for _ in range(4))
    assert K().gemm_pair_fits(*dev)
    K().gemm_pair(dev[0], dev[1], out, dev[2], dev[3], out2)
    K().gemm(dev[0], dev[1], alone, K().EPI_STORE_F32)
    K().gemm(dev[2], dev[3], alone2, K().EPI_STORE_F32)
    assert torch.equal(out, alone) and torch.equal(out2, alone2)
    for got, x, y in ((out, a, w), (out2, a2, w2)):
        x, y = x.double(), y.double()
        assert bool(((got.cpu().double() - x @ y.t()).abs() <= Kd * 2.0 ** -24 * (x.abs() @ y.abs().t())).all())


def test_two_products_what_is_taken():
    t = lambda r, c, dt=torch.bfloat16: torch.zeros(r, c, dtype=dt, device=DEV)
    fits = lambda M, N, Kd, dt=torch.bfloat16: K().gemm_pair_fits(t(M, Kd, dt), t(N, Kd, dt), t(M, Kd, dt), t(N, Kd, dt))
    assert fits(16, 4096, 64) and not fits(17, 64, 64) and not fits(1, 4097, 64) and not fits(1, 64, 72) and not fits(1, 64, 64, torch.float32)
    assert not K().gemm_pair_fits(t(1, 64), t(32, 64), t(1, 64), t(16, 64))
    off = torch.zeros(64 * 16 + 8, dtype=torch.bfloat16, device=DEV)[1:1 + 64 * 16].view(16, 64)
    assert not K().gemm_pair_fits(t(1, 64), off, t(1, 64), t(16, 64))


def test_embed_and_norm_what_is_taken():
    flat = torch.zeros(8200, device=DEV)
    fits = lambda D, at=0: K().embed_norm_fits(flat, flat, flat[at:at + D].view(1, D))
    assert [fits(D) for D in (1024, 1026, 1028, 8192, 8196)] == [False, False, True, True, False] and not fits(2048, 1)


@pytest.mark.parametrize("out_dtype", DTYPES)
@pytest.mark.parametrize("w_dtype", DTYPES)
@pytest.mark.parametrize("D", [50, 1000, 4100, 4096, 8192, 8196, 2050])
def test_rmsnorm(D, w_dtype, out_dtype):
    x = rnd((7, D), 2, scale=3.0)
    w = (1 + 0.1 * rnd((D,), 3)).to(w_dtype)
    out = torch.empty((7, D), dtype=out_dtype, device=DEV)
    K().rmsnorm(x.to(DEV), w.to(DEV), out, 1e-3)
    close(out, R.rmsnorm(x, w, 1e-3), out_dtype, "rmsnorm")
    # gathered rows, one of them padding
    idx = [6, 0, -1, 3]
    out = torch.empty((4, D), dtype=out_dtype, device=DEV)
    K().rmsnorm(x.to(DEV), w.to(DEV), out, 1e-3, i32(idx))
    want = R.rmsnorm(x[[6, 0, 0, 3]], w, 1e-3)
    want[2] = 0
    close(out, want, out_dtype, "rmsnorm rows")
    # eps inside the root, added to the mean: ones with eps 3 -> 1/2
    one = torch.ones((1, D), device=DEV)
    out = torch.empty((1, D), dtype=torch.float32, device=DEV)
    K().rmsnorm(one, torch.ones(D, device=DEV), out, 3.0)
    assert torch.allclose(out.cpu(), torch.full((1, D), 0.5))


# ------------------------------------------------------------------ GEMM

# more than 64 rows: K a multiple of 64 takes the kernels that load straight into LDS (128x128 tiles up to 159 rows,
# 256-row tiles in a ring of LDS slots from 160), any other K the register-staged one
GEMM_SHAPES = [(1, 16, 256), (3, 70, 96), (64, 130, 264), (65, 64, 80), (200, 333, 1000), (8, 4096 + 16, 136),
               (130, 100, 50), (65, 64, 64), (200, 333, 1024), (300, 20480 + 8, 128), (513, 130, 192),
               # K a multiple of 64 (operands staged in LDS by DMA): few and odd rows, every row count of a stage
               (5, 70, 192), (16, 4112, 128), (9, 100, 64), (12, 33, 320), (8, 26000, 64), (13, 13000, 128),
               (3, 4096, 1024), (20, 70, 192), (33, 4112, 128), (50, 100, 64), (64, 333, 320),
               # widths of the big models' projections and rows that end inside a tile
               (8, 3072, 128), (5, 6144, 64), (16, 5120, 192), (3, 2048, 64), (7, 1000, 64), (9, 6010, 128),
               (1, 3080, 256), (12, 4100, 64)]


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,Kd", GEMM_SHAPES)
def test_gemm_store_and_add(M, N, Kd, dtype, simple):
    k = K()
    a = rnd((M, Kd), 4, dtype)
    w = rnd((N, Kd), 5, dtype, scale=1 / math.sqrt(Kd))
    want = a.double() @ w.double().T
    k.FORCE_SIMPLE = simple
    try:
        out = torch.empty((M, N), dtype=torch.float32, device=DEV)
        k.gemm(a.to(DEV), w.to(DEV), out, k.EPI_STORE_F32)
        close(out, want, torch.float32, "gemm f32 out", factor=4 if dtype == torch.float32 else 1)
        out2 = torch.empty((M, N), dtype=dtype, device=DEV)
        k.gemm(a.to(DEV), w.to(DEV), out2, k.EPI_STORE)
        close(out2, want, dtype, "gemm store")
        res = rnd((M, N), 6)
        acc = res.to(DEV).clone()
        k.gemm(a.to(DEV), w.to(DEV), acc, k.EPI_ADD_F32)
        close(acc, want + res.double(), torch.float32, "gemm add", factor=4 if dtype == torch.float32 else 1)
    finally:
        k.FORCE_SIMPLE = False


# (rows, columns or hidden width, K, epilogue): prompt-step shapes with one, two and three k tiles and many, rows and columns that end
# inside a tile, many row tiles, with the workspace in which K may be split and without.  (Every way the launcher goes, asked for by
# name: test_gemm_of_every_tiling.)
PROMPT_GEMMS = [(2048, 6144, 192, "f32"), (2048, 4096, 256, "add"), (1000, 4100, 320, "bf16"),
                (2048, 14336, 128, "gated"), (2048, 28672, 128, "f32"), (512, 4096, 4096, "add"),
                (384, 1000, 2048, "gated"), (160, 4096, 2048, "f32"), (8192, 512, 64, "f32"), (300, 700, 128, "add"),
                (257, 513, 192, "bf16"), (161, 96, 704, "gated"), (4096, 8192, 64, "bf16"), (700, 24000, 256, "add")]


@pytest.mark.parametrize("with_workspace", [True, False])
@pytest.mark.parametrize("M,N,Kd,epi", PROMPT_GEMMS)
def test_gemm_of_prompt_steps(M, N, Kd, epi, with_workspace):
    k = K()
    from yalm_amd.parts.swiglu import interleave_gate_up
    a = rnd((M, Kd), 91, torch.bfloat16).to(DEV)
    if epi in ("gated", "gelu"):
        H = N
        wg = rnd((H, Kd), 92, torch.bfloat16, scale=1 / math.sqrt(Kd))
        wu = rnd((H, Kd), 93, torch.bfloat16, scale=1 / math.sqrt(Kd))
        w = interleave_gate_up(wg, wu).to(DEV)
        rows = w.shape[0]
        ad = a.double()
        act_fn, epi_code = gate("gelu" if M == 384 or epi == "gelu" else "silu")
        want = (act_fn(ad @ wg.to(DEV).double().T) * (ad @ wu.to(DEV).double().T)).cpu()
    else:
        w = rnd((N, Kd), 92, torch.bfloat16, scale=1 / math.sqrt(Kd)).to(DEV)
        rows = N
        want = (a.double() @ w.double().T).cpu()
    floats = k.gemm_workspace_floats(M, rows, Kd) if with_workspace else 0
    ws = torch.full((floats,), float("nan"), device=DEV) if floats else None
    if epi in ("gated", "gelu"):
        out = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
        k.gemm(a, w, out, epi_code, hidden=N, workspace=ws)
        close(out, want, torch.bfloat16, "gated", factor=2.0)
    elif epi == "f32":
        out = torch.full((M, N), float("nan"), device=DEV)
        k.gemm(a, w, out, k.EPI_STORE_F32, workspace=ws)
        close(out, want, torch.float32, "float32 out")
    elif epi == "bf16":
        out = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
        k.gemm(a, w, out, k.EPI_STORE, workspace=ws)
        close(out, want, torch.bfloat16, "bfloat16 out")
    else:
        res = rnd((M, N), 94)
        out = res.to(DEV).clone()
        k.gemm(a, w, out, k.EPI_ADD_F32, workspace=ws)
        close(out, want + res.double(), torch.float32, "residual add")


# Every way of the launcher's plan, as yalm_gemm_bf16_dma_choice names it: the tilings whole and in slices of K, and whole rounds of 256 x 256
# tiles with a second launch of each narrower tiling behind them; rows and columns that end inside a tile, fewer k tiles than the ring
# has stages and many.  The first shape for products that are stored, the second for those added to the residual stream.
EVERY_TILING = {
    "256 x 256": (10, (257, 24608, 192), (257, 24608, 192)), "256 x 256 in slices": (30, (193, 16416, 5120), (129, 16416, 5120)),
    "256 x 256, one k tile": (10, (2000, 6176, 64), (2000, 6176, 64)),
    "256 x 192": (11, (257, 21920, 64), (257, 21920, 64)), "256 x 192 in slices": (21, None, (193, 16448, 3072)),
    "256 x 128": (12, (193, 16416, 64), (193, 16416, 64)), "256 x 128 in slices": (42, (193, 5536, 5120), None),
    "256 x 128 in three slices": (32, None, (193, 8224, 3072)), "192 x 128": (13, (129, 16448, 64), (129, 16448, 64)),
    "192 x 128 in slices": (43, (129, 5408, 3072), (129, 5408, 3072)), "128 x 128": (14, (129, 10944, 64), (129, 10944, 64)),
    "128 x 128 in slices": (44, (130, 32, 1536), (130, 32, 1536)), "64 x 128": (15, (129, 32, 64), (129, 32, 64)),
    "64 x 128 in slices": (35, (129, 32, 1280), (129, 32, 1280)),
    "and 256 x 128": (1012, (769, 22944, 768), (769, 22944, 960)), "and 192 x 128": (1013, (769, 21024, 512), (513, 28352, 768)),
    "and 128 x 128": (1014, (769, 18848, 320), (513, 25536, 512)), "and 64 x 128": (1015, (513, 21824, 320), (769, 16416, 320))}


@pytest.mark.parametrize("way,epi", [(way, epi) for way in sorted(EVERY_TILING) for epi in ("f32", "bf16", "add", "gated", "gelu", "biased")
                                     if EVERY_TILING[way][2 if epi == "add" else 1] is not None])
def test_gemm_of_every_tiling(way, epi):
    from yalm_amd.ops import library
    taken, stored, added = EVERY_TILING[way]
    M, N, Kd = added if epi == "add" else stored
    k = K()
    choice = library.lib().yalm_gemm_bf16_dma_choice(M, N, Kd, k.gemm_workspace_floats(M, N, Kd), 1 if epi == "add" else 0)
    assert choice == taken, choice
    if epi != "biased":
        return test_gemm_of_prompt_steps(M, N // 2 if epi in ("gated", "gelu") else N, Kd, epi, True)
    from yalm_amd.parts.swiglu import interleave_gate_up
    H, D = N // 2, 51
    h, wg, wu = (rnd(size, s, torch.bfloat16, scale=f) for size, s, f in (((M, Kd), 91, 1.0), ((H, Kd), 92, Kd ** -0.5), ((H, Kd), 93, Kd ** -0.5)))
    bg, bu, x, xb = rnd((H,), 94), rnd((H,), 95), rnd((M, D), 96), rnd((D,), 97)
    hd, out, xd = h.to(DEV), torch.full((M, H), float("nan"), dtype=torch.bfloat16, device=DEV), x.to(DEV)
    n = k.gemm_workspace_floats(M, N, Kd)
    k.gemm_gated_bias(hd, interleave_gate_up(wg, wu).to(DEV), interleave_gate_up(bg[:, None], bu[:, None]).reshape(-1).contiguous().to(DEV), out, xd,
                      xb.to(DEV), workspace=torch.full((n,), float("nan"), device=DEV) if n else None)
    g, u = (hd.double() @ w.to(DEV).double().T + b.to(DEV).double() for w, b in ((wg, bg), (wu, bu)))
    close(out, (R.gelu(g) * u).cpu(), torch.bfloat16, "biased", factor=2.0)
    assert torch.equal(xd.cpu(), x + xb)


@pytest.mark.parametrize("M,N,tiling", [(200, 16400, 2), (150, 16400, 3), (300, 8208, 4), (150, 4112, 5)])
def test_no_sum_is_a_chain_of_more_than_512_products(M, N, tiling):
    """Tiles of 128 columns over 17 k tiles: the running sums of eight tiles, of eight and of one are added, whatever the depth of the ring.  The
    first product of the first eight is -2^24 and of the second 2^24, beside which the others, 2^-7 each and less than half a unit of that together
    in any instruction, are lost; the last tile's 64 stand alone and come to 1/2."""
    from yalm_amd.ops import library
    k, Kd = K(), 17 * 64
    assert library.lib().yalm_gemm_bf16_dma_choice(M, N, Kd, 0, 0) == 10 + tiling
    a, w = torch.full((M, Kd), 2.0 ** -3), torch.full((N, Kd), 2.0 ** -4)
    a[:, 0], a[:, 512], w[:, 0], w[:, 512] = -2.0 ** 12, 2.0 ** 12, 2.0 ** 12, 2.0 ** 12
    out = torch.full((M, N), float("nan"), device=DEV)
    k.gemm(a.bfloat16().to(DEV), w.bfloat16().to(DEV), out, k.EPI_STORE_F32)
    assert bool((out == 0.5).all()), out.unique()[:4]


def test_gemm_of_a_prompt_step_is_the_same_with_and_without_k_slices():
    """A product in K slices agrees with the whole one within float32 rounding, and a launch repeats itself bit
    for bit."""
    k = K()
    M, N, Kd = 512, 4096, 4096
    a = rnd((M, Kd), 95, torch.bfloat16).to(DEV)
    w = rnd((N, Kd), 96, torch.bfloat16, scale=1 / 64).to(DEV)
    floats = k.gemm_workspace_floats(M, N, Kd)
    assert floats >= 2 * M * N                                   # few tiles: the launcher would split K
    outs = []
    for ws in (torch.empty((floats,), device=DEV), None):
        out = torch.empty((M, N), device=DEV)
        k.gemm(a, w, out, k.EPI_STORE_F32, workspace=ws)
        outs.append(out)
    # slices are added in order, but ((a + b) + (c + d)) is another rounding than (((a + b) + c) + d)
    close(outs[0], outs[1].double().cpu(), torch.float32, "sliced against whole")
    out = torch.empty((M, N), device=DEV)
    k.gemm(a, w, out, k.EPI_STORE_F32, workspace=None)
    assert torch.equal(out, outs[1])                             # and a launch repeats itself bit for bit


def _random_gemm_shapes(n, seed):
    """Row counts on both sides of every kernel's limits (16, 64, 128, 256), widths from tiny to several
    workgroups' worth, K with and without the factors (8, 64) that choose the path."""
    rng = np.random.default_rng(seed)
    rows = [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 100, 127, 128, 129, 200, 255, 256, 257, 300]
    shapes = []
    for _ in range(n):
        M = int(rng.choice(rows))
        N = int(rng.choice([1, 15, 16, 17, 100, 255, 256, 300, 1000, 2050, 4096, 6200]))
        K = int(rng.choice([8, 24, 64, 72, 128, 192, 200, 320, 1024, 1032]))
        shapes.append((M, N, K))
    return shapes


@pytest.mark.parametrize("with_workspace", [False, True])
def test_gemm_random_shapes(with_workspace):
    """Every dispatch branch of the bfloat16 GEMM at shapes nobody tuned for, all epilogues."""
    from yalm_amd.parts.swiglu import interleave_gate_up
    k = K()
    for idx, (M, N, Kd) in enumerate(_random_gemm_shapes(40, 7 if with_workspace else 8)):
        a = rnd((M, Kd), 1000 + idx, torch.bfloat16)
        w = rnd((N, Kd), 2000 + idx, torch.bfloat16, scale=1 / math.sqrt(Kd))
        want = a.double() @ w.double().T
        ad, wd = a.to(DEV), w.to(DEV)
        ws = None
        if with_workspace:
            n = k.gemm_workspace_floats(M, max(N, 32 * ((N + 15) // 16)), Kd)
            ws = torch.full((n,), float("nan"), device=DEV) if n else None
        tag = "M %d N %d K %d" % (M, N, Kd)
        out = torch.empty((M, N), device=DEV)
        k.gemm(ad, wd, out, k.EPI_STORE_F32, workspace=ws)
        close(out, want, torch.float32, tag + " f32")
        out2 = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
        k.gemm(ad, wd, out2, k.EPI_STORE, workspace=ws)
        close(out2, want, torch.bfloat16, tag + " bf16")
        res = rnd((M, N), 3000 + idx)
        acc = res.to(DEV).clone()
        k.gemm(ad, wd, acc, k.EPI_ADD_F32, workspace=ws)
        close(acc, want + res.double(), torch.float32, tag + " add")
        wu = rnd((N, Kd), 4000 + idx, torch.bfloat16, scale=1 / math.sqrt(Kd))
        gated = R.silu(want) * (a.double() @ wu.double().T)
        outg = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
        k.gemm(ad, interleave_gate_up(w, wu).to(DEV), outg, k.EPI_GATED, hidden=N, workspace=ws)
        close(outg, gated, torch.bfloat16, tag + " gated", factor=2.0)


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,H,D", [(1, 16, 64), (5, 176, 64), (70, 100, 96), (64, 1000, 264), (3, 14336, 128),
                                   (70, 100, 128), (300, 10300, 64), (260, 1000, 256), (7, 100, 192), (13, 7000, 128),
                                   (16, 13000, 64), (9, 3300, 320), (24, 100, 192), (61, 1000, 128),
                                   (513, 12820, 64), (2048, 14336, 64)])   # 192 x 128 and 256 x 256 tiles
@pytest.mark.parametrize("act", ACTS)
def test_gemm_gated(M, H, D, dtype, simple, act):
    from yalm_amd.parts.swiglu import interleave_gate_up
    k = K()
    x = rnd((M, D), 7, dtype)
    wg = rnd((H, D), 8, dtype, scale=1 / math.sqrt(D))
    wu = rnd((H, D), 9, dtype, scale=1 / math.sqrt(D))
    g = x.double() @ wg.double().T
    u = x.double() @ wu.double().T
    act_fn, epi_code = gate(act)
    want = act_fn(g) * u
    k.FORCE_SIMPLE = simple
    try:
        out = torch.empty((M, H), dtype=dtype, device=DEV)
        k.gemm(x.to(DEV), interleave_gate_up(wg, wu).to(DEV), out, epi_code, hidden=H)
        close(out, want, dtype, "gated gemm")
    finally:
        k.FORCE_SIMPLE = False


# float32: a row's results have the same bits whatever the rows beside it, up to 64 of them (narrow and wide products, short and
# long sums, sums of no whole k tiles)
@pytest.mark.parametrize("epi", ["store", "add", "gated"])
@pytest.mark.parametrize("N,Kd", [(64, 32), (96, 36), (96, 544), (4096, 288), (4128, 96), (8192, 2048), (8192, 2080), (16416, 4128)])
def test_gemm_float32_rows_do_not_depend_on_their_number(N, Kd, epi):
    k = K()
    a, w, x = rnd((64, Kd), 95).to(DEV), rnd((N, Kd), 96).to(DEV), rnd((64, N), 97).to(DEV)
    H = N // 2 - 3 if N > 64 else N // 2

    def product(lo, hi):
        if epi == "gated":
            return k.gemm(a[lo:hi], w, torch.empty((hi - lo, H), device=DEV), k.EPI_GATED, hidden=H)
        return k.gemm(a[lo:hi], w, x[lo:hi].clone(), k.EPI_ADD_F32 if epi == "add" else k.EPI_STORE_F32)

    whole = product(0, 64)
    for lo, hi in [(0, n) for n in (1, 2, 4, 5, 7, 8, 15, 16, 17, 31, 32, 33, 48, 63)] + [(20, 21), (50, 64)]:
        assert torch.equal(product(lo, hi), whole[lo:hi]), (lo, hi)


# Every kernel and tile of the float32 products on the matrix cores (yalm_gemm_f32_choice), with edges of 1 to 31 rows and columns
# and K of 37 or 69 k tiles: each ring of two to four stages turns many times, and sums are folded in whole and broken runs.  More than 64
# rows of 512 k and more go by bfloat16 terms but for few tiles' worth, so most tiles there have K of 15 k tiles
@pytest.mark.parametrize("M,N,Kd,choice", [
    (1, 40, 1184, 11), (9, 4100, 1184, 12), (17, 3000, 1184, 21), (33, 4100, 1184, 22), (47, 2001, 1184, 41),
    (3, 8200, 2208, 111), (1, 20001, 2208, 112), (33, 11999, 2208, 121), (47, 40001, 2208, 122),
    (70, 41, 1184, 211), (129, 6144, 1184, 212), (129, 4001, 480, 212), (97, 5130, 480, 221), (161, 8201, 480, 222), (161, 16401, 480, 224),
    (161, 12001, 480, 233), (513, 5131, 480, 234), (321, 20001, 480, 244)])
def test_gemm_float32_every_tile(M, N, Kd, choice):
    from yalm_amd.ops import library
    k = K()
    assert library.lib().yalm_gemm_f32_choice(M, N, Kd, 0) == choice and library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 0) == -1
    a, w, x = rnd((M, Kd), 101).to(DEV), rnd((N, Kd), 102).to(DEV), rnd((M, N), 103).to(DEV)
    want = a.double() @ w.double().t()
    # K products and K additions in any order, the residual's addition once more (as below)
    bound = (2.0 * Kd + 2.0) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t() + x.double().abs())
    out = k.gemm(a, w, torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32)
    assert bool(((out.double() - want).abs() <= bound).all())
    # those bounds are of the worst case: the sums' own errors are chance's, some of a rounding's size, and a k tile left out or
    # taken twice (a thirty-seventh of the products) is a thousand times that
    assert float((out.double() - want).norm() / want.norm()) <= 1e-6
    got = k.gemm(a, w, x.clone(), k.EPI_ADD_F32).double() - x.double()
    assert bool(((got - want).abs() <= bound).all()) and float((got - want).norm() / want.norm()) <= 1e-6


@pytest.mark.parametrize("M,N,Kd,choice", [
    (1, 64, 1184, 12), (33, 3008, 1184, 22), (3, 8224, 2208, 112), (47, 40000, 2208, 122), (65, 64, 1184, 212), (161, 8224, 480, 222),
    (161, 16416, 480, 224), (513, 5152, 480, 234), (321, 20000, 480, 244)])
def test_gemm_float32_every_gated_tile(M, N, Kd, choice):
    from yalm_amd.ops import library
    k = K()
    assert library.lib().yalm_gemm_f32_choice(M, N, Kd, 1) == choice and library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 1) == -1
    H = N // 2 - 3
    a, w = rnd((M, Kd), 104).to(DEV), rnd((N, Kd), 105, scale=Kd ** -0.5).to(DEV)
    p = (a.double() @ w.double().t()).view(M, -1, 2, 16)
    gate, up = p[:, :, 0].reshape(M, -1)[:, :H], p[:, :, 1].reshape(M, -1)[:, :H]
    want = gate / (1.0 + torch.exp(-gate)) * up
    got = k.gemm(a, w, torch.full((M, H), 7.0, device=DEV), k.EPI_GATED, hidden=H).double()
    # gate and up are sums about 1e-6 off at sizes of 1 that the unit multiplies (its slope is at most 1.1), and its own roundings
    assert float((got - want).norm() / want.norm()) <= 4e-6
    assert float((got - want).abs().max()) <= 1e-4


# The larger tiles of float32 products, which only sums of less than 512 still take: 15 k tiles, so that each ring turns and sums
# are folded in a whole and a broken run
@pytest.mark.parametrize("M,N,choice", [(161, 16401, 224), (161, 12001, 233), (513, 5130, 234), (321, 20001, 244)])
def test_gemm_float32_short_sums_on_the_larger_tiles(M, N, choice):
    from yalm_amd.ops import library
    k, Kd = K(), 480
    assert library.lib().yalm_gemm_f32_choice(M, N, Kd, 0) == choice and library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 0) == -1
    a, w = rnd((M, Kd), 111).to(DEV), rnd((N, Kd), 112).to(DEV)
    want = a.double() @ w.double().t()
    out = k.gemm(a, w, torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32).double()
    assert bool(((out - want).abs() <= (2.0 * Kd + 2.0) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t())).all())
    assert float((out - want).norm() / want.norm()) <= 1e-6


# Every tile of the products by bfloat16 terms, with edges of 1 to 200 rows and columns, an even number of k tiles (16), odd ones (17
# and 37: the two groups of a workgroup have unlike numbers, folds are broken)
@pytest.mark.parametrize("Kd", [512, 544, 1184])
@pytest.mark.parametrize("M,N,tile", [(97, 5130, 0), (161, 8201, 1), (161, 12001, 2), (513, 5131, 3), (513, 8201, 4), (321, 20001, 5)])
def test_gemm_float32_by_terms(M, N, tile, Kd):
    from yalm_amd.ops import library
    k = K()
    assert library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 0) == tile
    a, w, x = rnd((M, Kd), 113).to(DEV), rnd((N, Kd), 114).to(DEV), rnd((M, N), 115).to(DEV)
    want = a.double() @ w.double().t()
    # as for the float32 products: six products of terms an element, the three left out together below 2^-25 of the product
    bound = (2.0 * Kd + 2.0) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t() + x.double().abs())
    out = k.gemm(a, w, torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32).double()
    assert bool(((out - want).abs() <= bound).all()) and float((out - want).norm() / want.norm()) <= 1e-6
    got = k.gemm(a, w, x.clone(), k.EPI_ADD_F32).double() - x.double()
    assert bool(((got - want).abs() <= bound).all()) and float((got - want).norm() / want.norm()) <= 1e-6


@pytest.mark.parametrize("M,N,tile", [(97, 5152, 0), (161, 8224, 1), (513, 5152, 3), (513, 8224, 4), (321, 20000, 5)])
@pytest.mark.parametrize("act", ACTS)
def test_gemm_float32_by_terms_gated(M, N, tile, act):
    from yalm_amd.ops import library
    k, Kd = K(), 544
    assert library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 1) == tile
    act_fn, epi = gate(act)
    H = N // 2 - 3
    a, w = rnd((M, Kd), 116).to(DEV), rnd((N, Kd), 117, scale=Kd ** -0.5).to(DEV)
    p = (a.double() @ w.double().t()).view(M, -1, 2, 16)
    gate_, up = p[:, :, 0].reshape(M, -1)[:, :H], p[:, :, 1].reshape(M, -1)[:, :H]
    want = act_fn(gate_.cpu()).to(DEV) * up
    got = k.gemm(a, w, torch.full((M, H), 7.0, device=DEV), epi, hidden=H).double()
    assert float((got - want).norm() / want.norm()) <= 4e-6            # as for the gated float32 products above
    assert float((got - want).abs().max()) <= 1e-4


# Products by terms of what no bfloat16 holds: infinities, NaN, numbers that round to infinity, numbers whose last terms
# vanish.  The sums are those of float32 products: not finite where a factor is not, the others untouched
@pytest.mark.parametrize("M,N,Kd", [(161, 8201, 544), (321, 20001, 512)])
def test_gemm_float32_by_terms_of_extreme_numbers(M, N, Kd):
    from yalm_amd.ops import library
    k = K()
    assert library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 0) >= 0
    a, w = rnd((M, Kd), 118), rnd((N, Kd), 119, scale=0.01)
    a[3, 17], a[40, 500], a[41, 5], a[M - 1, 0] = math.inf, -math.inf, math.nan, 3.4028234e38
    a[70] *= 1e-30
    a[71] *= 2.0 ** -100
    w[N - 2, 9] = math.inf
    w[5] *= 1e-6
    want = a.double() @ w.double().t()
    got = k.gemm(a.to(DEV), w.to(DEV), torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32).double().cpu()
    size = a.double().abs() @ w.double().abs().t()
    over = size.isfinite() & (size >= 3.4e38)                           # whose sums may pass float32's largest on the way
    inf = want.isinf()
    assert int(inf.sum()) > M + 2 * N - 6 and int((inf & over).sum()) == 0
    assert torch.equal(got.isnan() & ~over, want.isnan() & ~over)
    assert torch.equal(got.isinf() & ~over, inf & ~over)
    assert torch.equal(got[inf], want[inf])                             # of the same sign
    ok = size < 3.4e38
    assert int(ok.sum()) > (M - 4) * (N - 1) - 1
    assert bool(((got - want).abs()[ok] <= ((2.0 * Kd + 2.0) * 2.0 ** -24 * size + Kd * 2.0 ** -126)[ok]).all())
    assert float((got[71] - want[71])[:N - 2].norm() / want[71][:N - 2].norm()) <= 1e-6


# Sums that are not finite are made again; the sums beside them, of the same wave too, keep the bits that they have without such a
# neighbour: one row and one weight row of infinities and NaN, the last ones (which the rows behind the edge repeat) among them
@pytest.mark.parametrize("M,N,tile", [(97, 5130, 0), (161, 8201, 1), (513, 5131, 3), (321, 20001, 5)])
def test_gemm_float32_by_terms_beside_numbers_that_are_not_finite(M, N, tile):
    from yalm_amd.ops import library
    k, Kd = K(), 512
    assert library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 0) == tile
    a, w = rnd((M, Kd), 143).to(DEV), rnd((N, Kd), 144).to(DEV)
    plain = k.gemm(a, w, torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32)
    rows, cols = [5, 40, M - 1], [3, 77, N - 1]
    for r, c, v in zip(rows, cols, (math.inf, math.nan, -math.inf)):
        a[r, 9], w[c, 100] = v, v
    got = k.gemm(a, w, torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32)
    assert not bool(got[rows].isfinite().any()) and not bool(got[:, cols].isfinite().any())
    keep_m, keep_n = [m for m in range(M) if m not in rows], [n for n in range(N) if n not in cols]
    assert torch.equal(got[keep_m][:, keep_n], plain[keep_m][:, keep_n])


# Operands at the lower end of float32, whose last terms would fall off bfloat16's: every row (or weight row) at another power of
# two from 2^-100 into the subnormal numbers, the other operand large, so that the sums are ordinary numbers; a workgroup of one group
# and of two
@pytest.mark.parametrize("small", ["a", "w"])
@pytest.mark.parametrize("M,N,tile", [(97, 5130, 0), (513, 5131, 3)])
def test_gemm_float32_by_terms_of_small_numbers(M, N, tile, small):
    from yalm_amd.ops import library
    k, Kd = K(), 512
    assert library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 0) == tile
    scale = lambda n: torch.tensor([2.0 ** -(100 + i % 46) for i in range(n)], dtype=torch.float64)[:, None]
    a, w = (rnd((n, Kd), s, torch.float64) * (scale(n) if name == small else 2.0 ** 80) for n, s, name in ((M, 141, "a"), (N, 142, "w")))
    a, w = a.float(), w.float()
    want = a.double().to(DEV) @ w.double().to(DEV).t()
    got = k.gemm(a.to(DEV), w.to(DEV), torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32).double()
    axis = 1 if small == "a" else 0
    # as for ordinary numbers, row by row (column by column)
    assert float(((got - want).norm(dim=axis) / want.norm(dim=axis)).max()) <= 1e-6


# And at the upper end: sums beyond 2^80, operands beyond 2^104, and rows of both kinds beside ordinary ones
@pytest.mark.parametrize("up_a,up_w", [(70, 30), (110, -60), (-60, 115), (79, 0)])
@pytest.mark.parametrize("M,N,tile", [(97, 5130, 0), (513, 5131, 3)])
def test_gemm_float32_by_terms_of_large_numbers(M, N, tile, up_a, up_w):
    from yalm_amd.ops import library
    k, Kd = K(), 512
    assert library.lib().yalm_gemm_f32_split_choice(M, N, Kd, 0) == tile
    a, w = (rnd((n, Kd), s, torch.float64) * 2.0 ** up for n, s, up in ((M, 145, up_a), (N, 146, up_w)))
    a[::3] *= 2.0 ** -up_a
    a, w = a.float(), w.float()
    want = a.double().to(DEV) @ w.double().to(DEV).t()
    got = k.gemm(a.to(DEV), w.to(DEV), torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32).double()
    assert float(((got - want).norm(dim=1) / want.norm(dim=1)).max()) <= 1e-6


# float32 on the matrix cores: the edges of the smallest tiles and of the rules (16 | 17 and 32 | 33 rows, 4,096 and 8,192
# columns), of one k tile and a few, K short of one round of the waves, operands 4 bytes off
@pytest.mark.parametrize("M,N,Kd,off", [
    (1, 48, 32, 0), (15, 33, 64, 0), (16, 4096, 96, 0), (16, 8192, 64, 0), (17, 4097, 288, 0), (17, 4096, 288, 0), (32, 80, 544, 0),
    (33, 200, 128, 0), (64, 96, 1056, 0), (65, 129, 32, 0), (129, 160, 64, 0), (161, 3000, 160, 0), (700, 3072, 128, 0),
    (300, 7000, 96, 0), (7, 40, 64, 1), (70, 96, 64, 1)])
def test_gemm_float32_on_the_matrix_cores(M, N, Kd, off):
    k = K()
    a = rnd((M * Kd + off,), 91).to(DEV)[off:].view(M, Kd)
    w = rnd((N, Kd), 92).to(DEV)
    x = rnd((M, N), 93).to(DEV)
    want = a.double() @ w.double().t()
    # K products and K additions in any order: each is off by at most 2^-24 of what it holds, which the sum of the
    # products' sizes bounds; the residual's addition once more
    bound = (2.0 * Kd + 2.0) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t() + x.double().abs())
    out = torch.empty((M, N), dtype=torch.float32, device=DEV)
    assert bool(((k.gemm(a, w, out, k.EPI_STORE_F32).double() - want).abs() <= bound).all())
    got = k.gemm(a, w, x.clone(), k.EPI_ADD_F32).double()
    assert bool(((got - want - x.double()).abs() <= bound).all())
    if N >= 32:                                      # gate and up rows in blocks of 16
        H = N // 32 * 16 - 3 if N > 64 else N // 32 * 16
        rows = w[:32 * ((H + 15) // 16)].contiguous()
        p = (a.double() @ rows.double().t()).view(M, -1, 2, 16)
        gt, up = (p[:, :, i].reshape(M, -1)[:, :H] for i in (0, 1))
        got = k.gemm(a, rows, torch.empty((M, H), dtype=torch.float32, device=DEV), k.EPI_GATED, hidden=H).double()
        b = bound[:, :rows.shape[0]].reshape(M, -1, 2, 16)
        bg, bu = (b[:, :, i].reshape(M, -1)[:, :H] for i in (0, 1))
        # silu's slope is at most 1.1; its own and the product's rounding: a few units of the last place
        assert bool(((got - R.silu(gt) * up).abs() <= 1.1 * bg * (up.abs() + bu) + gt.abs() * bu + 16 * 2.0 ** -24 * (gt * up).abs()).all())


def test_gemm_vector_of_the_reference():
    """src/test.cpp:157-168: n = 256 inputs, d = 16 outputs, N(0,1), absolute 1e-4."""
    k = K()
    for seed in (0, 1):
        w = rnd((16, 256), seed)
        x = rnd((1, 256), seed + 10)
        out = torch.empty((1, 16), device=DEV)
        k.gemm(x.to(DEV), w.to(DEV), out, k.EPI_STORE_F32)
        assert (out.cpu().double() - x.double() @ w.double().T).abs().max() < 1e-4


# ------------------------------------------------------------------ rotation + cache write

def make_table(n_pos, hd, rd, theta):
    f = R.rope_inv_freq(hd, rd, theta)[: rd // 2]
    ang = torch.arange(n_pos, dtype=torch.float64)[:, None] * f[None, :]
    return torch.stack([torch.cos(ang), torch.sin(ang)], -1).float().contiguous()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd,rd", [(4, 2, 16, 16), (3, 1, 48, 48), (6, 3, 32, 16), (2, 2, 128, 128)])
def test_rope_kv_write(n_heads, n_kv, hd, rd, dtype):
    k = K()
    PAGE = k.PAGE
    n_pages, n_slots, ring = 9, 4, 3
    # two sequences: slot 2 with positions 60..69 (crosses a page), slot 0 with positions 0..4
    pos = list(range(60, 70)) + list(range(5))
    seq = [0] * 10 + [1] * 5
    T = len(pos)
    Q, KV = n_heads * hd, n_kv * hd
    qkv = rnd((T, Q + 2 * KV), 11)
    table = make_table(80, hd, rd, 10000.0)
    bt = torch.full((n_slots, ring), -1, dtype=torch.int32)
    bt[2, 0], bt[2, 1], bt[0, 0] = 5, 7, 1
    page_of = {0: {0: 5, 1: 7}, 1: {0: 1}}
    tile_of = {0: {0: 0, 1: 1}, 1: {0: 2}}            # staging: sequence 0 has tiles 0, 1; sequence 1 tile 2
    kp = torch.zeros((n_pages, n_kv, PAGE, hd), dtype=dtype, device=DEV)
    vp = torch.zeros((n_pages, n_kv, hd, PAGE), dtype=dtype, device=DEV)
    ks = torch.zeros((3, n_kv, PAGE, hd), dtype=dtype, device=DEV)
    vs = torch.zeros((3, n_kv, hd, PAGE), dtype=dtype, device=DEV)
    q_out = torch.empty((T, Q), dtype=dtype, device=DEV)
    k.rope_kv_write(qkv.to(DEV), q_out, ks, vs, i32([0, 2, 3]), kp, vp, bt.to(DEV), ring, i32(seq), i32(pos),
                    i32([2, 0]), i32([70, 5]), table.to(DEV), n_heads, n_kv, hd, rd)
    f = R.rope_inv_freq(hd, rd, 10000.0)
    p = torch.tensor(pos)
    q_want = R.rope_interleaved(qkv[:, :Q].reshape(T, n_heads, hd), p, f).reshape(T, Q)
    k_want = R.rope_interleaved(qkv[:, Q:Q + KV].reshape(T, n_kv, hd), p, f)
    v_want = qkv[:, Q + KV:].double().reshape(T, n_kv, hd)
    close(q_out, q_want, dtype, "q")
    kp, vp, ks, vs = kp.cpu(), vp.cpu(), ks.cpu(), vs.cpu()
    kp, vp = pages_as_rows(kp, vp)
    for t in range(T):
        page, tile, r = page_of[seq[t]][pos[t] // PAGE], tile_of[seq[t]][pos[t] // PAGE], pos[t] % PAGE
        close(ks[tile, :, r, :], k_want[t], dtype, "staged k")
        close(vs[tile, :, :, r], v_want[t], dtype, "staged v")
        assert torch.equal(kp[page, :, r, :], ks[tile, :, r, :])
        assert torch.equal(vp[page, :, :, r], vs[tile, :, :, r])
    # nothing else was touched
    touched = torch.zeros((n_pages, PAGE), dtype=torch.bool)
    for t in range(T):
        touched[page_of[seq[t]][pos[t] // PAGE], pos[t] % PAGE] = True
    assert (kp.float().abs().sum(dim=(1, 3)) > 0).equal(touched)


@pytest.mark.parametrize("M,n_heads,n_kv,hd,D", [(17, 4, 2, 16, 4096), (40, 3, 1, 48, 1024), (64, 8, 2, 128, 264),
                                                 (33, 2, 2, 64, 64), (65, 8, 2, 128, 4096), (200, 3, 1, 48, 1024),
                                                 (130, 2, 2, 64, 64)])
def test_gemm_partial_and_rotation_that_adds_the_slices(M, n_heads, n_kv, hd, D):
    """q/k/v projection of 17..64 rows whose K slices stay unadded, and the rotation kernel that adds them
    while it reads: the same q and cache pages as the product, added first, gives."""
    k = K()
    PAGE = k.PAGE
    Q, KV = n_heads * hd, n_kv * hd
    N = Q + 2 * KV
    h = rnd((M, D), 90, torch.bfloat16)
    w = rnd((N, D), 91, torch.bfloat16, scale=1 / math.sqrt(D))
    ws = torch.full((k.fused_workspace_floats(M, N, D),), float("nan"), device=DEV)
    slices = k.gemm_partial(h.to(DEV), w.to(DEV), ws)
    assert 1 <= slices and slices * M * N <= ws.numel()
    if D >= 1024 and N < 4096:
        assert slices > 1                                      # the case this test is for
    qkv = ws[:slices * M * N].reshape(slices, M, N).sum(dim=0)
    close(qkv, h.double() @ w.double().T, torch.float32, "sum of the slices")
    # one sequence per row, at positions 61 + row (so that some cross a page)
    table = make_table(200, hd, hd, 10000.0).to(DEV)
    pos = [61 + m for m in range(M)]
    bt = torch.arange(2 * M, dtype=torch.int32).reshape(M, 2).to(DEV)
    outs = []
    for source, n in ((qkv.contiguous(), 1), (ws, slices)):
        kp = torch.zeros((2 * M, n_kv, PAGE, hd), dtype=torch.bfloat16, device=DEV)
        vp = torch.zeros((2 * M, n_kv, hd, PAGE), dtype=torch.bfloat16, device=DEV)
        q = torch.zeros((M, Q), dtype=torch.bfloat16, device=DEV)
        k.rope_kv_write(source, q, None, None, None, kp, vp, bt, 2, i32(list(range(M))), i32(pos),
                        i32(list(range(M))), i32([p + 1 for p in pos]), table, n_heads, n_kv, hd, hd, slices=n)
        outs.append((q, kp, vp))
    for a, b, what in zip(outs[0], outs[1], ("q", "k pages", "v pages")):
        assert a.abs().sum() > 0
        close(b, a.double().cpu(), torch.bfloat16, what)       # the slices are added in another order than torch's sum
    with pytest.raises(ValueError):
        k.rope_kv_write(ws[:M * N], outs[0][0], None, None, None, None, None, None, 0, i32(list(range(M))), i32(pos),
                        i32(list(range(M))), i32([p + 1 for p in pos]), table, n_heads, n_kv, hd, hd, slices=2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd,rd,lens,ring", [(4, 2, 16, 16, [5, 130, 64], 3), (3, 1, 48, 24, [200, 1], 2),
                                                          (8, 2, 128, 128, [70, 257], 8), (2, 2, 64, 64, [300], 3),
                                                          (2, 1, 16, 6, [70, 5], 2), (3, 3, 18, 10, [130], 3)])
def test_rope_kv_write_tiles(n_heads, n_kv, hd, rd, lens, ring, dtype):
    """Whole prompts, a tile of 64 positions at a time: the same q, staging area and cache pages as the
    per-token kernel (which the tests above pin to the plain rotation), also where a prompt ends inside a
    tile and where a ring keeps the last pages only."""
    k = K()
    PAGE = k.PAGE
    B, T = len(lens), sum(lens)
    Q, KV = n_heads * hd, n_kv * hd
    qkv = rnd((T, Q + 2 * KV), 21).to(DEV)
    table = make_table(max(lens) + 3, hd, rd, 10000.0).to(DEV)
    tiles = [(n + PAGE - 1) // PAGE for n in lens]
    tile0 = np.concatenate([[0], np.cumsum(tiles)])
    cu = np.concatenate([[0], np.cumsum(lens)])
    n_tiles, n_pages = int(tile0[-1]), B * ring + 2
    order = np.random.default_rng(5).permutation(n_pages)
    bt = torch.full((B + 1, ring), -1, dtype=torch.int32)
    slots = [B - b for b in range(B)]                         # slots B, B-1, ..., 1
    nxt = 0
    for b in range(B):
        for c in range(min(ring, tiles[b])):
            bt[slots[b], c] = int(order[nxt])
            nxt += 1
    seq = np.repeat(np.arange(B), lens)
    pos = np.concatenate([np.arange(n) for n in lens])

    def buffers():
        return (torch.zeros((n_pages, n_kv, PAGE, hd), dtype=dtype, device=DEV),
                torch.zeros((n_pages, n_kv, hd, PAGE), dtype=dtype, device=DEV),
                torch.zeros((n_tiles, n_kv, PAGE, hd), dtype=dtype, device=DEV),
                torch.zeros((n_tiles, n_kv, hd, PAGE), dtype=dtype, device=DEV),
                torch.zeros((T, Q), dtype=dtype, device=DEV))
    kp0, vp0, ks0, vs0, q0 = buffers()
    k.rope_kv_write(qkv, q0, ks0, vs0, i32(tile0), kp0, vp0, bt.to(DEV), ring, i32(seq), i32(pos), i32(slots),
                    i32(lens), table, n_heads, n_kv, hd, rd)
    kp1, vp1, ks1, vs1, q1 = buffers()
    assert k.rope_kv_write_tiles(qkv, q1, ks1, vs1, i32(cu), i32(tile0), kp1, vp1, bt.to(DEV), ring, i32(slots),
                                 i32(lens), table, n_heads, n_kv, hd, rd)
    for a, b, what in ((q0, q1, "q"), (ks0, ks1, "staged k"), (vs0, vs1, "staged v"), (kp0, kp1, "k pages"),
                       (vp0, vp1, "v pages")):
        assert torch.equal(a, b), what
    assert q0.abs().sum() > 0 and kp0.abs().sum() > 0
    # the K slices of a product instead of the product: added in order, as the per-token kernel adds them
    parts = torch.stack([rnd((T, Q + 2 * KV), 30 + s).to(DEV) for s in range(3)]).reshape(-1)
    kp2, vp2, ks2, vs2, q2 = buffers()
    k.rope_kv_write(parts, q2, ks2, vs2, i32(tile0), kp2, vp2, bt.to(DEV), ring, i32(seq), i32(pos), i32(slots),
                    i32(lens), table, n_heads, n_kv, hd, rd, slices=3)
    kp3, vp3, ks3, vs3, q3 = buffers()
    assert k.rope_kv_write_tiles(parts, q3, ks3, vs3, i32(cu), i32(tile0), kp3, vp3, bt.to(DEV), ring, i32(slots),
                                 i32(lens), table, n_heads, n_kv, hd, rd, slices=3)
    for a, b, what in ((q2, q3, "q"), (ks2, ks3, "staged k"), (vs2, vs3, "staged v"), (kp2, kp3, "k pages"),
                       (vp2, vp3, "v pages")):
        assert torch.equal(a, b), what + " from slices"
    assert not torch.equal(q2, q0)
    with pytest.raises(ValueError):
        k.rope_kv_write_tiles(parts[:2 * T * (Q + 2 * KV)], q3, ks3, vs3, i32(cu), i32(tile0), kp3, vp3, bt.to(DEV),
                              ring, i32(slots), i32(lens), table, n_heads, n_kv, hd, rd, slices=3)


def test_rope_kv_write_ring_keeps_the_last_pages_only():
    k = K()
    PAGE = k.PAGE
    n_kv, hd, ring = 1, 16, 2
    L = 3 * PAGE + 5                         # pages 0..3 exist, the ring keeps pages 2 and 3
    qkv = rnd((L, 2 * hd + hd), 12)          # one query head
    bt = torch.tensor([[4, 6]], dtype=torch.int32)
    kp = torch.zeros((8, n_kv, PAGE, hd), device=DEV)
    vp = torch.zeros((8, n_kv, hd, PAGE), device=DEV)
    q_out = torch.empty((L, hd), device=DEV)
    k.rope_kv_write(qkv.to(DEV), q_out, None, None, None, kp, vp, bt.to(DEV), ring, i32([0] * L),
                    i32(list(range(L))), i32([0]), i32([L]), None, 1, n_kv, hd, 0)
    kp = pages_as_rows(kp.cpu(), vp.cpu())[0]
    # absolute page 2 -> column 0 (page 4), page 3 -> column 1 (page 6)
    assert torch.equal(kp[4, 0], qkv[2 * PAGE:3 * PAGE, hd:2 * hd])
    assert torch.equal(kp[6, 0, :5], qkv[3 * PAGE:, hd:2 * hd])
    assert kp[6, 0, 5:].abs().sum() == 0
    assert torch.equal(q_out.cpu(), qkv[:, :hd])           # no table: no rotation


# ------------------------------------------------------------------ attention

def packed_attention_reference(q, k, v, lens, n_heads, n_kv, hd, window):
    outs, o = [], 0
    for n in lens:
        outs.append(R.attention(q[o:o + n].reshape(n, n_heads, hd), k[o:o + n].reshape(n, n_kv, hd),
                                v[o:o + n].reshape(n, n_kv, hd), window).reshape(n, n_heads * hd))
        o += n
    return torch.cat(outs)


def stage(kk, v, lens, n_kv, hd, dtype, poison=True):
    """Keys and values of packed sequences in the staging format of a prefill step."""
    PAGE = K().PAGE
    tile0 = np.concatenate([[0], np.cumsum([(n + PAGE - 1) // PAGE for n in lens])])
    fill = float("nan") if poison else 0.0
    ks = torch.full((int(tile0[-1]), n_kv, PAGE, hd), fill, dtype=dtype)
    vs = torch.full((int(tile0[-1]), n_kv, hd, PAGE), fill, dtype=dtype)
    o = 0
    for b, n in enumerate(lens):
        for p in range(n):
            ks[tile0[b] + p // PAGE, :, p % PAGE, :] = kk[o + p].reshape(n_kv, hd)
            vs[tile0[b] + p // PAGE, :, :, p % PAGE] = v[o + p].reshape(n_kv, hd)
        o += n
    return ks, vs, tile0


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd,window,lens", [
    (4, 2, 16, 0, [5, 17, 1]), (3, 1, 32, 16, [2, 30, 70]), (6, 3, 48, 100, [130, 64]), (8, 2, 128, 0, [200]),
    (2, 2, 80, 7, [65, 3]), (5, 5, 64, 0, [129]), (4, 1, 64, 70, [300, 64, 1]), (8, 2, 128, 100, [17, 257]),
    (6, 2, 96, 50, [150, 64, 333]), (9, 3, 32, 0, [257, 1]), (4, 2, 112, 30, [200, 64]), (5, 1, 16, 0, [131, 7])])
def test_attn_prefill(n_heads, n_kv, hd, window, lens, dtype, simple):
    k = K()
    T = sum(lens)
    q = rnd((T, n_heads * hd), 13, dtype)
    kk = rnd((T, n_kv * hd), 14, dtype)
    v = rnd((T, n_kv * hd), 15, dtype)
    cu = np.concatenate([[0], np.cumsum(lens)])
    seq = np.repeat(np.arange(len(lens)), lens)
    pos = np.concatenate([np.arange(n) for n in lens])
    ks, vs, tile0 = stage(kk, v, lens, n_kv, hd, dtype)
    out = torch.empty((T, n_heads * hd), dtype=dtype, device=DEV)
    k.FORCE_SIMPLE = simple
    try:
        k.attn_prefill(q.to(DEV), ks.to(DEV), vs.to(DEV), out, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv,
                       hd, window)
    finally:
        k.FORCE_SIMPLE = False
    close(out, packed_attention_reference(q, kk, v, lens, n_heads, n_kv, hd, window), dtype, "prefill attention")


@pytest.mark.parametrize("slices", [1, 3])
@pytest.mark.parametrize("n_heads,n_kv,hd,rd,lens", [
    (4, 2, 128, 128, [1]), (8, 2, 128, 128, [33]), (8, 2, 128, 64, [64, 1, 15]), (3, 1, 128, 0, [16, 17, 48, 49, 63]),
    (2, 2, 64, 64, [64]), (6, 3, 64, 6, [31, 32, 1, 64]), (4, 4, 64, 0, [2, 65 - 1])])
def test_attn_tile(n_heads, n_kv, hd, rd, lens, slices):
    """Prompts of one tile each in one launch: the bits of the rotation kernel with the attention kernel behind it, in the result
    and in the pages of the cache, at both ends of a tile and of a wave's 16 queries; a sequence without a slot writes no page."""
    k = K()
    PAGE = k.PAGE
    B, T = len(lens), sum(lens)
    Q, KV = n_heads * hd, n_kv * hd
    parts = torch.stack([rnd((T, Q + 2 * KV), 40 + s) for s in range(slices)]).to(DEV)
    qkv = parts[0] if slices == 1 else parts.reshape(-1)
    table = make_table(PAGE, hd, rd, 10000.0).to(DEV) if rd else None
    cu, tile0 = np.concatenate([[0], np.cumsum(lens)]), np.arange(B + 1)
    seq, pos = np.repeat(np.arange(B), lens), np.concatenate([np.arange(n) for n in lens])
    slots = [B - b for b in range(B)]
    if B > 2:
        slots[1] = -1
    bt = torch.full((B + 1, 2), -1, dtype=torch.int32)
    bt[1:, 0] = torch.from_numpy(np.random.default_rng(5).permutation(B + 3)[:B].astype(np.int32))
    bt = bt.to(DEV)

    def pages():
        return (torch.zeros((B + 3, n_kv, PAGE, hd), dtype=torch.bfloat16, device=DEV),
                torch.zeros((B + 3, n_kv, hd, PAGE), dtype=torch.bfloat16, device=DEV))
    (kp0, vp0), (kp1, vp1) = pages(), pages()
    q = torch.empty((T, Q), dtype=torch.bfloat16, device=DEV)
    ks = torch.full((B, n_kv, PAGE, hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    vs = torch.full((B, n_kv, hd, PAGE), float("nan"), dtype=torch.bfloat16, device=DEV)
    want, got = torch.empty_like(q), torch.full_like(q, float("nan"))
    k.rope_kv_write(qkv, q, ks, vs, i32(tile0), kp0, vp0, bt, 2, i32(seq), i32(pos), i32(slots), i32(lens), table, n_heads, n_kv,
                    hd, rd, slices=slices)
    k.attn_prefill(q, ks, vs, want, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv, hd, 0)
    assert k.attn_tile_fits(qkv, got, kp1, vp1, hd, 0) and not k.attn_tile_fits(qkv, got, kp1, vp1, hd, PAGE - 1)
    k.attn_tile(qkv, got, kp1, vp1, bt, 2, i32(cu), i32(slots), table, n_heads, n_kv, hd, rd, slices=slices)
    assert torch.equal(got, want)
    assert torch.equal(kp0, kp1) and torch.equal(vp0, vp1) and kp0.abs().sum() > 0


@pytest.mark.parametrize("n_heads,n_kv,hd,rd,lens,slices", [(16, 1, 128, 128, [33, 64], 2), (71, 1, 64, 64, [5, 64, 17], 1), (32, 2, 128, 64, [40], 8)])
def test_attn_tile_of_wide_groups_and_many_slices(n_heads, n_kv, hd, rd, lens, slices):
    test_attn_tile(n_heads, n_kv, hd, rd, lens, slices)


def test_attn_tile_says_which_steps_it_takes():
    """Operands off 16 bytes, more sequences than a launch has room for and more tiles than sequences are left to the kernels
    that it stands for."""
    k = K()
    hd, B = 64, 3
    qkv, kp = torch.zeros(1 + B * 3 * hd, device=DEV), torch.zeros(B, 1, k.PAGE, hd, dtype=torch.bfloat16, device=DEV)
    vp, out = torch.zeros(B, 1, hd, k.PAGE, dtype=torch.bfloat16, device=DEV), torch.zeros(1 + B * hd, dtype=torch.bfloat16, device=DEV)

    def fits(x=qkv[:-1], o=out[:-1], *rest):
        return k.attn_tile_fits(x, o, kp, vp, hd, 0, *rest)
    assert fits() and not fits(qkv[1:]) and not fits(o=out[1:])
    assert k.attn_tile_fits(qkv, out, kp, vp, hd, 0, 65535) and not k.attn_tile_fits(qkv, out, kp, vp, hd, 0, 65536)
    table, cu = torch.arange(B, dtype=torch.int32, device=DEV).reshape(B, 1), i32([0, 1, 2, 3])
    with pytest.raises(RuntimeError):
        k.attn_tile(qkv[:-1].view(B, 3 * hd), out[:-1].view(B, hd), kp, vp, table, 1, cu, i32([0, 1, 2]), None, 1, 1, hd, 0, n_tiles=B + 1)
    k.attn_tile(qkv[:-1].view(B, 3 * hd), out[:-1].view(B, hd), kp, vp, table, 1, cu, i32([0, 1, 2]), None, 1, 1, hd, 0, n_tiles=B)
    assert out.abs().sum() == 0


def masked_attention_float64(q, k, v, n_heads, n_kv, hd, window, bias=None):
    """softmax(q k^T / sqrt(hd) + mask) v for one sequence, all positions at once (float64).  bias ([n_heads,
    distances], optional): bias[h, min(i - j, distances - 1)] is added to the score of query i and key j."""
    n = q.shape[0]
    qh = q.double().reshape(n, n_heads, hd).transpose(0, 1)
    kh = k.double().reshape(n, n_kv, hd).transpose(0, 1).repeat_interleave(n_heads // n_kv, dim=0)
    vh = v.double().reshape(n, n_kv, hd).transpose(0, 1).repeat_interleave(n_heads // n_kv, dim=0)
    i = torch.arange(n)[:, None]
    j = torch.arange(n)[None, :]
    visible = (j <= i) & ((i - j < window) if window else torch.ones((n, n), dtype=torch.bool))
    out = torch.empty((n_heads, n, hd), dtype=torch.float64)
    for h in range(n_heads):                          # a head at a time: [n, n] scores
        s = (qh[h] @ kh[h].T) / math.sqrt(hd)
        if bias is not None:
            s = s + bias[h].double()[(i - j).clamp(0, bias.shape[1] - 1)]
        s = s.masked_fill(~visible, float("-inf"))
        out[h] = torch.softmax(s, dim=-1) @ vh[h]
    return out.transpose(0, 1).reshape(n, n_heads * hd)


@pytest.mark.parametrize("n_heads,n_kv,hd,window,lens", [(40, 8, 64, 0, [1700]), (40, 8, 128, 300, [1500, 260]),
                                                         (32, 8, 128, 0, [2048]), (40, 8, 96, 0, [1500]),
                                                         (40, 10, 32, 200, [2200, 70]), (12, 4, 96, 0, [1300]),
                                                         (40, 8, 80, 0, [1500]), (24, 8, 48, 100, [2300, 65]),
                                                         (12, 4, 16, 0, [1300]), (40, 8, 112, 0, [1700]),
                                                         (16, 1, 144, 0, [1500, 70]), (32, 1, 160, 0, [700]), (9, 1, 176, 100, [600, 129]),
                                                         (20, 4, 192, 0, [900, 1]), (16, 1, 208, 0, [300]), (8, 2, 224, 0, [640]),
                                                         (5, 1, 240, 70, [400, 65]), (16, 1, 256, 0, [700, 64])])
def test_attn_prefill_with_many_and_with_few_workgroups(n_heads, n_kv, hd, window, lens):
    """The matrix-core prefill kernel has two forms: workgroups of eight waves that take a tile's keys in two
    halves (launches of at most two workgroups a compute unit, the third case) and of four waves (more, the
    first two).  Both against a float64 masked softmax, itself checked against the plain implementation."""
    k = K()
    dtype = torch.bfloat16
    small = [rnd((70, 2 * 16), 31), rnd((70, 16), 32), rnd((70, 16), 33)]
    assert torch.allclose(masked_attention_float64(*small, 2, 1, 16, 9),
                          R.attention(small[0].reshape(70, 2, 16), small[1].reshape(70, 1, 16),
                                      small[2].reshape(70, 1, 16), 9).reshape(70, 32), atol=1e-12)
    T = sum(lens)
    q = rnd((T, n_heads * hd), 13, dtype)
    kk = rnd((T, n_kv * hd), 14, dtype)
    v = rnd((T, n_kv * hd), 15, dtype)
    cu = np.concatenate([[0], np.cumsum(lens)])
    seq = np.repeat(np.arange(len(lens)), lens)
    pos = np.concatenate([np.arange(n) for n in lens])
    ks, vs, tile0 = stage(kk, v, lens, n_kv, hd, dtype)
    out = torch.empty((T, n_heads * hd), dtype=dtype, device=DEV)
    order = i32(k.prefill_tile_order(lens))
    k.attn_prefill(q.to(DEV), ks.to(DEV), vs.to(DEV), out, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv, hd,
                   window, order)
    want, o = [], 0
    for n in lens:
        want.append(masked_attention_float64(q[o:o + n], kk[o:o + n], v[o:o + n], n_heads, n_kv, hd, window))
        o += n
    close(out, torch.cat(want), dtype, "prefill attention")


@pytest.mark.parametrize("n_heads,n_kv,hd,window,lens", [
    (8, 2, 128, 0, [200]), (5, 5, 64, 0, [129, 1, 640]), (4, 1, 64, 70, [300, 64, 1]), (40, 8, 128, 0, [700]),
    (24, 8, 64, 100, [1100, 90]), (8, 2, 128, 0, [2200, 90, 2100])])
def test_attn_prefill_in_a_given_tile_order(n_heads, n_kv, hd, window, lens):
    """The order of the tiles (with more workgroups than compute units it is folded) changes no
    bit of the result, and every position is still written."""
    k = K()
    dtype = torch.bfloat16
    T = sum(lens)
    q = rnd((T, n_heads * hd), 23, dtype).to(DEV)
    kk = rnd((T, n_kv * hd), 24, dtype)
    v = rnd((T, n_kv * hd), 25, dtype)
    cu = np.concatenate([[0], np.cumsum(lens)])
    seq = np.repeat(np.arange(len(lens)), lens)
    pos = np.concatenate([np.arange(n) for n in lens])
    ks, vs, tile0 = stage(kk, v, lens, n_kv, hd, dtype, poison=False)
    ks, vs = ks.to(DEV), vs.to(DEV)
    outs = []
    for order in (None, i32(k.prefill_tile_order(lens))):
        out = torch.full((T, n_heads * hd), float("nan"), dtype=dtype, device=DEV)
        k.attn_prefill(q, ks, vs, out, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv, hd, window, order)
        outs.append(out.cpu())
    assert not torch.isnan(outs[1].float()).any()
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("off", [(1, 0), (0, 2), (3, 5)])
def test_attn_prefill_with_stages_off_sixteen_bytes(off):
    """At head size 128 tiles that go straight into LDS have to lie on 16 bytes; others go through registers, with the same bits."""
    k = K()
    lens, n_heads, n_kv, hd, dtype = [200, 33], 4, 2, 128, torch.bfloat16
    T = sum(lens)
    q, kk, v = rnd((T, n_heads * hd), 43, dtype), rnd((T, n_kv * hd), 44, dtype), rnd((T, n_kv * hd), 45, dtype)
    cu = np.concatenate([[0], np.cumsum(lens)])
    seq = np.repeat(np.arange(len(lens)), lens)
    pos = np.concatenate([np.arange(n) for n in lens])
    ks, vs, tile0 = stage(kk, v, lens, n_kv, hd, dtype)

    def moved(t, by):
        flat = torch.empty(t.numel() + 8, dtype=dtype, device=DEV)
        view = flat[by:by + t.numel()].view(t.shape)
        view.copy_(t)
        return view

    out, on_sixteen = (torch.empty((T, n_heads * hd), dtype=dtype, device=DEV) for _ in range(2))
    k.attn_prefill(q.to(DEV), moved(ks, off[0]), moved(vs, off[1]), out, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv, hd, 0)
    k.attn_prefill(q.to(DEV), moved(ks, 0), moved(vs, 0), on_sixteen, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv, hd, 0)
    assert torch.equal(out, on_sixteen)
    want, o = [], 0
    for n in lens:
        want.append(masked_attention_float64(q[o:o + n], kk[o:o + n], v[o:o + n], n_heads, n_kv, hd, 0))
        o += n
    close(out, torch.cat(want), dtype, "prefill attention")


def paged_case(lens, n_kv, hd, window, dtype, seed, poison=True, stored=True):
    """Random keys/values of sequences of the given lengths laid out in pages the way
    the cache does (ring for a window), the rest of the pool poisoned with NaN.  stored=False: the pages in
    rows, for a caller that changes them before pages_as_stored."""
    k = K()
    PAGE = k.PAGE
    B = len(lens)
    full = max((n + PAGE - 1) // PAGE for n in lens)
    ring = min(full, (window + PAGE - 1) // PAGE + 1) if window else full
    n_pages = B * ring + 3
    kp = torch.full((n_pages, n_kv, PAGE, hd), float("nan") if poison else 0.0, dtype=dtype)
    vp = torch.full((n_pages, n_kv, hd, PAGE), float("nan") if poison else 0.0, dtype=dtype)
    order = np.random.default_rng(seed).permutation(n_pages)
    bt = torch.full((B + 2, ring), -1, dtype=torch.int32)
    slots = list(np.random.default_rng(seed + 1).permutation(B + 2)[:B])
    keys, vals = [], []
    nxt = 0
    for b, n in enumerate(lens):
        kb = rnd((n, n_kv, hd), seed + 10 * b, dtype)
        vb = rnd((n, n_kv, hd), seed + 10 * b + 1, dtype)
        keys.append(kb)
        vals.append(vb)
        last_ap = (n - 1) // PAGE
        for ap in range(max(0, last_ap - ring + 1), last_ap + 1):
            page = int(order[nxt])
            nxt += 1
            bt[slots[b], ap % ring] = page
            rows = range(ap * PAGE, min(n, (ap + 1) * PAGE))
            for p in rows:
                kp[page, :, p % PAGE, :] = kb[p]
                vp[page, :, :, p % PAGE] = vb[p]
    if stored:
        kp, vp = pages_as_stored(kp, vp)
    return kp, vp, bt, [int(s) for s in slots], ring, keys, vals


def one_query_reference(q, keys, vals, window):
    """The last position's attention (src/infer.cpp:218-250 per head over the visible rows)."""
    n_heads, hd = q.shape
    n, n_kv = keys.shape[0], keys.shape[1]
    lo = max(0, n - window) if window else 0
    out = torch.zeros((n_heads, hd), dtype=torch.float64)
    for h in range(n_heads):
        g = h // (n_heads // n_kv)
        p = R.attention_probs_one_query(q[h], keys[lo:n, g], hd)
        out[h] = p @ vals[lo:n, g].double()
    return out


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd,window,lens,splits", [
    (4, 2, 16, 0, [5, 64, 65, 1], 1), (3, 1, 32, 16, [2, 30, 200], 2), (6, 3, 48, 100, [130, 640, 99], 3),
    (8, 2, 128, 0, [1000, 3], 7), (2, 2, 80, 0, [129], 4), (32, 8, 128, 0, [300], 2), (5, 5, 64, 70, [700, 64], 16),
    (6, 2, 96, 0, [900, 65, 2], 5), (12, 3, 96, 130, [400, 129], 2), (16, 1, 32, 0, [2000, 7], 9),
    (10, 2, 112, 0, [777, 3], 4), (9, 3, 80, 64, [500, 64], 3), (4, 4, 16, 0, [129, 1000], 5),
    (34, 2, 64, 0, [300, 65], 3), (40, 1, 128, 100, [700], 4), (51, 3, 32, 0, [129, 2], 2),   # more than 16 heads a group
    (16, 1, 144, 0, [700, 3], 4), (32, 1, 160, 0, [300], 2), (20, 1, 176, 100, [400, 64], 3), (8, 2, 192, 0, [900, 65], 5),
    (16, 1, 208, 0, [129], 1), (5, 1, 224, 0, [500, 2], 4), (3, 3, 240, 70, [300], 2), (16, 1, 256, 0, [700, 64], 3),
    (40, 2, 256, 0, [333], 1)])   # one wide head
def test_attn_decode(n_heads, n_kv, hd, window, lens, splits, dtype, simple):
    _attn_decode_case(n_heads, n_kv, hd, window, lens, splits, dtype, simple, None)


@pytest.mark.parametrize("said", ["longest", 1, 100000])
@pytest.mark.parametrize("n_heads,n_kv,hd,window,lens,splits", [
    (8, 2, 128, 0, [1000, 3, 517, 64, 65], 4), (4, 1, 64, 0, [40, 900], 7), (5, 5, 64, 150, [700, 64, 164, 150, 128], 3),
    (8, 2, 128, 100, [164, 150, 128, 100, 99], 2)])
def test_attn_decode_with_the_length_of_the_longest_sequence(n_heads, n_kv, hd, window, lens, splits, said):
    """Splits of the longest sequence's split size: the same results, whatever length the step says its longest
    sequence has (the truth, too little, too much), also where a window makes a shorter sequence span more pages
    than the longest does; and the workgroups take the rows in another order than the rows'."""
    _attn_decode_case(n_heads, n_kv, hd, window, lens, splits, torch.bfloat16, False, max(lens) if said == "longest" else said)


@pytest.mark.parametrize("n_heads,n_kv,hd,window,lens,splits", [
    (8, 2, 128, 0, [1000, 3, 517, 64, 65], 4), (4, 1, 64, 0, [40, 900], 7), (5, 5, 80, 150, [700, 64, 164], 3), (2, 1, 32, 0, [400, 9], 2)])
def test_attn_decode_float32_of_a_row_does_not_depend_on_the_others(n_heads, n_kv, hd, window, lens, splits):
    k = K()
    B = len(lens)
    kp, vp, bt, slots, ring, _, _ = paged_case(lens, n_kv, hd, window, torch.float32, 24)
    kp, vp, bt, q = kp.to(DEV), vp.to(DEV), bt.to(DEV), rnd((B, n_heads * hd), 25).to(DEV)
    partial = torch.empty(k.attn_decode_workspace_floats(B, n_heads, hd, splits), device=DEV)

    def decode(rows, longest):
        out = torch.full((len(rows), n_heads * hd), 7.0, device=DEV)
        return k.attn_decode(q[rows], kp, vp, bt, ring, i32([slots[r] for r in rows]), i32([lens[r] for r in rows]), out, partial,
                             n_heads, n_kv, hd, window, splits, step_max_len=None if longest is None else i32([longest]))

    together = decode(list(range(B)), max(lens))
    assert torch.equal(decode(list(range(B)), None), together) and torch.equal(decode(list(range(B)), 100000), together)
    for r in range(B):
        assert torch.equal(decode([r], lens[r])[0], together[r])


@pytest.mark.parametrize("missing", [-1, -7, 1 << 20])
@pytest.mark.parametrize("hd", [32, 64, 112, 128])
def test_attn_decode_float32_passes_over_a_page_that_does_not_exist(hd, missing):
    """As the general kernel does: the page's keys are not among those that a query sees."""
    k = K()
    lens, n_heads, n_kv, splits = [300, 64, 130], 4, 2, 2
    kp, vp, bt, slots, ring, _, _ = paged_case(lens, n_kv, hd, 0, torch.float32, 26)
    bt[slots[0], 1] = missing
    bt[slots[2], 0] = missing
    q = rnd((3, n_heads * hd), 27).to(DEV)
    partial = torch.empty(k.attn_decode_workspace_floats(3, n_heads, hd, splits), device=DEV)
    got = []
    for simple in (False, True):
        k.FORCE_SIMPLE = simple
        try:
            out = torch.full((3, n_heads * hd), 7.0, device=DEV)
            k.attn_decode(q, kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots), i32(lens), out, partial, n_heads, n_kv, hd, 0, splits)
        finally:
            k.FORCE_SIMPLE = False
        got.append(out)
    # sums of at most 300 terms, weights that sum to one, in two orders
    assert torch.isfinite(got[1]).all() and bool(((got[0] - got[1]).abs() <= 2 * 300 * 2.0 ** -24 * 5.0).all())


# the splits merged by the last workgroup to arrive: against the kernel that merges them, launch after launch with the same
# counters; splits that find nothing to do, a padding row, more splits than lanes, several groups of 16 heads, a sink logit
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd,window,lens,splits,sink", [
    (4, 2, 16, 0, [5, 640], 2, False), (8, 2, 128, 0, [3000, 3, 700], 16, False), (34, 2, 64, 0, [300, 65], 3, True),
    (5, 1, 80, 100, [700, 64], 5, True), (2, 1, 32, 0, [70 * 64 * 4], 70, False), (40, 1, 128, 0, [900], 9, False),
    (3, 1, 256, 0, [400, 1], 4, False), (4, 2, 256, 0, [400, 1], 4, False), (8, 2, 64, 0, [64 * 17, 200], 17, True), (2, 2, 192, 0, [64 * 33, 64 * 66], 33, False)])
def test_attn_decode_merged_by_the_last_workgroup(n_heads, n_kv, hd, window, lens, splits, sink, dtype):
    k = K()
    B = len(lens)
    kp, vp, bt, slots, ring, keys, vals = paged_case(lens, n_kv, hd, window, dtype, 20)
    kp, vp, bt = kp.to(DEV), vp.to(DEV), bt.to(DEV)
    logit = rnd((n_heads,), 62).to(DEV) if sink else None
    counters = torch.zeros(k.attn_decode_counters(B + 1, n_heads, n_kv), dtype=torch.int32, device=DEV)
    for turn in range(3):
        q = torch.cat([rnd((B, n_heads * hd), 80 + turn, dtype), torch.zeros((1, n_heads * hd), dtype=dtype)]).to(DEV)
        got = []
        for c in (None, counters):
            out = torch.full((B + 1, n_heads * hd), 7.0, dtype=dtype, device=DEV)
            lse = torch.full((B + 1, n_heads), 7.0, device=DEV)
            partial = torch.full((k.attn_decode_workspace_floats(B + 1, n_heads, hd, splits),), float("nan"), device=DEV)
            k.attn_decode(q, kp, vp, bt, ring, i32(slots + [-1]), i32(lens + [0]), out, partial, n_heads, n_kv, hd, window, splits,
                          lse=lse, sink_logit=logit, counters=c)
            got.append((out.double(), lse.double()))
        # the same partial results, added in the same order: the same bits
        (a, la), (b, lb) = got
        assert torch.isfinite(b).all() and torch.equal(a, b) and torch.equal(la, lb)
        assert int(counters.abs().sum()) == 0
    with pytest.raises(ValueError):
        k.attn_decode(q, kp, vp, bt, ring, i32(slots + [-1]), i32(lens + [0]), out, partial, n_heads, n_kv, hd, window, splits,
                      counters=counters[:-1])


# more heads than a workgroup has waves: the kernel behind merges (inside, the waves would take the heads in turn), so whatever
# the counters hold is left alone
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd", [(5, 1, 64), (16, 2, 128), (40, 1, 96), (3, 1, 256), (16, 1, 192)])
def test_attn_decode_of_many_heads_is_merged_behind(n_heads, n_kv, hd, dtype):
    k = K()
    lens, splits = [700, 64], 3
    kp, vp, bt, slots, ring, _, _ = paged_case(lens, n_kv, hd, 0, dtype, 21)
    q = rnd((2, n_heads * hd), 22, dtype).to(DEV)
    partial = torch.empty(k.attn_decode_workspace_floats(2, n_heads, hd, splits), device=DEV)
    counters = torch.full((k.attn_decode_counters(2, n_heads, n_kv),), 1000, dtype=torch.int32, device=DEV)
    got = []
    for c in (None, counters):
        out = torch.full((2, n_heads * hd), 7.0, dtype=dtype, device=DEV)
        k.attn_decode(q, kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots), i32(lens), out, partial, n_heads, n_kv, hd, 0, splits,
                      counters=c)
        got.append(out)
    assert torch.equal(got[0], got[1]) and int((counters - 1000).abs().sum()) == 0


# float32 on the matrix cores against the general kernels: head sizes with pages in rows and in blocks, one tile and many, a
# window, blocks of positions, every shape of the scores, one split and several, more than 16 heads a group, rows in another
# order with splits of the longest sequence's size, a value that is infinite (a query that does not see it must not notice)
@pytest.mark.parametrize("shape", ["plain", "bias", "softcap", "sink", "slopes", "log", "infinite"])
@pytest.mark.parametrize("n_heads,n_kv,hd,window,block,lens,splits", [
    (4, 2, 64, 0, 0, [5, 64, 65], 1), (6, 3, 80, 100, 0, [130, 300], 3), (8, 2, 128, 0, 0, [200, 1, 129], 2),
    (18, 1, 64, 70, 0, [150, 64], 1), (3, 3, 96, 0, 96, [257, 17], 2), (2, 1, 112, 0, 0, [66], 1)])
def test_attention_float32_on_the_matrix_cores(n_heads, n_kv, hd, window, block, lens, splits, shape):
    k = K()
    T, B = sum(lens), len(lens)
    more = {"bias": {"score_bias": rnd((n_heads, 50), 61).to(DEV)}, "softcap": {"softcap": 2.5},
            "sink": {"sink_logit": rnd((n_heads,), 62).to(DEV)}, "slopes": {"slopes": rnd((n_heads,), 63, scale=0.1).abs().to(DEV)},
            "log": {"log_distance": (rnd((n_heads,), 64).abs().to(DEV), rnd((n_heads,), 65).abs().to(DEV))}}.get(shape, {})
    q, kk, v = (rnd((T, n * hd), 66 + i) for i, n in enumerate((n_heads, n_kv, n_kv)))
    if shape == "infinite":
        v[lens[0] - 1, 0] = float("inf")             # the first sequence's last position, which only its last query sees
        v[T - lens[-1], -1] = float("-inf")          # the last sequence's first position
    cu = np.concatenate([[0], np.cumsum(lens)])
    seq = np.repeat(np.arange(B), lens)
    pos = np.concatenate([np.arange(n) for n in lens])
    ks, vs, tile0 = stage(kk, v, lens, n_kv, hd, torch.float32)
    kp, vp, bt, slots, ring, _, _ = paged_case(lens, n_kv, hd, window, torch.float32, 20, stored=False)
    if shape == "infinite":
        for b, n in enumerate(lens):                 # the longest sequence's last value, and one a page or so before it
            for at in {n - 1, max(0, n - 70)}:
                vp[bt[slots[b], at // 64 % ring], 0, 3, at % 64] = float("inf")
    kp, vp = pages_as_stored(kp, vp)
    qd = rnd((B, n_heads * hd), 70)
    got = {}
    for simple in (False, True):
        out, o32, lse = (torch.full((T, n), 7.0, device=DEV) for n in (n_heads * hd, n_heads * hd, n_heads))
        dec, dlse = (torch.full((B, n), 7.0, device=DEV) for n in (n_heads * hd, n_heads))
        partial = torch.empty(k.attn_decode_workspace_floats(B, n_heads, hd, splits), device=DEV)
        k.FORCE_SIMPLE = simple
        try:
            k.attn_prefill(q.to(DEV), ks.to(DEV), vs.to(DEV), out, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv, hd,
                           window, lse=lse, out_f32=o32, block=block, **more)
            k.attn_decode(qd.to(DEV), kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots), i32(lens), dec, partial, n_heads,
                          n_kv, hd, window, splits, lse=dlse, block=block, step_max_len=None if simple else i32([max(lens)]),
                          seq_order=None if simple else i32(list(range(B))[::-1]), **more)
        finally:
            k.FORCE_SIMPLE = False
        got[simple] = [t.cpu().double() for t in (out, o32, lse, dec, dlse)]
    # both sum the same terms in float32 in another order: scores of a few tens off by 1e-5 of themselves at most, and the
    # probabilities with them
    for what, a, b in zip(("prefill", "prefill unrounded", "prefill lse", "decode", "decode lse"), got[False], got[True]):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a[a.isinf()], b[a.isinf()]) and torch.equal(a.isinf(), b.isinf()), what
        fine = b.isfinite()
        err = ((a - b).abs()[fine] / b[fine].abs().clamp(min=1.0)).max().item()
        assert err <= 2e-5, "%s: %.3e" % (what, err)
    assert shape == "infinite" or got[False][0].isfinite().all()


def _attn_decode_case(n_heads, n_kv, hd, window, lens, splits, dtype, simple, step_max_len):
    k = K()
    B = len(lens)
    kp, vp, bt, slots, ring, keys, vals = paged_case(lens, n_kv, hd, window, dtype, 20)
    q = rnd((B, n_heads * hd), 16, dtype)
    # one padding row at the end
    qd = torch.cat([q, torch.zeros((1, n_heads * hd), dtype=dtype)]).to(DEV)
    out = torch.full((B + 1, n_heads * hd), 5.0, dtype=dtype, device=DEV)
    partial = torch.empty(k.attn_decode_workspace_floats(B + 1, n_heads, hd, splits), device=DEV)
    k.FORCE_SIMPLE = simple
    try:
        k.attn_decode(qd, kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots + [-1]), i32(lens + [0]), out, partial,
                      n_heads, n_kv, hd, window, splits, step_max_len=None if step_max_len is None else i32([step_max_len]),
                      seq_order=None if step_max_len is None else i32(list(np.random.default_rng(5).permutation(B + 1))))
    finally:
        k.FORCE_SIMPLE = False
    for b, n in enumerate(lens):
        want = one_query_reference(q[b].double().reshape(n_heads, hd), keys[b], vals[b], window).reshape(-1)
        close(out[b], want, dtype, "decode attention row %d" % b)
    assert (out[B] == 0).all()


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd,window,lens,n_bias", [
    (4, 2, 16, 0, [5, 130, 64], 200), (6, 3, 64, 70, [300, 1], 40), (8, 2, 128, 0, [257], 300), (3, 1, 48, 20, [90, 65], 7),
    (40, 8, 128, 0, [1500], 900), (40, 8, 96, 200, [1100, 1200], 64), (12, 4, 32, 0, [1300], 2000), (16, 1, 64, 0, [70, 2], 3),
    (6, 2, 80, 0, [300, 65], 100), (10, 5, 112, 40, [200], 50), (36, 2, 64, 0, [150, 70], 90)])
def test_attn_with_a_score_bias(n_heads, n_kv, hd, window, lens, n_bias, dtype, simple):
    """A term added to every score by the distance of query and key (a table a head, the last entry for every
    distance beyond it): prompt and decode kernels against a float64 softmax with the same term.  The table is steep
    (a slope a head plus noise), so that dropping it, taking another head's row or counting the distance from the
    wrong end changes the result by far more than rounding.  Both kinds of kernels take it; the long prompts reach
    each launch shape of the matrix-core prompt kernel."""
    k = K()
    k.FORCE_SIMPLE = simple
    try:
        _score_bias_case(k, n_heads, n_kv, hd, window, lens, n_bias, dtype)
    finally:
        k.FORCE_SIMPLE = False


def _score_bias_case(k, n_heads, n_kv, hd, window, lens, n_bias, dtype):
    slopes = 2.0 ** -(torch.arange(n_heads, dtype=torch.float64) * 3.0 / n_heads)
    bias = (-slopes[:, None] * torch.arange(n_bias, dtype=torch.float64)[None, :] + rnd((n_heads, n_bias), 77).double()).float()
    T = sum(lens)
    q = rnd((T, n_heads * hd), 13, dtype)
    kk = rnd((T, n_kv * hd), 14, dtype)
    v = rnd((T, n_kv * hd), 15, dtype)
    cu = np.concatenate([[0], np.cumsum(lens)])
    seq = np.repeat(np.arange(len(lens)), lens)
    pos = np.concatenate([np.arange(n) for n in lens])
    ks, vs, tile0 = stage(kk, v, lens, n_kv, hd, dtype)
    out = torch.empty((T, n_heads * hd), dtype=dtype, device=DEV)
    k.attn_prefill(q.to(DEV), ks.to(DEV), vs.to(DEV), out, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv, hd,
                   window, score_bias=bias.to(DEV))
    want, plain, o = [], [], 0
    for n in lens:
        want.append(masked_attention_float64(q[o:o + n], kk[o:o + n], v[o:o + n], n_heads, n_kv, hd, window, bias))
        plain.append(masked_attention_float64(q[o:o + n], kk[o:o + n], v[o:o + n], n_heads, n_kv, hd, window))
        o += n
    want, plain = torch.cat(want), torch.cat(plain)
    assert (want - plain).abs().max() > 0.1                     # the bias matters here
    close(out, want, dtype, "prefill attention with a score bias")
    # decode: the last query of every sequence over the cache pages
    B = len(lens)
    kp, vp, bt, slots, ring, keys, vals = paged_case(lens, n_kv, hd, window, dtype, 20)
    qd = rnd((B, n_heads * hd), 16, dtype)
    outd = torch.empty((B, n_heads * hd), dtype=dtype, device=DEV)
    partial = torch.empty(k.attn_decode_workspace_floats(B, n_heads, hd, 3), device=DEV)
    k.attn_decode(qd.to(DEV), kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots), i32(lens), outd, partial,
                  n_heads, n_kv, hd, window, 3, score_bias=bias.to(DEV))
    for b, n in enumerate(lens):
        lo = max(0, n - window) if window else 0
        got_want = torch.zeros((n_heads, hd), dtype=torch.float64)
        for h in range(n_heads):
            g = h // (n_heads // n_kv)
            sc = keys[b][lo:n, g].double() @ qd[b].double().reshape(n_heads, hd)[h] / math.sqrt(hd)
            sc = sc + bias[h].double()[(n - 1 - torch.arange(lo, n)).clamp(0, n_bias - 1)]
            got_want[h] = torch.softmax(sc, dim=0) @ vals[b][lo:n, g].double()
        close(outd[b], got_want.reshape(-1), dtype, "decode attention with a score bias, row %d" % b)
    with pytest.raises(Exception):                              # a table for another number of heads
        k.attn_decode(qd.to(DEV), kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots), i32(lens), outd, partial,
                      n_heads, n_kv, hd, window, 3, score_bias=bias[:-1].contiguous().to(DEV))


@pytest.mark.parametrize("dtype", DTYPES)
def test_attn_decode_finds_a_far_key(dtype):
    """One key among a thousand, in an early page, carries all the weight: the query
    is scaled along that key, so a kernel that skips or misplaces a page misses it."""
    k = K()
    n_heads, n_kv, hd, n = 4, 1, 64, 1000
    for far in (3, 64 * 7 + 63, 998):
        kp, vp, bt, slots, ring, keys, vals = paged_case([n], n_kv, hd, 0, dtype, 30)
        q = (keys[0][far, 0].double() * 40.0).to(dtype).repeat(n_heads)[None]
        out = torch.empty((1, n_heads * hd), dtype=dtype, device=DEV)
        partial = torch.empty(k.attn_decode_workspace_floats(1, n_heads, hd, 5), device=DEV)
        k.attn_decode(q.to(DEV), kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots), i32([n]), out, partial, n_heads,
                      n_kv, hd, 0, 5)
        got = out.cpu().double().reshape(n_heads, hd)
        assert (got - vals[0][far, 0].double()).abs().max() < 0.05, far

@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hd,window,n", [(64, 70, 300), (128, 64, 200), (128, 100, 513), (32, 16, 90), (48, 33, 200), (112, 64, 150), (16, 8, 70)])
def test_attn_window_edge_decides(hd, window, n, dtype, simple):
    """The key just outside the window has by far the largest score and a value of 1000; the key
    just inside has the next largest and a value of 7.  A window off by one, in either kernel,
    gives 1000 or loses the 7: among a hundred random keys it would hide in the rounding."""
    k = K()
    n_heads, n_kv = 4, 2
    unit = torch.zeros(hd, dtype=torch.float64)
    unit[3] = 1.0
    k.FORCE_SIMPLE = simple
    try:
        # decode: the query at position n - 1 sees positions n - window ... n - 1
        kp, vp, bt, slots, ring, keys, vals = paged_case([n], n_kv, hd, window, dtype, 40, stored=False)
        inside, outside = n - window, n - window - 1
        PAGE = k.PAGE
        for pos, strength, value in ((inside, 30.0, 7.0), (outside, 60.0, 1000.0)):
            page = int(bt[slots[0], (pos // PAGE) % ring])
            if pos // PAGE > (n - 1) // PAGE - ring:          # the ring still holds this position's page
                kp[page, :, pos % PAGE, :] = (unit * strength).to(dtype)
                vp[page, :, :, pos % PAGE] = value
        kp, vp = pages_as_stored(kp, vp)
        q = (unit * 8.0).to(dtype).repeat(n_heads)[None]
        out = torch.empty((1, n_heads * hd), dtype=dtype, device=DEV)
        partial = torch.empty(k.attn_decode_workspace_floats(1, n_heads, hd, 3), device=DEV)
        k.attn_decode(q.to(DEV), kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots), i32([n]), out, partial, n_heads,
                      n_kv, hd, window, 3)
        assert (out.cpu().double() - 7.0).abs().max() < 0.1, "decode"

        # prefill: keys grow stronger towards the past, so that for query i the strongest visible key is the
        # oldest one, i - window + 1, and the one before it would be stronger still.  The strength T - j is
        # split over two elements (16 a + b) so that bfloat16 holds it exactly; scores of neighbours differ by 16.
        T = n
        s_q = 16.0 * math.sqrt(hd)
        qrow = torch.zeros(hd, dtype=torch.float64)
        qrow[3], qrow[4] = 16.0 * s_q, s_q
        qq = qrow.to(dtype).repeat(T, n_heads)
        kk = torch.zeros((T, n_kv * hd), dtype=dtype)
        v = torch.zeros((T, n_kv * hd), dtype=dtype)
        for j in range(T):
            krow = torch.zeros(hd, dtype=torch.float64)
            krow[3], krow[4] = (T - j) // 16, (T - j) % 16
            kk[j] = krow.to(dtype).repeat(n_kv)
            v[j] = float(j % 50)
        ks, vs, tile0 = stage(kk, v, [T], n_kv, hd, dtype)
        out = torch.empty((T, n_heads * hd), dtype=dtype, device=DEV)
        k.attn_prefill(qq.to(DEV), ks.to(DEV), vs.to(DEV), out, i32([0, T]), i32(tile0), i32([0] * T),
                       i32(list(range(T))), n_heads, n_kv, hd, window)
        got = out.cpu().double()[:, 0]
        want = torch.tensor([float(max(0, i - window + 1) % 50) for i in range(T)], dtype=torch.float64)
        assert (got - want).abs().max() < 0.1, "prefill, first bad position %d" % int(((got - want).abs() >= 0.1).nonzero()[0])
    finally:
        k.FORCE_SIMPLE = False



def test_attn_vector_of_the_reference():
    """src/test.cpp:67-126 through both attention kernels (head size padded from 3 to 16 with zeros)."""
    k = K()
    hd = 16
    q = torch.zeros((4, 2 * hd))
    q[3, 1], q[3, hd + 2] = 1e4, 1e4
    kv = torch.zeros((4, hd))
    kv[0, 0], kv[1, 1], kv[2, 2], kv[3, 0] = 1, 1, 1, -1
    out = torch.empty((4, 2 * hd), device=DEV)
    ks, vs, tile0 = stage(kv, kv, [4], 1, hd, torch.float32, poison=False)
    # the reference divides by sqrt(3); here sqrt(16): the scores stay far apart, the result is the same
    k.attn_prefill(q.to(DEV), ks.to(DEV), vs.to(DEV), out, i32([0, 4]), i32(tile0), i32([0] * 4), i32([0, 1, 2, 3]), 2,
                   1, hd, 0)
    got = out.cpu()[3].reshape(2, hd)
    assert torch.allclose(got[0, :3], torch.tensor([0., 1, 0]), atol=1e-4)
    assert torch.allclose(got[1, :3], torch.tensor([0., 0, 1]), atol=1e-4)


# ------------------------------------------------------------------ attention sinks

def window_lse_float64(q, k, window):
    """Logarithm of the sum of exp(score) over the keys a window shows, [T, n_heads]."""
    T, n_heads, hd = q.shape
    group = n_heads // k.shape[1]
    out = torch.zeros((T, n_heads), dtype=torch.float64)
    for i in range(T):
        lo = max(0, i - window + 1) if window else 0
        for h in range(n_heads):
            out[i, h] = torch.logsumexp((k[lo:i + 1, h // group].double() @ q[i, h].double()) / math.sqrt(hd), 0)
    return out


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd,rd,window,sinks,lens", [
    (4, 2, 16, 16, 5, 2, [30, 3, 1, 8]), (6, 3, 48, 24, 37, 3, [150, 41]), (8, 2, 128, 128, 94, 2, [300, 96, 97]),
    (4, 1, 64, 32, 70, 4, [200, 64]), (2, 2, 32, 0, 9, 1, [40])])
def test_attn_prefill_with_sinks(n_heads, n_kv, hd, rd, window, sinks, lens, dtype, simple):
    """Sinks stored from the staging area, the attention kernel's log-sum-exp, and the sinks behind the
    window mixed in with their keys turned, against the plain implementation's closed form."""
    k = K()
    T, B = sum(lens), len(lens)
    q = rnd((T, n_heads * hd), 33, dtype)
    kk = rnd((T, n_kv * hd), 34, dtype)
    v = rnd((T, n_kv * hd), 35, dtype)
    cu = np.concatenate([[0], np.cumsum(lens)])
    seq = np.repeat(np.arange(B), lens)
    pos = np.concatenate([np.arange(n) for n in lens])
    ks, vs, tile0 = stage(kk, v, lens, n_kv, hd, dtype)
    n_slots = B + 3
    slots = [int(x) for x in np.random.default_rng(5).permutation(n_slots)[:B]]
    sink_k = torch.full((n_slots, n_kv, sinks, hd), 7.0, dtype=dtype, device=DEV)
    sink_v = torch.full((n_slots, n_kv, sinks, hd), 7.0, dtype=dtype, device=DEV)
    table = make_table(max(lens) + 1, hd, rd, 80.0).to(DEV) if rd else None
    out = torch.empty((T, n_heads * hd), dtype=dtype, device=DEV)
    lse = torch.empty((T, n_heads), dtype=torch.float32, device=DEV)
    qd, ksd, vsd = q.to(DEV), ks.to(DEV), vs.to(DEV)
    k.FORCE_SIMPLE = simple
    try:
        k.sink_store(ksd, vsd, i32(tile0), i32(slots), i32(lens), sink_k, sink_v)
        # the unrounded result beside the rounded one: the row with the sinks mixed in is then rounded once
        o32 = torch.full((T, n_heads * hd), float("nan"), device=DEV) if dtype == torch.bfloat16 else None
        k.attn_prefill(qd, ksd, vsd, out, i32(cu), i32(tile0), i32(seq), i32(pos), n_heads, n_kv, hd, window, lse=lse,
                       out_f32=o32)
        plain_window = out.clone()
        if o32 is not None:
            assert torch.equal(o32.to(dtype), out)
        k.attn_sink_mix(qd, out, lse, sink_k, sink_v, i32(seq), i32(pos), i32(slots), table, n_heads, rd, window,
                        src_f32=o32)
    finally:
        k.FORCE_SIMPLE = False
    inv = R.rope_inv_freq(hd, rd, 80.0)
    o = 0
    for b, n in enumerate(lens):
        qb, kb, vb = (t[o:o + n].reshape(n, -1, hd) for t in (q, kk, v))
        have = min(n, sinks)
        assert torch.equal(sink_k[slots[b], :, :have].cpu(), kb[:have].transpose(0, 1)), "stored sink keys"
        assert torch.equal(sink_v[slots[b], :, :have].cpu(), vb[:have].transpose(0, 1)), "stored sink values"
        assert (sink_k[slots[b], :, have:] == 7.0).all(), "sinks that the sequence does not have yet stay untouched"
        close(lse[o:o + n], window_lse_float64(qb, kb, window), torch.float32, "log-sum-exp of sequence %d" % b)
        want = R.attention(qb, kb, vb, window, sinks, inv).reshape(n, -1)
        close(out[o:o + n], want, dtype, "prefill attention with sinks, sequence %d" % b)
        if n > window + 1:         # the sinks matter: without them the result is another
            assert (plain_window[o:o + n].double().cpu() - want).abs().max() > 1e-2
        o += n
    unused = [s for s in range(n_slots) if s not in slots]
    assert (sink_k[unused] == 7.0).all() and (sink_v[unused] == 7.0).all()


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_heads,n_kv,hd,rd,window,sinks,lens,splits", [
    (4, 2, 16, 16, 5, 2, [30, 7, 6, 1, 2], 1), (6, 3, 48, 24, 37, 3, [150, 41, 40, 39, 3], 2),
    (8, 2, 128, 128, 94, 2, [300, 96, 97, 95], 1), (32, 8, 128, 128, 94, 2, [700, 200], 3),
    (4, 1, 64, 32, 70, 4, [200, 73, 74, 2], 2), (2, 2, 32, 0, 9, 1, [40, 1], 70)])
def test_attn_decode_with_sinks(n_heads, n_kv, hd, rd, window, sinks, lens, splits, dtype, simple):
    """A decode step's sinks: the sequences still at their first positions store the key they just wrote;
    the others have theirs from before; the merge of the splits takes in the sinks that a query's window
    no longer covers."""
    k = K()
    B = len(lens)
    kp, vp, bt, slots, ring, keys, vals = paged_case(lens, n_kv, hd, window, dtype, 40)
    n_slots = bt.shape[0]
    q = rnd((B, n_heads * hd), 36, dtype)
    sink_k = torch.full((n_slots, n_kv, sinks, hd), float("nan"), dtype=dtype)
    sink_v = torch.full((n_slots, n_kv, sinks, hd), float("nan"), dtype=dtype)
    for b, n in enumerate(lens):          # what earlier steps stored; the newest position is this step's to store
        have = min(sinks, n - 1)
        sink_k[slots[b], :, :have] = keys[b][:have].transpose(0, 1)
        sink_v[slots[b], :, :have] = vals[b][:have].transpose(0, 1)
    sink_k, sink_v = sink_k.to(DEV), sink_v.to(DEV)
    table = make_table(max(lens) + 1, hd, rd, 80.0).to(DEV) if rd else None
    qd = torch.cat([q, torch.zeros((1, n_heads * hd), dtype=dtype)]).to(DEV)
    out = torch.full((B + 1, n_heads * hd), 5.0, dtype=dtype, device=DEV)
    partial = torch.empty(k.attn_decode_workspace_floats(B + 1, n_heads, hd, splits), device=DEV)
    seq_slot, seq_len = i32(slots + [-1]), i32(lens + [0])
    k.FORCE_SIMPLE = simple
    try:
        k.attn_decode(qd, kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, seq_slot, seq_len, out, partial, n_heads, n_kv, hd,
                      window, splits, sinks=(sink_k, sink_v, table, rd, True))
    finally:
        k.FORCE_SIMPLE = False
    inv = R.rope_inv_freq(hd, rd, 80.0)
    for b, n in enumerate(lens):
        have = min(sinks, n)
        assert torch.equal(sink_k[slots[b], :, :have].cpu(), keys[b][:have].transpose(0, 1)), "sink keys of row %d" % b
        assert torch.equal(sink_v[slots[b], :, :have].cpu(), vals[b][:have].transpose(0, 1)), "sink values of row %d" % b
        qf = torch.zeros((n, n_heads, hd), dtype=torch.float64)
        qf[-1] = q[b].double().reshape(n_heads, hd)
        want = R.attention(qf, keys[b], vals[b], window, sinks, inv)[-1].reshape(-1)
        close(out[b], want, dtype, "decode attention with sinks, row %d (%d keys)" % (b, n))
    assert (out[B] == 0).all()


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
def test_attn_decode_leaves_the_log_sum_exp(dtype, simple):
    k = K()
    n_heads, n_kv, hd, window = 8, 2, 128, 94
    for lens, splits in (([300, 5, 96], 1), ([300, 5, 96], 3)):
        B = len(lens)
        kp, vp, bt, slots, ring, keys, vals = paged_case(lens, n_kv, hd, window, dtype, 41)
        q = rnd((B, n_heads * hd), 37, dtype)
        out = torch.empty((B, n_heads * hd), dtype=dtype, device=DEV)
        lse = torch.empty((B, n_heads), dtype=torch.float32, device=DEV)
        partial = torch.empty(k.attn_decode_workspace_floats(B, n_heads, hd, splits), device=DEV)
        k.FORCE_SIMPLE = simple
        try:
            k.attn_decode(q.to(DEV), kp.to(DEV), vp.to(DEV), bt.to(DEV), ring, i32(slots), i32(lens), out, partial,
                          n_heads, n_kv, hd, window, splits, lse=lse)
        finally:
            k.FORCE_SIMPLE = False
        for b, n in enumerate(lens):
            qf = torch.zeros((n, n_heads, hd), dtype=torch.float64)
            qf[-1] = q[b].double().reshape(n_heads, hd)
            close(lse[b], window_lse_float64(qf, keys[b], window)[-1], torch.float32, "log-sum-exp of row %d" % b)


@pytest.mark.parametrize("dtype", DTYPES)
def test_a_sink_far_behind_the_window_decides(dtype):
    """One sink key is made so that, turned by the number of positions the sinks have been pushed on at
    this query (position - window - sinks + 1), it is the query itself, at a position many windows on:
    the result is that sink's value if and only if the key is turned by exactly that much."""
    k = K()
    hd, window, sinks, n = 64, 20, 2, 333
    table = make_table(n, hd, hd, 4.0)
    inv = R.rope_inv_freq(hd, hd, 4.0)
    base = torch.zeros(hd, dtype=torch.float64)
    base[0::2] = 6.0                                   # every pair along its first axis
    pos = n - 1
    turn = pos - window - sinks + 1
    qrot = R.rope_interleaved(base.reshape(1, 1, hd), torch.tensor([pos]), inv).reshape(1, hd)
    kj = R.rope_interleaved(base.reshape(1, 1, hd), torch.tensor([pos - turn]), inv).reshape(hd)
    sink_k = torch.zeros((1, 1, sinks, hd), dtype=dtype)
    sink_v = torch.zeros((1, 1, sinks, hd), dtype=dtype)
    sink_k[0, 0, 1] = kj.to(dtype)
    sink_v[0, 0, 0, 0] = 1.0
    sink_v[0, 0, 1, 1] = 1.0
    out = torch.zeros((1, hd), dtype=dtype, device=DEV)
    out[0, 2] = 1.0                                    # what the window gave
    lse = torch.full((1, 1), 100.0, dtype=torch.float32, device=DEV)
    k.attn_sink_mix(qrot.to(dtype).to(DEV), out, lse, sink_k.to(DEV), sink_v.to(DEV), i32([0]), i32([pos]), i32([0]),
                    table.to(DEV), 1, hd, window)
    got = out.cpu().double()[0]
    # turned right, the sink scores |base|^2 / sqrt(hd) = 144 against 100 for the window; one position off
    # it would score 120 (the plain rotation says so) and still win, hence the second run below
    assert got[1] > 0.999 and got[0] < 1e-3 and got[2] < 1e-3, got[:3]
    right = R.rope_interleaved(kj.reshape(1, 1, hd), torch.tensor([turn]), inv).reshape(hd)
    assert abs(float(right @ qrot[0]) / math.sqrt(hd) - 144.0) < 1e-6
    for wrong in (turn - 1, turn + 1, 0):
        off = R.rope_interleaved(kj.reshape(1, 1, hd), torch.tensor([wrong]), inv).reshape(hd)
        assert float(off @ qrot[0]) / math.sqrt(hd) < 121.0
    # with the window at 132 a sink turned one position off (120) would lose; the right one (144) wins
    out2 = torch.zeros((1, hd), dtype=dtype, device=DEV)
    out2[0, 2] = 1.0
    lse.fill_(132.0)
    k.attn_sink_mix(qrot.to(dtype).to(DEV), out2, lse, sink_k.to(DEV), sink_v.to(DEV), i32([0]), i32([pos]), i32([0]),
                    table.to(DEV), 1, hd, window)
    got2 = out2.cpu().double()[0]
    assert got2[1] > 0.999 and got2[2] < 1e-3, got2[:3]


# ------------------------------------------------------------------ sampling

def test_argmax_and_sample():
    k = K()
    V = 1000
    g = torch.Generator().manual_seed(40)
    logits = torch.randn((6, V), generator=g) * 3
    logits[0, 17] = logits[0, 900] = 50.0                # a tie: the lowest index wins
    logits[1, V - 1] = 60.0
    out = torch.empty(6, dtype=torch.int32, device=DEV)
    k.argmax(logits.to(DEV), out)
    assert out.cpu().tolist() == [R.sample_argmax(l) for l in logits]
    assert out[0] == 17 and out[1] == V - 1
    for temp in (1.0, 0.8, 2.5):
        u = torch.tensor([0.0, 0.999999, 0.5, 0.25, 0.9, 0.1])
        k.sample(logits.to(DEV), u.to(DEV), temp, out)
        got = out.cpu().tolist()
        for r in range(6):
            p = torch.softmax(logits[r].double() / temp, 0)
            c = torch.cumsum(p, 0)
            want = R.sample_temperature(logits[r], temp, float(u[r]))
            # equal up to an edge of the running sum: the picked token's interval contains u within rounding
            lo = float(c[got[r]] - p[got[r]])
            assert got[r] == want or (lo - 1e-5 <= float(u[r]) <= float(c[got[r]]) + 1e-5), (temp, r, got[r], want)
    # the distribution on a toy of 4 logits: frequencies match softmax
    l4 = torch.tensor([[0.0, 1.0, 2.0, -1.0]]).repeat(4000, 1)
    u = torch.rand(4000, generator=g)
    out = torch.empty(4000, dtype=torch.int32, device=DEV)
    k.sample(l4.to(DEV), u.to(DEV), 1.0, out)
    freq = torch.bincount(out.cpu().long(), minlength=4).double() / 4000
    assert (freq - torch.softmax(l4[0].double(), 0)).abs().max() < 0.03
    prob = torch.empty(6, device=DEV)
    k.token_prob(logits.to(DEV), i32([0, 1, 2, 3, 4, 999]), prob)
    want = [R.sample_prob(logits[r], i) for r, i in enumerate([0, 1, 2, 3, 4, 999])]
    assert torch.allclose(prob.cpu().double(), torch.tensor(want, dtype=torch.float64), rtol=1e-4, atol=1e-9)


@pytest.mark.parametrize("V", [4, 7, 255, 1029, 32003, 128256])
def test_sampling_at_vocabularies_of_any_size(V):
    """Rows that do not start on a 16-byte boundary (odd V), fewer entries than a wave's tile, and
    vocabularies that give every wave several tiles: the first maximum, the walk of the running sum
    and the probability of a token against the plain functions."""
    k = K()
    g = torch.Generator().manual_seed(41 + V)
    n = 5
    logits = torch.randn((n, V), generator=g) * 3
    logits[0, 0] = logits[0, V - 1] = 40.0                   # ties at both ends: the first wins
    logits[1, V - 1] = 41.0                                  # the last entry (the scalar tail)
    logits[2, min(V - 1, 2)] = logits[2, V // 2] = 42.0
    dl = logits.to(DEV)
    out = torch.empty(n, dtype=torch.int32, device=DEV)
    k.argmax(dl, out)
    assert out.cpu().tolist() == [R.sample_argmax(l) for l in logits]
    flat = torch.randn((n, V), generator=g)                  # flat rows: the walk ends deep inside the row
    for rows, temp in ((logits, 1.0), (flat, 0.7), (flat, 3.0)):
        d = rows.to(DEV)
        for us in ([0.0, 0.999999, 0.5, 0.25, 0.9], [0.1, 0.33, 0.66, 0.75, 1.0]):
            u = torch.tensor(us)
            k.sample(d, u.to(DEV), temp, out)
            got = out.cpu().tolist()
            for r in range(n):
                assert 0 <= got[r] < V
                p = torch.softmax(rows[r].double() / temp, 0)
                c = torch.cumsum(p, 0)
                want = R.sample_temperature(rows[r], temp, float(u[r]))
                lo = float(c[got[r]] - p[got[r]])
                assert got[r] == want or (lo - 1e-5 <= float(u[r]) <= float(c[got[r]]) + 1e-5), (V, temp, r, got[r], want)
    idx = [0, V - 1, V // 2, min(V - 1, 3), V // 3]
    prob = torch.empty(n, device=DEV)
    k.token_prob(dl, i32(idx), prob)
    want = [R.sample_prob(logits[r], i) for r, i in enumerate(idx)]
    assert torch.allclose(prob.cpu().double(), torch.tensor(want, dtype=torch.float64), rtol=1e-4, atol=1e-9)


# ------------------------------------------------------------------ fused decode GEMMs

@pytest.mark.parametrize("M,N,Kd", [(1, 64, 256), (8, 4096 + 32, 136), (7, 100, 96), (3, 17000, 64), (2, 4096, 4096), (8, 48, 4096)])
def test_gemm_norm(M, N, Kd):
    """rmsnorm folded into the product: against the plain rmsnorm followed by a float64 product."""
    k = K()
    x = rnd((M, Kd), 50, scale=3.0)
    nw = 1 + 0.1 * rnd((Kd,), 51)
    w = rnd((N, Kd), 52, torch.bfloat16, scale=1 / math.sqrt(Kd))
    want = R.rmsnorm(x, nw, 1e-5) @ w.double().T
    out = torch.empty((M, N), device=DEV)
    k.gemm_norm(x.to(DEV), nw.to(DEV), 1e-5, w.to(DEV), out, k.EPI_STORE_F32)
    close(out, want, torch.bfloat16, "gemm_norm")          # the activations are rounded to bfloat16 on the way


@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("M,H,D", [(8, 14336, 4096), (1, 14336, 192), (16, 14336, 1024), (11, 13003, 64), (4, 12810, 320),
                                   (9, 20000, 128), (3, 28672, 256)])
def test_gemm_gated_wide_at_up_to_16_rows(M, H, D, act):
    """Up to 16 rows and a gated matrix wide enough for the workgroups of 128 weight rows: hidden widths that are no
    multiples of 8 or of 64, one and many stages of K, with and without the row scale of the norm chain; every hidden
    column is written, nothing beyond them."""
    from yalm_amd.parts.swiglu import interleave_gate_up
    k = K()
    act_fn, epi_code = gate(act)
    x = rnd((M, D), 53, torch.bfloat16, scale=2.0)
    wg = rnd((H, D), 55, torch.bfloat16, scale=1 / math.sqrt(D))
    wu = rnd((H, D), 56, torch.bfloat16, scale=1 / math.sqrt(D))
    w = interleave_gate_up(wg, wu).to(DEV)
    g, u = x.double() @ wg.double().T, x.double() @ wu.double().T
    out = torch.full((M + 1, H), 7.0, dtype=torch.bfloat16, device=DEV)
    k.gemm(x.to(DEV), w, out[:M], epi_code, hidden=H)
    close(out[:M], act_fn(g) * u, torch.bfloat16, "gated product")
    assert (out[M] == 7.0).all()
    # the same behind the norm chain: the sums are scaled row by row before the activation
    ss = (x.double() ** 2).sum(dim=1, keepdim=True).float() * torch.tensor([[0.25, 0.5, 0.25]])
    eps = 1e-5
    scale = 1.0 / torch.sqrt((x.double() ** 2).sum(dim=1, keepdim=True) / D + eps)
    out2 = torch.full((M + 1, H), 7.0, dtype=torch.bfloat16, device=DEV)
    k.gemm_chain(x.to(DEV), w, out2[:M], epi_code, hidden=H, scale_from=(ss.to(DEV).contiguous(), eps))
    close(out2[:M], act_fn(g * scale) * (u * scale), torch.bfloat16, "gated product with a row scale", factor=2.0)
    assert (out2[M] == 7.0).all()


@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("M,H,D", [(1, 176, 64), (8, 1000, 264), (5, 14336, 128)])
def test_gemm_norm_gated(M, H, D, act):
    from yalm_amd.parts.swiglu import interleave_gate_up
    k = K()
    x = rnd((M, D), 53, scale=2.0)
    nw = 1 + 0.1 * rnd((D,), 54)
    wg = rnd((H, D), 55, torch.bfloat16, scale=1 / math.sqrt(D))
    wu = rnd((H, D), 56, torch.bfloat16, scale=1 / math.sqrt(D))
    h = R.rmsnorm(x, nw, 1e-6)
    act_fn, epi_code = gate(act)
    want = act_fn(h @ wg.double().T) * (h @ wu.double().T)
    out = torch.empty((M, H), dtype=torch.bfloat16, device=DEV)
    k.gemm_norm(x.to(DEV), nw.to(DEV), 1e-6, interleave_gate_up(wg, wu).to(DEV), out, epi_code, hidden=H)
    close(out, want, torch.bfloat16, "gemm_norm gated", factor=1.5)


@pytest.mark.parametrize("n_heads,n_kv,hd,rd,D", [(4, 2, 16, 16, 64), (3, 1, 48, 48, 80), (6, 3, 32, 16, 96),
                                                   (32, 8, 128, 128, 256)])
def test_gemm_norm_qkv_rope(n_heads, n_kv, hd, rd, D):
    """norm + q/k/v + rotation + cache write in one kernel against the plain parts."""
    k = K()
    PAGE = k.PAGE
    M = 5
    pos = [0, 63, 64, 130, 7]
    slots = [3, 0, -1, 2, 1]                       # row 2 is a padding row
    Q, KV = n_heads * hd, n_kv * hd
    x = rnd((M, D), 57, scale=2.0)
    nw = 1 + 0.1 * rnd((D,), 58)
    w = rnd((Q + 2 * KV, D), 59, torch.bfloat16, scale=1 / math.sqrt(D))
    table = make_table(200, hd, rd, 10000.0)
    ring, n_pages = 4, 12
    bt = torch.arange(4 * ring, dtype=torch.int32).reshape(4, ring) % n_pages
    kp = torch.zeros((n_pages, n_kv, PAGE, hd), dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros((n_pages, n_kv, hd, PAGE), dtype=torch.bfloat16, device=DEV)
    q_out = torch.zeros((M, Q), dtype=torch.bfloat16, device=DEV)
    k.gemm_norm_qkv_rope(x.to(DEV), nw.to(DEV), 1e-5, w.to(DEV), q_out, kp, vp, bt.to(DEV), ring, i32(pos), i32(slots),
                         table.to(DEV), n_heads, n_kv, hd, rd)
    qkv = R.rmsnorm(x, nw, 1e-5) @ w.double().T
    f = R.rope_inv_freq(hd, rd, 10000.0)
    p = torch.tensor(pos)
    q_want = R.rope_interleaved(qkv[:, :Q].reshape(M, n_heads, hd), p, f).reshape(M, Q)
    k_want = R.rope_interleaved(qkv[:, Q:Q + KV].reshape(M, n_kv, hd), p, f)
    v_want = qkv[:, Q + KV:].reshape(M, n_kv, hd)
    close(q_out, q_want, torch.bfloat16, "q", factor=1.5)
    kp, vp = pages_as_rows(kp.cpu(), vp.cpu())
    touched = torch.zeros((n_pages, PAGE), dtype=torch.bool)
    for m in range(M):
        if slots[m] < 0:
            continue
        page, r = int(bt[slots[m], (pos[m] // PAGE) % ring]), pos[m] % PAGE
        close(kp[page, :, r, :], k_want[m], torch.bfloat16, "k row %d" % m, factor=1.5)
        close(vp[page, :, :, r], v_want[m], torch.bfloat16, "v row %d" % m, factor=1.5)
        touched[page, r] = True
    assert (kp.float().abs().sum(dim=(1, 3)) > 0).equal(touched)
    assert (vp.float().abs().sum(dim=(1, 2)) > 0).equal(touched)


# Workgroups of 96 weight rows, which take what 64 rows would leave to a second round of compute units: the fewest and the most rows, a
# last workgroup of one row, sums of one, two and seven stages of K
@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("N,Kd", [(16385, 128), (16417, 128), (24576, 64), (22113, 448)])
def test_decode_gemm_of_96_rows(M, N, Kd):
    from yalm_amd.parts.swiglu import interleave_gate_up
    k = K()
    x, w = rnd((M, Kd), 130, torch.bfloat16).to(DEV), rnd((N, Kd), 131, torch.bfloat16, scale=Kd ** -0.5).to(DEV)
    want = x.double() @ w.double().t()
    # float32 sums of exact products: K roundings of the sum of magnitudes
    bound = 2.0 ** -23 * Kd * (x.double().abs() @ w.double().abs().t())
    got = k.gemm(x, w, torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32).double()
    assert bool(((got - want).abs() <= bound).all())
    old = rnd((M, N), 132).to(DEV)
    got = k.gemm(x, w, old.clone(), k.EPI_ADD_F32).double()
    assert bool(((got - want - old.double()).abs() <= bound + 2.0 ** -23 * (want.abs() + old.double().abs())).all())
    H = N // 2
    wg = interleave_gate_up(w[:H], w[H:2 * H])
    out = k.gemm(x, wg, torch.full((M, H), 7.0, dtype=torch.bfloat16, device=DEV), k.EPI_GATED, hidden=H)
    g, u = want[:, :H], want[:, H:2 * H]
    close(out, (g / (1 + torch.exp(-g)) * u).cpu(), torch.bfloat16, "gated")


# Rows in turn over eight waves, K of fewer k tiles than waves and of many; the sum of squares over one wave (to 1,024), over four
# by 16 bytes (to 8,192) and element by element (beyond); one and two column tiles a workgroup
@pytest.mark.parametrize("M,N,Kd", [(1, 40, 32), (16, 100, 96), (3, 512, 256), (9, 4100, 1024), (13, 33, 1056), (16, 4112, 4096), (2, 50, 8192),
                                    (5, 16, 8224), (8, 17000, 2048)])
def test_gemm_norm_float32(M, N, Kd):
    """The norm folded into a float32 product has the bits of the norm's own kernel and the product behind it."""
    from yalm_amd.parts.swiglu import interleave_gate_up
    k = K()
    x, nw = rnd((M, Kd), 120, scale=3.0).to(DEV), (1 + 0.1 * rnd((Kd,), 121)).to(DEV)
    w = rnd((N, Kd), 122, scale=Kd ** -0.5).to(DEV)
    assert k.can_fuse_norm(M, Kd, torch.float32, N)
    h = k.rmsnorm(x, nw, torch.empty_like(x), 1e-5)
    got = k.gemm_norm(x, nw, 1e-5, w, torch.full((M, N), 7.0, device=DEV), k.EPI_STORE_F32)
    assert torch.equal(got, k.gemm(h, w, torch.empty_like(got), k.EPI_STORE_F32))
    H = N // 2 - 3
    gu = interleave_gate_up(w[:H], w[H:2 * H])
    if not k.can_fuse_norm(M, Kd, torch.float32, gu.shape[0], gate=True):
        return
    for epi in k.GATED:
        got = k.gemm_norm(x, nw, 1e-5, gu, torch.full((M, H), 7.0, device=DEV), epi, hidden=H)
        assert torch.equal(got, k.gemm(h, gu, torch.empty_like(got), epi, hidden=H))


def test_gemm_norm_float32_refuses_what_it_does_not_take():
    k = K()
    for M, N, Kd in ((17, 64, 64), (4, 8192, 4096), (4, 64, 48)):
        assert not k.can_fuse_norm(M, Kd, torch.float32, N)
        with pytest.raises(Exception):
            k.gemm_norm(torch.zeros((M, Kd), device=DEV), torch.ones(Kd, device=DEV), 1e-5, torch.zeros((N, Kd), device=DEV),
                        torch.empty((M, N), device=DEV), k.EPI_STORE_F32)


# Either side of the lines up to which a float32 step folds a norm into the product behind it: what follows from them is asked of the
# parts (whose weights' shapes are all that they look at)
@pytest.mark.parametrize("part,M,N,D,folded", [
    ("head", 1, 128256, 2048, False), ("head", 16, 128256, 1024, False), ("head", 3, 512, 256, True), ("head", 16, 8192, 1024, True),
    ("head", 1, 8193, 1024, False), ("head", 1, 4096, 1056, False), ("head", 17, 512, 256, False),
    ("mlp", 16, 8192, 1024, True), ("mlp", 1, 8224, 1024, False), ("mlp", 4, 2048, 2048, False),
    ("attention", 16, 6144, 4096, True), ("attention", 1, 8192, 1024, True), ("attention", 1, 12288, 2048, False)])
def test_float32_steps_fold_a_norm_where_it_pays(part, M, N, D, folded):
    from types import SimpleNamespace as NS
    from yalm_amd.parts.attention import GQAttention
    from yalm_amd.parts.embedding import LMHead
    from yalm_amd.parts.swiglu import SwiGLU
    w = torch.empty((N, D), device="meta")
    kind, fields = {"head": (LMHead, dict(weight=w)), "mlp": (SwiGLU, dict(w_gate_up=w, w_down=w, unit=None)),
                    "attention": (GQAttention, dict(wo=w, head_dim=64, q_dim=N // 2, kv_dim=N // 4))}[part]
    one = kind.__new__(kind)
    vars(one).update(fields, dim=D)
    ctx, norm = NS(mode="decode", normed={}), NS(fused=lambda: None)
    assert one.fuses_norm(norm, torch.empty((M, D), device="meta"), ctx) == folded


@pytest.mark.parametrize("n_heads,n_kv,hd,rd,D", [(4, 2, 16, 16, 64), (3, 1, 48, 32, 96), (6, 3, 32, 0, 96), (32, 8, 128, 128, 256)])
@pytest.mark.parametrize("M", [5, 11])
def test_gemm_norm_qkv_rope_float32(n_heads, n_kv, hd, rd, D, M):
    """norm + q/k/v + rotation + cache write of a float32 decode step in one kernel: the bits of the kernels one by one, which a step
    of 17 rows takes."""
    k = K()
    pos = ([0, 63, 64, 130, 7] + list(range(190, 196)))[:M]
    slots = ([3, 0, -1, 2, 1] + list(range(4, 10)))[:M]                    # row 2 is a padding row
    Q, KV = n_heads * hd, n_kv * hd
    x, nw = rnd((M, D), 57, scale=2.0).to(DEV), (1 + 0.1 * rnd((D,), 58)).to(DEV)
    w = rnd((Q + 2 * KV, D), 59, scale=1 / math.sqrt(D)).to(DEV)
    table = make_table(200, hd, rd, 10000.0).to(DEV) if rd else None
    ring, n_pages = 4, 44
    bt = torch.arange(11 * ring, dtype=torch.int32, device=DEV).reshape(11, ring)
    pages = [torch.zeros((2, n_pages, n_kv) + s, device=DEV) for s in ((k.PAGE, hd), (hd, k.PAGE))]
    q = torch.zeros((2, M, Q), device=DEV)
    assert k.can_fuse_norm(M, D, torch.float32, Q + 2 * KV)
    k.gemm_norm_qkv_rope(x, nw, 1e-5, w, q[0], pages[0][0], pages[1][0], bt, ring, i32(pos), i32(slots), table, n_heads, n_kv, hd, rd)
    h = k.rmsnorm(x, nw, torch.empty_like(x), 1e-5)
    qkv = k.gemm(h, w, torch.empty((M, Q + 2 * KV), device=DEV), k.EPI_STORE_F32)
    k.rope_kv_write(qkv, q[1], None, None, None, pages[0][1], pages[1][1], bt, ring, i32(list(range(M))), i32(pos), i32(slots),
                    i32([p + 1 for p in pos]), table, n_heads, n_kv, hd, rd)
    assert torch.equal(q[0], q[1])
    for p in pages:
        assert torch.equal(p[0], p[1]) and bool((p[0] != 0).any())


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("n_heads,n_kv,hd,rd,D", [(4, 2, 16, 16, 64), (3, 1, 48, 48, 80), (6, 3, 32, 16, 192),
                                                   (32, 8, 128, 128, 128), (24, 8, 128, 128, 64), (10, 5, 64, 64, 256)])
def test_gemm_chain_qkv_rope(n_heads, n_kv, hd, rd, D, M):
    """The q/k/v projection of a decode step from activations a producer emitted (already multiplied by the
    norm's weights, with partial sums of squares), with rotation and cache write in its epilogue; among the
    shapes the 6144 and 5120 weight rows of the big models' projections."""
    k = K()
    PAGE = k.PAGE
    rng = np.random.default_rng(M)
    pos = [int(p) for p in rng.integers(0, 190, size=M)]
    slots = [int(s) for s in rng.permutation(M + 2)[:M]]
    if M > 2:
        slots[2] = -1                                  # a padding row
    Q, KV = n_heads * hd, n_kv * hd
    x = rnd((M, D), 57, scale=2.0)
    nw = 1 + 0.1 * rnd((D,), 58)
    w = rnd((Q + 2 * KV, D), 59, torch.bfloat16, scale=1 / math.sqrt(D))
    xn = (x * nw).to(torch.bfloat16)
    parts = 3
    ss = torch.zeros((M, parts))
    for p_, cols in enumerate(np.array_split(np.arange(D), parts)):
        ss[:, p_] = (x[:, cols].double() ** 2).sum(dim=1).float()
    table = make_table(200, hd, rd, 10000.0)
    ring, n_pages = 3, 64
    bt = torch.tensor(rng.permutation(n_pages)[: (M + 2) * ring].reshape(M + 2, ring), dtype=torch.int32)
    kp = torch.zeros((n_pages, n_kv, PAGE, hd), dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros((n_pages, n_kv, hd, PAGE), dtype=torch.bfloat16, device=DEV)
    q_out = torch.zeros((M, Q), dtype=torch.bfloat16, device=DEV)
    k.gemm_chain_qkv_rope(xn.to(DEV), (ss.to(DEV), 1e-5), w.to(DEV), q_out, kp, vp, bt.to(DEV), ring, i32(pos),
                          i32(slots), table.to(DEV), n_heads, n_kv, hd, rd)
    scale = 1.0 / torch.sqrt((x.double() ** 2).mean(dim=1, keepdim=True) + 1e-5)
    qkv = (xn.double() @ w.double().T) * scale
    f = R.rope_inv_freq(hd, rd, 10000.0)
    p = torch.tensor(pos)
    q_want = R.rope_interleaved(qkv[:, :Q].reshape(M, n_heads, hd), p, f).reshape(M, Q)
    k_want = R.rope_interleaved(qkv[:, Q:Q + KV].reshape(M, n_kv, hd), p, f)
    v_want = qkv[:, Q + KV:].reshape(M, n_kv, hd)
    close(q_out, q_want, torch.bfloat16, "q", factor=1.5)
    kp, vp = pages_as_rows(kp.cpu(), vp.cpu())
    touched = torch.zeros((n_pages, PAGE), dtype=torch.bool)
    for m in range(M):
        if slots[m] < 0:
            continue
        page, r = int(bt[slots[m], (pos[m] // PAGE) % ring]), pos[m] % PAGE
        close(kp[page, :, r, :], k_want[m], torch.bfloat16, "k row %d" % m, factor=1.5)
        close(vp[page, :, :, r], v_want[m], torch.bfloat16, "v row %d" % m, factor=1.5)
        touched[page, r] = True
    assert (kp.float().abs().sum(dim=(1, 3)) > 0).equal(touched)
    assert (vp.float().abs().sum(dim=(1, 2)) > 0).equal(touched)


@pytest.mark.parametrize("M", [1, 7, 9, 16, 33])
@pytest.mark.parametrize("parts", [1, 63, 65, 256, 257, 600])
def test_gemm_chain_scales_of_any_number_of_parts(M, parts):
    """A chained consumer adds a row's partial sums of squares four times 64 at a time: every remainder, one and two rows a
    wave, K with fewer stages than waves.  Float32 sums of exact products: 2 sqrt(K) roundings of half a unit, and three of the scale."""
    k = K()
    for Kd, N in ((64, 70), (1024, 4112)):
        x = rnd((M, Kd), 70, torch.bfloat16)
        w = rnd((N, Kd), 71, torch.bfloat16, scale=1 / math.sqrt(Kd))
        ss = rnd((M, parts), 72).abs() * Kd / parts + 0.01
        out = torch.full((M + 1, N), 7.0, device=DEV)
        k.gemm_chain(x.to(DEV), w.to(DEV), out[:M], k.EPI_STORE_F32, scale_from=(ss.to(DEV).contiguous(), 1e-5))
        want = x.double() @ w.double().T / torch.sqrt(ss.double().sum(1, keepdim=True) / Kd + 1e-5)
        size = x.double().abs() @ w.double().abs().T / torch.sqrt(ss.double().sum(1, keepdim=True) / Kd + 1e-5)
        off = ((out[:M].double().cpu() - want).abs() / size).max().item()
        assert off <= (2 * math.sqrt(Kd) + 3) * 2.0 ** -24, "M %d, %d parts, K %d: %g" % (M, parts, Kd, off)
        assert bool((out[M] == 7.0).all())


@pytest.mark.parametrize("M,N,Kd", [(1, 64, 256), (8, 4096, 1000), (33, 80, 96), (64, 4096, 264), (5, 16400, 64),
                                    (11, 192, 192), (16, 4096, 128), (9, 1024, 64), (8, 3072, 128), (3, 3000, 64),
                                    (20, 3072, 64)])
def test_gemm_chain_producer_and_consumer(M, N, Kd):
    """A residual-add GEMM that emits the next norm's activations and partial sums of squares,
    and a consumer that scales by them: together they equal rmsnorm(x_new) @ W2^T."""
    k = K()
    a = rnd((M, Kd), 60, torch.bfloat16)
    w = rnd((N, Kd), 61, torch.bfloat16, scale=1 / math.sqrt(Kd))
    res = rnd((M, N), 62, scale=2.0)
    nw = 1 + 0.1 * rnd((N,), 63)
    x = res.to(DEV).clone()
    if N >= 16384:                                      # too wide to emit: refused
        with pytest.raises(Exception):
            k.gemm_chain(a.to(DEV), w.to(DEV), x, k.EPI_ADD_F32,
                         emit=(nw.to(DEV), torch.empty((M, N), dtype=torch.bfloat16, device=DEV),
                               torch.empty((M, k.gemm_chain_parts(N)), device=DEV)))
        return
    xn = torch.zeros((M, N), dtype=torch.bfloat16, device=DEV)
    ss = torch.zeros((M, k.gemm_chain_parts(N)), device=DEV)
    k.gemm_chain(a.to(DEV), w.to(DEV), x, k.EPI_ADD_F32, emit=(nw.to(DEV), xn, ss))
    x_want = res.double() + a.double() @ w.double().T
    close(x, x_want, torch.float32, "residual")
    close(xn, x_want * nw.double(), torch.bfloat16, "emitted activations")
    assert torch.allclose(ss.sum(dim=1).cpu().double(), (x_want ** 2).sum(dim=1), rtol=1e-5)
    # consumers: float32 store and gated
    H = 48
    from yalm_amd.parts.swiglu import interleave_gate_up
    w2 = rnd((70, N), 64, torch.bfloat16, scale=1 / math.sqrt(N))
    out = torch.empty((M, 70), device=DEV)
    k.gemm_chain(xn, w2.to(DEV), out, k.EPI_STORE_F32, scale_from=(ss, 1e-5))
    want = R.rmsnorm(x_want, nw, 1e-5) @ w2.double().T
    close(out, want, torch.bfloat16, "chained consumer", factor=1.5)
    wg = rnd((H, N), 65, torch.bfloat16, scale=1 / math.sqrt(N))
    wu = rnd((H, N), 66, torch.bfloat16, scale=1 / math.sqrt(N))
    outg = torch.empty((M, H), dtype=torch.bfloat16, device=DEV)
    h = R.rmsnorm(x_want, nw, 1e-5)
    for act in ACTS:
        act_fn, epi_code = gate(act)
        k.gemm_chain(xn, interleave_gate_up(wg, wu).to(DEV), outg, epi_code, hidden=H, scale_from=(ss, 1e-5))
        close(outg, act_fn(h @ wg.double().T) * (h @ wu.double().T), torch.bfloat16, "chained gated " + act, factor=2.0)


@pytest.mark.parametrize("with_workspace", [True, False])
@pytest.mark.parametrize("M,N,Kd", [(17, 4096, 4096), (64, 100, 264), (48, 6144, 1000), (33, 4096, 14336)])
def test_gemm_batches_of_17_to_64_rows(M, N, Kd, with_workspace):
    """The kernel for 17..64 rows, with K split across workgroups (given scratch) and without."""
    k = K()
    a = rnd((M, Kd), 70, torch.bfloat16)
    w = rnd((N, Kd), 71, torch.bfloat16, scale=1 / math.sqrt(Kd))
    want = a.double() @ w.double().T
    ws = torch.empty(k.gemm_workspace_floats(M, N, Kd), device=DEV) if with_workspace else None
    out = torch.empty((M, N), device=DEV)
    k.gemm(a.to(DEV), w.to(DEV), out, k.EPI_STORE_F32, workspace=ws)
    close(out, want, torch.float32, "f32 out")
    out2 = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    k.gemm(a.to(DEV), w.to(DEV), out2, k.EPI_STORE, workspace=ws)
    close(out2, want, torch.bfloat16, "bf16 out")
    res = rnd((M, N), 72)
    acc = res.to(DEV).clone()
    k.gemm(a.to(DEV), w.to(DEV), acc, k.EPI_ADD_F32, workspace=ws)
    close(acc, want + res.double(), torch.float32, "add")


@pytest.mark.parametrize("with_workspace", [True, False])
@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("M,H,D", [(64, 14336, 256), (20, 1000, 264), (40, 176, 4096)])
def test_gemm_gated_batches_of_17_to_64_rows(M, H, D, with_workspace, act):
    from yalm_amd.parts.swiglu import interleave_gate_up
    k = K()
    x = rnd((M, D), 73, torch.bfloat16)
    wg = rnd((H, D), 74, torch.bfloat16, scale=1 / math.sqrt(D))
    wu = rnd((H, D), 75, torch.bfloat16, scale=1 / math.sqrt(D))
    act_fn, epi_code = gate(act)
    want = act_fn(x.double() @ wg.double().T) * (x.double() @ wu.double().T)
    w = interleave_gate_up(wg, wu).to(DEV)
    ws = torch.empty(k.gemm_workspace_floats(M, w.shape[0], D), device=DEV) if with_workspace else None
    out = torch.empty((M, H), dtype=torch.bfloat16, device=DEV)
    k.gemm(x.to(DEV), w, out, epi_code, hidden=H, workspace=ws)
    close(out, want, torch.bfloat16, "gated")


@pytest.mark.parametrize("M,N,Kd", [(65, 4096, 4096), (128, 1000, 14336), (130, 333, 1024), (256, 4096, 2112),
                                    (70, 100, 4160)])
def test_gemm_of_more_than_64_rows_splits_k(M, N, Kd):
    """A batch of more than 64 rows whose output has few tiles: K in slices, given the scratch (whole, and
    too small for all the slices the kernel would like), and the same products without it."""
    k = K()
    a = rnd((M, Kd), 76, torch.bfloat16)
    w = rnd((N, Kd), 77, torch.bfloat16, scale=1 / math.sqrt(Kd))
    want = a.double() @ w.double().T
    res = rnd((M, N), 78)
    full = k.gemm_workspace_floats(M, N, Kd)
    assert full >= 2 * M * N and full % (M * N) == 0
    for floats in (full, 2 * M * N, 0):
        ws = torch.full((floats,), float("nan"), device=DEV) if floats else None
        out = torch.empty((M, N), device=DEV)
        k.gemm(a.to(DEV), w.to(DEV), out, k.EPI_STORE_F32, workspace=ws)
        close(out, want, torch.float32, "f32 out, %d floats" % floats)
        out2 = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
        k.gemm(a.to(DEV), w.to(DEV), out2, k.EPI_STORE, workspace=ws)
        close(out2, want, torch.bfloat16, "bf16 out, %d floats" % floats)
        acc = res.to(DEV).clone()
        k.gemm(a.to(DEV), w.to(DEV), acc, k.EPI_ADD_F32, workspace=ws)
        close(acc, want + res.double(), torch.float32, "add, %d floats" % floats)
    assert k.gemm_workspace_floats(8192, 4096, 4096) == 0       # enough tiles: no slices


@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("M,H,D", [(100, 1000, 4096), (128, 176, 2048), (65, 3000, 1024)])
def test_gemm_gated_of_more_than_64_rows_splits_k(M, H, D, act):
    from yalm_amd.parts.swiglu import interleave_gate_up
    k = K()
    x = rnd((M, D), 79, torch.bfloat16)
    wg = rnd((H, D), 84, torch.bfloat16, scale=1 / math.sqrt(D))
    wu = rnd((H, D), 85, torch.bfloat16, scale=1 / math.sqrt(D))
    act_fn, epi_code = gate(act)
    want = act_fn(x.double() @ wg.double().T) * (x.double() @ wu.double().T)
    w = interleave_gate_up(wg, wu).to(DEV)
    floats = k.gemm_workspace_floats(M, w.shape[0], D)
    assert floats >= 2 * M * w.shape[0]
    out = torch.empty((M, H), dtype=torch.bfloat16, device=DEV)
    k.gemm(x.to(DEV), w, out, epi_code, hidden=H, workspace=torch.full((floats,), float("nan"), device=DEV))
    close(out, want, torch.bfloat16, "gated")


@pytest.mark.parametrize("small_workspace", [False, True])
@pytest.mark.parametrize("M,N,Kd", [(17, 4096, 4096), (64, 100, 264), (40, 4096, 14336), (33, 96, 64),
                                    (65, 4096, 4096), (130, 333, 1024), (300, 20488, 128), (256, 96, 14336)])
def test_gemm_add_norm(M, N, Kd, small_workspace):
    """Residual add and the next RMSNorm in one, more than 16 rows: x += a W^T; h = rmsnorm(x) * w."""
    k = K()
    a = rnd((M, Kd), 80, torch.bfloat16)
    w = rnd((N, Kd), 81, torch.bfloat16, scale=1 / math.sqrt(Kd))
    x0 = rnd((M, N), 82, scale=2.0)
    nw = (1 + 0.1 * rnd((N,), 83)).float()
    eps = 1e-5
    x = x0.clone().to(DEV)
    h = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    ws = torch.empty(M * N if small_workspace else k.fused_workspace_floats(M, N, Kd), device=DEV)
    k.gemm_add_norm(a.to(DEV), w.to(DEV), x, nw.to(DEV), eps, h, ws)
    want_x = x0.double() + a.double() @ w.double().T
    close(x, want_x, torch.float32, "residual", factor=4)
    close(h, R.rmsnorm(want_x, nw, eps), torch.bfloat16, "normed")
    with pytest.raises(ValueError):
        k.gemm_add_norm(a.to(DEV), w.to(DEV), x, nw.to(DEV), eps, h, torch.empty(M * N - 1, device=DEV))


@pytest.mark.parametrize("small_workspace", [False, True])
@pytest.mark.parametrize("M,N,Kd,N2", [(17, 4096, 4096, 6144), (64, 104, 264, 48), (40, 4096, 14336, 320),
                                       (33, 96, 64, 200), (65, 4096, 4096, 1000), (128, 1088, 1024, 96)])
def test_gemm_add_emit_and_its_consumers(M, N, Kd, N2, small_workspace):
    """The norm chain of 17..128 rows: x += a W^T with the next norm only prepared (activations times the norm's
    weights, partial sums of squares), and the consumers that scale their sums row by row: a plain product, a gated
    one, and K slices left for another kernel to add.  Together they must give what a finished norm in front of the
    same products gives."""
    k = K()
    a = rnd((M, Kd), 90, torch.bfloat16)
    w = rnd((N, Kd), 91, torch.bfloat16, scale=1 / math.sqrt(Kd))
    x0 = rnd((M, N), 92, scale=2.0)
    x0[M // 2] *= 37.0                                   # rows of very different sizes: every row has its own scale
    x0[0] *= 1e-3
    nw = (1 + 0.1 * rnd((N,), 93)).float()
    eps = 1e-5
    x = x0.clone().to(DEV)
    xn = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    parts = k.gemm_add_emit_parts(N)
    assert parts == (N + 1023) // 1024
    ss = torch.full((M, parts), float("nan"), device=DEV)
    ws = torch.empty(M * N if small_workspace else k.fused_workspace_floats(M, N, Kd), device=DEV)
    assert k.can_add_emit(M, Kd, torch.bfloat16) and not k.can_add_emit(16, Kd, torch.bfloat16)
    k.gemm_add_emit(a.to(DEV), w.to(DEV), x, nw.to(DEV), xn, ss, ws)
    want_x = x0.double() + a.double() @ w.double().T
    close(x, want_x, torch.float32, "residual", factor=4)
    close(xn, want_x * nw.double(), torch.bfloat16, "activations times the norm's weights")
    close(ss.sum(dim=1), (want_x ** 2).sum(dim=1), torch.float32, "sums of squares", factor=4)
    h = R.rmsnorm(want_x, nw, eps)                       # what the consumers' products must be products of
    # a plain consumer (the head's epilogue) and the K slices of one
    w2 = rnd((N2, N), 94, torch.bfloat16, scale=1 / math.sqrt(N))
    want = h @ w2.double().T
    out = torch.empty((M, N2), device=DEV)
    ws2 = torch.full((k.gemm_workspace_floats(M, N2, N),), float("nan"), device=DEV)
    k.gemm(xn, w2.to(DEV), out, k.EPI_STORE_F32, workspace=ws2, scale_from=(ss, eps))
    close(out, want, torch.bfloat16, "scaled product")
    if k.can_gemm_partial(M, N, torch.bfloat16):
        ws3 = torch.full((k.fused_workspace_floats(M, N2, N),), float("nan"), device=DEV)
        slices = k.gemm_partial(xn, w2.to(DEV), ws3, scale_from=(ss, eps))
        close(ws3[:slices * M * N2].view(slices, M, N2).sum(dim=0), want, torch.bfloat16, "scaled slices")
    # a gated consumer
    H = 72
    wg = rnd((H, N), 95, torch.bfloat16, scale=1 / math.sqrt(N))
    wu = rnd((H, N), 96, torch.bfloat16, scale=1 / math.sqrt(N))
    from yalm_amd.parts.swiglu import interleave_gate_up
    wgu = interleave_gate_up(wg, wu).to(DEV)
    mid = torch.empty((M, H), dtype=torch.bfloat16, device=DEV)
    ws4 = torch.full((k.gemm_workspace_floats(M, wgu.shape[0], N),), float("nan"), device=DEV)
    for act in ACTS:
        act_fn, epi_code = gate(act)
        k.gemm(xn, wgu, mid, epi_code, hidden=H, workspace=ws4, scale_from=(ss, eps))
        close(mid, act_fn(h @ wg.double().T) * (h @ wu.double().T), torch.bfloat16, "scaled gated product " + act, factor=2)
    with pytest.raises(Exception):                        # a row scale is for these batches only
        k.gemm(xn[:8].contiguous(), w2.to(DEV), out[:8].contiguous(), k.EPI_STORE_F32, scale_from=(ss[:8].contiguous(), eps))


# ------------------------------------------------------------------ recurrences by tiles

@pytest.mark.parametrize("kind", ["hgrn2", "gla", "lightning"])
@pytest.mark.parametrize("d,dv", [(32, 32), (20, 96), (64, 64), (128, 128), (100, 32), (32, 48), (64, 33), (128, 48), (64, 16)])
def test_recurrences_by_tiles_of_many_workgroups(kind, d, dv):
    """From a workgroup and a half a compute unit on, whole groups of 32 columns share a workgroup of the walk over tiles: read-outs and
    states have the bits that each sequence has alone (which goes 16 columns a workgroup)."""
    k = K()
    H, rank, lens = 16, 5, [1, 64, 65, 130, 17, 200] * 4
    units = torch.cuda.get_device_properties(0).multi_processor_count
    assert 2 * H * ((dv + 31) // 32) * len(lens) >= 3 * units > 2 * H * ((dv + 31) // 32)
    T, Hd, Hv = sum(lens), H * d, H * dv
    width = {"hgrn2": 2 * Hd + Hv, "gla": 2 * Hd + 2 * Hv + rank, "lightning": 2 * Hd + Hv}[kind]
    proj, start = rnd((T, width), 1).to(DEV), rnd((len(lens), Hv * d), 2, scale=0.3).to(DEV)
    bias, lower, w = rnd((Hd,), 3).to(DEV), rnd((Hd,), 4).abs().clamp(0, 0.9).to(DEV), (1 + 0.1 * rnd((dv,), 5)).to(DEV)
    w2 = torch.zeros(Hd, k.gla_padded_rank(rank))
    w2[:, :rank] = rnd((Hd, rank), 6)
    w2 = w2.to(DEV)
    powers = (torch.linspace(0.9, 1.0, H, dtype=torch.float64)[:, None] ** torch.arange(65)).float().contiguous().to(DEV)
    scratch = lambda name, shape, dt: torch.full(shape, float("nan"), dtype=dt, device=DEV)

    def run(rows, lens, state):
        n = sum(lens)
        out, raw = (torch.full((n, Hv), float("nan"), device=DEV) for _ in range(2))
        ends = lambda sizes: [0] + torch.tensor(sizes).cumsum(0).tolist()
        tile0 = ends([(x + 63) // 64 for x in lens])
        places = (i32(ends(lens)), i32(list(range(len(lens)))), i32(tile0), tile0[-1])
        if kind == "hgrn2":
            k.hgrn2_tiles(rows, bias, lower, w, state, raw, *places, out, H, d, dv, 1e-5, scratch)
        elif kind == "gla":
            k.gla_tiles(rows, w2, bias, w, state, raw, *places, out, H, d, dv, rank, d ** -0.5, 16.0, 1e-5, scratch)
        else:
            k.lightning_tiles(rows, powers, state, raw, *places, H, d, dv, scratch)
        return raw
    state = start.clone()
    raw, at = run(proj, lens, state), 0
    assert bool(torch.isfinite(raw).all())
    for b, n in enumerate(lens):
        if b % 5 == 0 or n == 200:
            alone = start[b:b + 1].clone()
            assert torch.equal(run(proj[at:at + n].contiguous(), [n], alone), raw[at:at + n]) and torch.equal(alone[0], state[b]), b
        at += n
