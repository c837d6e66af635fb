"""Tile GEMM of the prefill projections (mc_model_gemm_tiles) and the norm that
consumes its split sums, against float64 products.

Bounds: a K-term fp32 sum in any order is within K 2^-24 sum |x w| of the exact
one (each addition rounds by at most 2^-24 of a partial sum of at most
sum |x w|); a bf16 result adds half an ulp, 2^-9 of it. The SwiGLU output moves
by at most 1.1 |u| per unit of the gate (|silu'| < 1.1) and |silu(g)| per unit
of the up value, both rounded to bf16 first.
"""
import ctypes as C

import numpy as np
import pytest

from _util import from_dev, to_dev

pytestmark = pytest.mark.gpu

AUTO = 0xFFFFFFFF
# tile table rows: (BM, weight rows of a tile, takes plain, takes swiglu)
SHAPES = [(32, 64, 1, 0), (48, 64, 1, 0), (64, 64, 1, 0), (64, 64, 0, 1), (64, 96, 0, 1),
          (96, 64, 1, 1), (128, 64, 1, 1), (128, 96, 1, 1), (128, 128, 1, 1), (128, 192, 0, 1),
          (192, 128, 1, 1), (256, 128, 1, 1), (160, 256, 1, 1), (192, 192, 1, 1),
          (256, 160, 1, 0), (256, 192, 1, 1), (192, 256, 1, 1), (256, 256, 1, 1)]


def P(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def stream():
    import torch
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.fixture(scope="module")
def lib(pkg):
    return pkg._native.lib()


def run(lib, orc, dev, M, N, K, swi, splits, shape, part, seed):
    """Error of one call over its bound (<= 1 passes) and whether the guard
    rows around the output are untouched."""
    import torch
    rng = np.random.default_rng(seed)
    rows = 2 * N if swi else N
    w = orc.f32_to_bf16(rng.standard_normal((rows, K), dtype=np.float32) / np.float32(K ** 0.5))
    x = orc.f32_to_bf16(rng.standard_normal((M, K), dtype=np.float32))
    outs = splits if part else 1
    dt = torch.float32 if part else torch.int16
    y = torch.full(((outs * M + 2) * N,), -1, dtype=dt, device=dev)
    mid = y[N:-N]
    dw, dx = to_dev(w, dev), to_dev(x, dev)
    r = lib.mc_model_gemm_tiles(P(dw), P(dx), None if part else P(mid),
                                P(mid) if part else None, M, N, K, swi, splits, shape, stream())
    assert r == 0, r
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    guard = np.all(y[:N] == -1) and np.all(y[-N:] == -1)
    got = y[N:-N] if part else orc.bf16_to_f32(y[N:-N].view(np.uint16))
    got = got.astype(np.float64).reshape(outs, M, N)
    xf, wf = (orc.bf16_to_f32(a).astype(np.float64) for a in (x, w))
    step = K // outs
    ref = np.stack([xf[:, s * step:(s + 1) * step] @ wf[:, s * step:(s + 1) * step].T
                    for s in range(outs)])
    acc = step * 2.0 ** -24 * np.stack(
        [np.abs(xf[:, s * step:(s + 1) * step]) @ np.abs(wf[:, s * step:(s + 1) * step]).T
         for s in range(outs)])
    bound = acc + (0.0 if part else 2.0 ** -8 * np.abs(ref))
    if swi:
        g, u = ref[0, :, :N], ref[0, :, N:]
        eg, eu = bound[0, :, :N], bound[0, :, N:]
        s = g / (1.0 + np.exp(-g))
        ref = (s * u)[None]
        bound = (1.1 * eg * (np.abs(u) + eu) + np.abs(s) * eu + 2.0 ** -8 * np.abs(s * u))[None]
    return float(np.max(np.abs(got - ref) / (bound + 1e-30))), bool(guard)


@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_every_tile_shape_at_its_edges(lib, orc, dev, shape):
    """Each tile shape at one row, one row either side of a whole tile and two
    tiles and a remainder, over whole and part n tiles, with the fewest K steps and with
    more steps than LDS stages; plain, split sums and SwiGLU as it takes them."""
    bm, bn, plain, swi = SHAPES[shape]
    N = bn // 64 * 64 + 64  # the last n tile is part empty
    for M in (1, bm - 1, bm, bm + 1, 2 * bm + 17):
        if plain:
            for K, splits, part in ((128, 1, 0), (896, 1, 0), (768, 3, 1), (1024, 8, 1),
                                    (384, 1, 1)):
                err, guard = run(lib, orc, dev, M, N, K, 0, splits, shape, part, M + K)
                assert err <= 1.0 and guard, (shape, M, K, splits, err, guard)
        if swi:
            for K in (128, 640):
                err, guard = run(lib, orc, dev, M, N, K, 1, 1, shape, 0, M + K)
                assert err <= 1.0 and guard, (shape, M, K, err, guard)


@pytest.mark.parametrize("M,N,K,swi,splits,part", [
    (33, 2560, 2048, 0, 1, 0), (201, 2048, 2048, 0, 2, 1), (48, 2048, 6144, 0, 8, 1),
    (300, 2560, 2048, 0, 1, 0), (100, 6144, 2048, 1, 1, 0), (511, 2048, 6144, 0, 4, 1),
    (1025, 6144, 2048, 1, 1, 0), (2065, 2048, 256, 0, 1, 1),
    (8455, 2048, 256, 0, 1, 0), (20011, 2048, 128, 0, 1, 0), (65535, 64, 128, 0, 1, 0)])
def test_planned_shape(lib, orc, dev, M, N, K, swi, splits, part):
    """The shape the plan takes for the model's projections, more than one
    round of workgroups, ragged row counts and the largest chunk."""
    err, guard = run(lib, orc, dev, M, N, K, swi, splits, AUTO, part, M)
    assert err <= 1.0 and guard, (err, guard)


def second_launch_rows(lib, M, N, K, form):
    """Rows that the plan of least estimated time leaves to its second launch."""
    p = (C.c_uint32 * 4)()
    assert lib.mc_model_debug_gemm_tiles_plan(M, N, K, form, 1, 1, p) == 0
    return M - p[0]


@pytest.mark.parametrize("M,N,K,swi,part", [(8455, 2048, 2048, 0, 0), (8455, 2048, 2048, 0, 1),
                                            (1300, 6144, 2048, 1, 0), (8448, 1536, 256, 1, 0)])
def test_two_launches(lib, orc, dev, M, N, K, swi, part):
    """Sizes that the plan cuts into whole rounds of a large tile and the rows
    left over: the second launch's rows and outputs follow the first's."""
    assert second_launch_rows(lib, M, N, K, swi) > 0
    err, guard = run(lib, orc, dev, M, N, K, swi, 1, AUTO, part, M)
    assert err <= 1.0 and guard, (err, guard)


@pytest.mark.parametrize("splits", range(1, 9))
def test_norm_of_split_sums(lib, orc, dev, splits):
    """mc_model_rmsnorm_splits equals mc_model_rmsnorm_rows on the sums added
    in split order in fp32 and rounded to bf16, bit for bit."""
    import torch
    rng = np.random.default_rng(splits)
    rows = 5
    part = rng.standard_normal((splits, rows, 2048), dtype=np.float32)
    tot = part[0].copy()
    for s in range(1, splits):
        tot += part[s]
    res = orc.f32_to_bf16(rng.standard_normal((rows, 2048), dtype=np.float32) * 3)
    g = orc.f32_to_bf16(1 + 0.1 * rng.standard_normal(2048, dtype=np.float32))
    eps = C.c_float(1e-6)
    out = []
    dg = to_dev(g, dev)
    for form in (0, 1):
        r, o = to_dev(res, dev), torch.zeros(rows * 2048, dtype=torch.int16, device=dev)
        if form:
            d = torch.from_numpy(part).to(dev)
            assert lib.mc_model_rmsnorm_splits(P(r), P(d), splits, P(dg), P(o), rows, eps,
                                               stream()) == 0
        else:
            d = to_dev(orc.f32_to_bf16(tot), dev)
            assert lib.mc_model_rmsnorm_rows(P(r), P(d), P(dg), P(o), rows, 2048, eps,
                                             stream()) == 0
        torch.cuda.synchronize()
        out.append((from_dev(r), from_dev(o)))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("shape", [0, 1, 2, 5, 6, 7, 8, 10, 11, 12, 13, 15, 16, 17,
                                   AUTO])
def test_rope_form(lib, pkg, orc, dev, shape):
    """mc_model_gemm_tiles_rope equals the plain tiles followed by
    mc_kv_rope_append bit for bit (q columns and every page slot), for whole
    and part tiles, page sizes below and above a tile's rows and, planned, several
    rounds of workgroups."""
    check_rope_form(lib, pkg, orc, dev, shape, 256)


@pytest.mark.parametrize("M,K", [(6500, 2048), (7936, 2048), (13100, 256)])
def test_rope_form_in_two_launches(lib, pkg, orc, dev, M, K):
    """Sizes whose qkv projection the plan cuts in two: the second launch's rows
    are rotated and appended at their own positions."""
    assert second_launch_rows(lib, M, 2560, K, 2) > 0
    check_rope_form(lib, pkg, orc, dev, AUTO, K, ((M, 41, 32),))


def check_rope_form(lib, pkg, orc, dev, shape, K, sizes=None):
    import torch
    N, layer = 2560, 1
    bm = SHAPES[shape][0] if shape != AUTO else 0
    rng = np.random.default_rng(7)
    w = to_dev(orc.f32_to_bf16(rng.standard_normal((N, K), dtype=np.float32) /
                               np.float32(K ** 0.5)), dev)
    if sizes is None:
        sizes = (((1, 0, 32), (bm + 1, 3001, 16), (2 * bm + 17, 77, 64)) if bm else
                 ((33, 5, 1), (300, 900, 32), (8455, 40, 32)))
    for M, base, page in sizes:
        npage = (base + M + page - 1) // page + 2
        pt = to_dev(rng.permutation(npage).astype(np.uint32), dev)
        x = to_dev(orc.f32_to_bf16(rng.standard_normal((M, K), dtype=np.float32)), dev)
        pos = to_dev(np.array([base], np.uint32), dev)
        lay = pkg._native.LayoutT(npage, page, 2, 0)
        out = []
        for fused in (0, 1):
            y = torch.zeros((M + 1, N), dtype=torch.int16, device=dev)
            pool = torch.full((2 * npage * page, 512), 99, dtype=torch.int16, device=dev)
            if fused:
                assert lib.mc_kv_rope_table(P(y), M, P(pos), 5e6, None, stream()) == 0
                assert lib.mc_model_gemm_tiles_rope(P(w), P(x), P(y), M, K, P(pos), layer, P(pt),
                                                    P(pool), lay, shape, stream()) == 0
            else:
                assert lib.mc_model_gemm_tiles(P(w), P(x), P(y), None, M, N, K, 0, 1, shape,
                                               stream()) == 0
                assert lib.mc_kv_rope_append(P(y), M, P(pos), layer, P(pt), P(pool), lay, 5e6,
                                             None, stream()) == 0
            torch.cuda.synchronize()
            out.append((y[:, :2048].clone(), y[M].clone(), pool))
        assert torch.equal(out[0][0], out[1][0]), (shape, M)
        assert torch.equal(out[0][2], out[1][2]), (shape, M)
        assert not out[1][1].any(), (shape, M)


def test_rejects_bad_arguments(lib, pkg, dev):
    """Sizes and combinations outside the contract are MC_E_INVALID_ARGUMENT,
    with nothing launched."""
    import torch
    buf = torch.zeros(1 << 20, dtype=torch.int16, device=dev)
    p, odd = P(buf), C.c_void_p(buf.data_ptr() + 2)
    f = lib.mc_model_gemm_tiles
    for a in ((p, p, p, None, 0, 64, 128, 0, 1, AUTO), (p, p, p, None, 8, 96, 128, 0, 1, AUTO),
              (p, p, p, None, 8, 64, 192, 0, 1, AUTO), (p, p, p, p, 8, 64, 128, 0, 1, AUTO),
              (p, p, None, None, 8, 64, 128, 0, 1, AUTO), (p, p, p, None, 8, 64, 128, 2, 1, AUTO),
              (p, p, p, None, 8, 64, 256, 0, 2, AUTO), (p, p, None, p, 8, 64, 128, 1, 1, AUTO),
              (p, p, None, p, 8, 64, 256, 0, 3, AUTO), (p, p, None, p, 8, 64, 2304, 0, 9, AUTO),
              (odd, p, p, None, 8, 64, 128, 0, 1, AUTO), (p, odd, p, None, 8, 64, 128, 0, 1, AUTO),
              (p, p, p, None, 8, 64, 128, 0, 1, 18), (p, p, p, None, 8, 64, 128, 0, 1, 3),
              (p, p, p, None, 8, 64, 128, 1, 1, 0), (p, p, p, None, 8, 64, 128, 1, 1, 14)):
        assert f(*a, stream()) == 1, a[4:]
    assert lib.mc_model_rmsnorm_splits(p, p, 9, p, p, 1, C.c_float(1e-6), stream()) == 1
    assert lib.mc_model_rmsnorm_splits(p, p, 0, p, p, 1, C.c_float(1e-6), stream()) == 1
    lay = pkg._native.LayoutT(4, 32, 2, 0)
    g = lib.mc_model_gemm_tiles_rope
    for a in ((p, p, p, 0, 128, p, 0, p, p, lay, AUTO), (p, p, p, 8, 192, p, 0, p, p, lay, AUTO),
              (p, p, p, 8, 128, p, 2, p, p, lay, AUTO), (p, p, p, 8, 128, p, 0, None, p, lay, AUTO),
              (p, p, odd, 8, 128, p, 0, p, p, lay, AUTO), (p, p, p, 8, 128, p, 0, p, p, lay, 14)):
        assert g(*a, stream()) == 1, a[3:]
    assert lib.mc_kv_rope_table(p, 0, p, 5e6, None, stream()) == 1
