"""Every tile shape of the GEMM launchers gives a row the same bits: launches
at the edges of each shape's range of rows (one row, a ragged last block, the
last count of a shape and the first of the next) against the first rows of one
larger launch on the same data, alone and beside another launch. The larger
launches are the ones the per-kernel tests compare with the oracle."""
import numpy as np
import pytest

import oracle

from test_kernels_gpu import (K_PATCH, K_PATCH_S, K_QKV, K_QKV_LN, K_RESID, K_RESID_S, K_SWIGLU, K_SWIGLU_LN, _keys, allocf, eng,  # noqa: F401
                              f16, read_heads, readf, slot_stats, up, upf)

pytestmark = pytest.mark.gpu


def run(e, kernel, scalars, bindings, beside=None):
    """One launch, or with `beside` as one of two branches of a plan."""
    key = next(_keys)
    if beside is None:
        e.record(key, [(kernel, scalars, bindings)])
    else:
        e.record_branches(key, [[(kernel, scalars, bindings)], [(kernel, scalars, beside)]])
    e.replay(key)
    e.synchronize()


@pytest.mark.parametrize("kdim", [384, 1536])
def test_resid_rows_do_not_depend_on_the_tile(eng, kdim):  # noqa: F811
    rng = np.random.default_rng(kdim)
    most = 11000
    a, x0 = f16(rng.normal(size=(most, kdim))), f16(rng.normal(size=(most, 384)) * 2 + 0.5)
    w = upf(eng, f16(rng.normal(size=(384, kdim)) * 0.03))
    b = up(eng, (rng.normal(size=384) * 0.1).astype(np.float32))
    ls = up(eng, rng.uniform(0.5, 1.5, size=384).astype(np.float32))

    def launch(rows, beside=False):
        ar = upf(eng, a[:rows])
        x, st = upf(eng, x0[:rows]), eng.allocate(rows * 48)
        other = [ar, w, b, ls, upf(eng, x0[:rows]), eng.allocate(rows * 48)] if beside else None
        run(eng, K_RESID_S, [rows, kdim], [ar, w, b, ls, x, st], other)
        plain = upf(eng, x0[:rows])
        run(eng, K_RESID, [rows, kdim], [ar, w, b, ls, plain])
        y = readf(eng, x, rows, 384)
        assert np.array_equal(readf(eng, plain, rows, 384), y)
        return y, eng.read(st, np.float32, (rows, 12))

    want, want_stats = launch(most)
    for rows in (1, 32, 33, 65, 1344, 1345, 2688, 2689, 5119, 5120, 5376, 5377, 10880, 10881):
        for beside in (False, True):
            got, stats = launch(rows, beside)
            assert np.array_equal(got, want[:rows]), (rows, beside)
            assert np.array_equal(stats, want_stats[:rows]), (rows, beside)


@pytest.mark.parametrize("grid,most,counts", [(4, 300, (1, 2, 42, 43, 85, 86, 170, 171)), (14, 26, (1, 4, 5, 8, 9, 14, 15, 17, 18)),
                                              (59, 2, (1,))])
def test_qkv_rows_do_not_depend_on_the_tile(eng, grid, most, counts):  # noqa: F811
    rng = np.random.default_rng(grid)
    T = grid * grid + 5
    tpad = (T + 127) // 128 * 128
    x = f16(rng.normal(size=(most * T, 384)) * 1.5 + 0.5)
    w = upf(eng, f16(rng.normal(size=(1152, 384)) * 0.05))
    wsum, b = (up(eng, (rng.normal(size=1152) * 0.1).astype(np.float32)) for _ in range(2))
    cos, sin = (up(eng, t) for t in oracle.rope_tables(grid))

    def launch(images, beside=False):
        xr, st, nb = upf(eng, x[:images * T]), up(eng, slot_stats(x[:images * T])), images * 6 * tpad * 64 * 2
        got = []
        for kernel, first in ((K_QKV, [xr, w, b]), (K_QKV_LN, [xr, st, w, wsum, b])):
            out, other = ([eng.allocate(nb) for _ in range(3)] for _ in range(2))
            run(eng, kernel, [images, grid, tpad], first + [cos, sin] + out, first + [cos, sin] + other if beside else None)
            got += [read_heads(eng, r, images, tpad) for r in out]
        return got

    want = launch(most)
    for images in counts:
        for beside in (False, True):
            for name, g, r in zip(("q", "k", "v", "q LN", "k LN", "v LN"), launch(images, beside), want):
                assert np.array_equal(g, r[:images]), (images, beside, name)


def test_swiglu_rows_do_not_depend_on_the_tile(eng):  # noqa: F811
    rng = np.random.default_rng(8)
    most = 8400
    x = f16(rng.normal(size=(most, 384)) * 1.5 + 0.5)
    w = upf(eng, f16(rng.normal(size=(3072, 384)) * 0.05))
    wsum, b = (up(eng, (rng.normal(size=3072) * 0.1).astype(np.float32)) for _ in range(2))

    def launch(rows):
        xr, st, got = upf(eng, x[:rows]), up(eng, slot_stats(x[:rows])), []
        for kernel, binds in ((K_SWIGLU, [xr, w, b]), (K_SWIGLU_LN, [xr, st, w, wsum, b])):
            act = allocf(eng, rows, 1536)
            run(eng, kernel, [rows], binds + [act])
            got.append(readf(eng, act, rows, 1536))
        return got

    want = launch(most)
    for rows in (1, 33, 640, 641, 1280, 1281, 2048, 2049, 5119, 5120):
        for name, g, r in zip(("plain", "LN"), launch(rows), want):
            assert np.array_equal(g, r[:rows]), (rows, name)


@pytest.mark.parametrize("grid,most,counts", [(1, 1400, (1, 31, 33, 1344, 1345)), (3, 160, (1, 4, 149, 150)),
                                              (14, 8, (1, 3, 6, 7)), (37, 2, (1,))])
def test_patch_rows_do_not_depend_on_the_tile(eng, grid, most, counts):  # noqa: F811
    rng = np.random.default_rng(grid)
    T, S = grid * grid + 5, 16 * grid
    px = rng.normal(size=(most, 3, S, S)).astype(np.float32)
    w = up(eng, f16(rng.normal(size=(384, 768)) * 0.02))
    b, prefix = up(eng, rng.normal(size=384).astype(np.float32)), up(eng, rng.normal(size=(5, 384)).astype(np.float32))
    pstats = up(eng, rng.normal(size=(5, 12)).astype(np.float32))

    def launch(images):
        p, x, xs, st = up(eng, px[:images]), *(allocf(eng, images * T, 384) for _ in range(2)), eng.allocate(images * T * 48)
        run(eng, K_PATCH, [images, grid], [p, w, b, prefix, x])
        run(eng, K_PATCH_S, [images, grid], [p, w, b, prefix, pstats, xs, st])
        y = readf(eng, x, images * T, 384)
        assert np.array_equal(readf(eng, xs, images * T, 384), y)
        return y, eng.read(st, np.float32, (images * T, 12))

    want, want_stats = launch(most)
    for images in counts:
        got, stats = launch(images)
        assert np.array_equal(got, want[:images * T]), images
        assert np.array_equal(stats, want_stats[:images * T]), images


@pytest.mark.parametrize("images", [1, 26])
def test_qkv_rotation_rounds_the_second_halfs_product(eng, images):  # noqa: F811
    # Identity weights and no bias, so the sums are the inputs and the outputs
    # show the rotation's own rounding: of lo cos - up sin and up cos + lo sin
    # the products with up are rounded to float32, those with lo are fused, and the
    # sum is rounded once, to float16.
    grid, T, tpad = 14, 201, 256
    rng = np.random.default_rng(images)
    x = f16(rng.normal(size=(images * T, 384)))
    w = upf(eng, f16(np.tile(np.eye(384), (3, 1))))
    cos, sin = oracle.rope_tables(grid)
    nb = images * 6 * tpad * 64 * 2
    out = [eng.allocate(nb) for _ in range(3)]
    run(eng, K_QKV, [images, grid, tpad], [upf(eng, x), w, up(eng, np.zeros(1152, np.float32)), up(eng, cos), up(eng, sin)] + out)
    h = x.reshape(images, T, 6, 64).transpose(0, 2, 1, 3).astype(np.float64)
    lo, hi = h[:, :, 5:, :32], h[:, :, 5:, 32:]
    c, s = (t[:, :32].astype(np.float64) for t in (cos, sin))
    want = h.copy()
    want[:, :, 5:, :32] = lo * c - (hi * s).astype(np.float32)
    want[:, :, 5:, 32:] = lo * s + (hi * c).astype(np.float32)
    for r, ref in zip(out, (want, want, h)):
        got, ref = read_heads(eng, r, images, tpad)[:, :, :T], ref.astype(np.float16)
        assert np.array_equal(got, ref), f"{int((got != ref).sum())} of {ref.size} differ"
