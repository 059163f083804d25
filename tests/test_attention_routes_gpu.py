"""Every attention kernel a sequence can run on gives an image the same bits:
launches on both sides of each rule's edge (one round of workgroups for the
wave-per-block and the 64-query kernels, more than one for the unrolled walk)
against one larger launch of the same images, and the sequences around the
edge of the two-halves walk against the float64 oracle."""
import numpy as np
import pytest

import oracle

from test_kernels_gpu import K_ATTN, _keys, allocf, check, eng, f16, heads_frag, readf, run, up  # noqa: F401

pytestmark = pytest.mark.gpu


def launch(e, mats, images, grid, beside=False):
    T = grid * grid + 5
    tpad = (T + 127) // 128 * 128
    ins = [up(e, heads_frag(m[:images * T], images, T, tpad)) for m in mats]
    out = allocf(e, images * T, 384)
    if beside:  # one of two branches of a plan
        key, other = next(_keys), allocf(e, images * T, 384)
        e.record_branches(key, [[(K_ATTN, [images, grid, tpad], ins + [o])] for o in (out, other)])
        e.replay(key)
        e.synchronize()
        assert np.array_equal(readf(e, other, images * T, 384), readf(e, out, images * T, 384), equal_nan=True)
    else:
        run(e, K_ATTN, [images, grid, tpad], ins + [out])
    return readf(e, out, images * T, 384)


def inputs(grid, images, scale=2.0):
    rng = np.random.default_rng(grid)
    rows = images * (grid * grid + 5)
    return [f16(rng.normal(size=(rows, 384)) * s) for s in (scale, 1.0, 1.0)]


# (grid, images of the large launch, images of the others): 1 to 14 key blocks
# (a wave per block up to 256 workgroups of 32 queries), 16 and 19 blocks
# (64-query workgroups up to 256 of them, 192 beside another launch), 1029
# tokens (64 queries to 2 images, 128 from 3, the unrolled walk from 5 and
# beside another launch), 2030 tokens.
ROUTES = [(4, 50, (1, 42, 43)), (7, 24, (1, 21, 22)), (8, 20, (1, 14, 15)), (10, 14, (1, 10, 11)), (12, 12, (1, 8, 9)),
          (13, 10, (1, 7, 8)), (14, 10, (1, 6, 7)), (15, 8, (1, 5, 6)), (16, 8, (1, 4, 5)), (17, 6, (1, 4, 5)),
          (18, 5, (1, 3, 4)), (19, 5, (1, 3, 4)), (20, 5, (1, 3, 4)), (21, 6, (1, 3, 4)), (22, 8, (1, 4, 5, 6)), (24, 8, (1, 4, 5)), (32, 6, (1, 2, 3, 4, 5)),
          (45, 3, (1, 2))]


# ramp: the scores grow along the keys, so the running max has to move.
@pytest.mark.parametrize("ramp", [False, True])
@pytest.mark.parametrize("grid,most,counts", ROUTES)
def test_images_do_not_depend_on_the_launch(eng, grid, most, counts, ramp):  # noqa: F811
    q, k, v = inputs(grid, most)
    T = grid * grid + 5
    if ramp:
        k = f16(k * np.tile(np.linspace(0.1, 8.0, T), most)[:, None])
    mats = [q, k, v]
    want = launch(eng, mats, most, grid)
    assert np.all(np.isfinite(want))
    for images in counts:
        for beside in (False, True):
            got = launch(eng, mats, images, grid, beside)
            assert np.array_equal(got, want[:images * T]), (images, beside)


@pytest.mark.parametrize("grid", [1, 5, 7, 21, 22, 25])
@pytest.mark.parametrize("scale", [0.0, 4.0])
def test_edges_match_the_oracle(eng, grid, scale):  # noqa: F811
    # P is rounded to f16 (2^-11 relative) before a product whose weights sum
    # to one, and the output to f16: 2^-9 max|V| bounds both, as in the
    # per-kernel attention test.
    q, k, v = inputs(grid, 2, scale)
    T = grid * grid + 5
    got = launch(eng, [q, k, v], 2, grid)
    for i in range(2):
        rows = slice(i * T, (i + 1) * T)
        want = oracle.attention(*(m[rows].astype(np.float64) for m in (q, k, v)))
        check(got[rows], want, atol=2.0**-9 * np.abs(v[rows].astype(np.float64)).max(), what=f"T={T} image {i}")


# Scores of -inf over the whole first key block (keys 0..31) and one later one:
# the softmax runs over the other keys, whichever kernel takes the launch.
@pytest.mark.parametrize("grid,images,most", [(8, 1, 20), (14, 6, 10), (16, 4, 8), (21, 3, 6), (22, 5, 8), (32, 2, 6)])
def test_first_block_of_minus_infinities(eng, grid, images, most):  # noqa: F811
    q, k, v = inputs(grid, most)
    T = grid * grid + 5
    q[:, ::64] = np.abs(q[:, ::64]) + np.float16(0.5)
    k.reshape(most, T, 384)[:, :32, ::64] = -np.inf
    k.reshape(most, T, 384)[:, 40, ::64] = -np.inf
    want = launch(eng, [q, k, v], most, grid)
    got = launch(eng, [q, k, v], images, grid)
    assert np.array_equal(got, want[:images * T])
    assert np.array_equal(launch(eng, [q, k, v], images, grid, beside=True), got)
    r = slice(0, T)
    ref = oracle.attention(*(m[r].astype(np.float64) for m in (q, k, v)))
    check(got[r], ref, atol=2.0**-9 * np.abs(v[r].astype(np.float64)).max(), what=f"T={T}")


# A score of +inf or NaN, or a NaN value, makes its query's (its key's) outputs
# NaN, the same ones on every kernel.
@pytest.mark.parametrize("key", [3, 37])
@pytest.mark.parametrize("what", ["k=+inf", "k=nan", "v=nan"])
@pytest.mark.parametrize("grid,images,most", [(8, 1, 20), (14, 6, 10), (16, 4, 8), (22, 5, 8), (32, 2, 6)])
def test_infinities_and_nan_do_not_depend_on_the_launch(eng, grid, images, most, what, key):  # noqa: F811
    q, k, v = inputs(grid, most)
    T = grid * grid + 5
    (k if what[0] == "k" else v).reshape(most, T, 384)[:, key, :2] = np.inf if "inf" in what else np.nan
    want = launch(eng, [q, k, v], most, grid)
    got = launch(eng, [q, k, v], images, grid)
    assert np.isnan(got).any() and not np.isnan(got).all()
    assert np.array_equal(got, want[:images * T], equal_nan=True)
    assert np.array_equal(launch(eng, [q, k, v], images, grid, beside=True), got, equal_nan=True)
