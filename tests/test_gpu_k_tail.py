"""The ring kernel on a K that is not whole 128-byte slabs: its first two slabs overlap and what both hold is zeroed in the
first.  Exact inputs, so any piece counted twice or lost shows."""
import itertools

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
MFMA = 4
TYPES = (O.S8S8S32, O.BF16BF16F32, O.F16F16F16, O.E4M3E4M3F16, O.F32F32F32)


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def exact_kind(types):
    return O.FILL_INT8_UNIFORM if types == O.S8S8S32 else O.FILL_SMALL_INT


@pytest.mark.parametrize("la,lb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("types", TYPES)
def test_every_tail_is_counted_once(G, types, la, lb):
    """Two to eight slabs (the ring holds five half slabs), the smallest and the largest tail of
    K-contiguous operands and, where both operands lie along M and N, single K rows; whole and ragged M and N."""
    es = np.dtype(O.IN_DTYPE[types]).itemsize
    slab, piece = 128 // es, 16 // es
    tails = [piece, slab - piece] if la == 0 or lb == 1 else [1, slab // 2 + 1, slab - 1]
    for whole, tail, (variant, m, n) in itertools.product((1, 2, 3, 4, 5, 7), tails, ((5, 256, 256), (6, 272, 528), (11, 128, 384), (11, 144, 272))):
        if n * m > 256 * 400 and whole > 3:
            continue
        k = whole * slab + tail
        a, b, c = O.make_inputs(types, m, n, k, kind=exact_kind(types), seed=k)
        print("case", types, la, lb, variant, m, n, k, flush=True)
        got = G.run_gemm(types, a, b, c, m, n, k, la, lb, 1, 1, MFMA, variant)
        assert np.array_equal(got, O.gemm(types, a, b, c, m, n, k, la, lb, 1, 1)), (types, la, lb, variant, m, n, k)


@pytest.mark.parametrize("la,lb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("types", (O.S8S8S32, O.BF16BF16F32, O.F16F16F16))
def test_nine_buffers_and_a_tail(G, types, la, lb):
    """128 x 128 tiles that have a compute unit to themselves, from eight whole slabs on: the ring of nine buffers, one turn of
    it and two, whole and ragged M and N."""
    es = np.dtype(O.IN_DTYPE[types]).itemsize
    slab, piece = 128 // es, 16 // es
    tails = [0, piece, slab - piece] + ([] if la == 0 or lb == 1 else [1, slab // 2 + 1])
    for whole, tail, (m, n) in itertools.product((8, 9, 10, 17, 18), tails, ((256, 128), (144, 272))):
        k = whole * slab + tail
        p = G.capi.plan(types, m, n, k, la, lb, MFMA, 11)
        assert p.lds_bytes == 9 * 256 * 64, "nine buffers"
        a, b, c = O.make_inputs(types, m, n, k, kind=exact_kind(types), seed=k)
        print("case", types, la, lb, m, n, k, flush=True)
        got = G.run_gemm(types, a, b, c, m, n, k, la, lb, 1, 1, MFMA, 11)
        assert np.array_equal(got, O.gemm(types, a, b, c, m, n, k, la, lb, 1, 1)), (types, la, lb, m, n, k)


@pytest.mark.parametrize("variant", (5, 6))
@pytest.mark.parametrize("types", TYPES)
def test_a_tail_where_work_groups_walk_several_tiles(G, types, variant):
    """288 tiles of 256 x 256: the first slab of the next tile is asked for before the current one is stored, and is cut when it
    has landed.  First rows, rows of second tiles and the last rows."""
    es = np.dtype(O.IN_DTYPE[types]).itemsize
    m, n = 4360, 4096
    for k, lb in ((128 // es + 16 // es, 1), (3 * (128 // es) - 16 // es, 0)):
        a, b, c = O.make_inputs(types, m, n, k, kind=exact_kind(types), seed=k)
        print("case", types, variant, m, n, k, lb, flush=True)
        got = G.run_gemm(types, a, b, c, m, n, k, 0, lb, 2, 1, MFMA, variant)
        for rows in ((0, 8), (2040, 2056), (4096 - 4, 4096 + 4), (m - 8, m)):
            ref = O.gemm(types, a, b, c, m, n, k, 0, lb, 2, 1, rows=rows)
            assert np.array_equal(got[rows[0]:rows[1]], ref[rows[0]:rows[1]]), (types, variant, k, lb, rows)
        one = G.run_gemm(types, a, b, c, m, n, k, 0, lb, 2, 1, MFMA, variant + 4)
        assert np.array_equal(got, one)


@pytest.mark.parametrize("la,lb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("types", TYPES)
def test_a_tail_of_two_slabs_on_the_launchers_choice(G, types, la, lb):
    """One slab and a piece, two slabs less a piece: the launcher's own tile, which the ring kernel's start would hold up, and
    the ring kernel itself."""
    es = np.dtype(O.IN_DTYPE[types]).itemsize
    slab, piece = 128 // es, 16 // es
    m, n = 2560 + 48, 3072 + 16
    for k in (slab + piece, 2 * slab - piece):
        a, b, c = O.make_inputs(types, m, n, k, kind=exact_kind(types), seed=k)
        print("case", types, m, n, k, la, lb, flush=True)
        got = G.run_gemm(types, a, b, c, m, n, k, la, lb, 1, 1, MFMA, 0)
        for rows in ((0, 8), (1276, 1284), (m - 8, m)):
            ref = O.gemm(types, a, b, c, m, n, k, la, lb, 1, 1, rows=rows)
            assert np.array_equal(got[rows[0]:rows[1]], ref[rows[0]:rows[1]]), (types, k, la, lb, rows)
        assert np.array_equal(got, G.run_gemm(types, a, b, c, m, n, k, la, lb, 1, 1, MFMA, 5))


@pytest.mark.parametrize("types,inf", [(O.BF16BF16F32, 0x7F80), (O.F32F32F32, np.inf)])
@pytest.mark.parametrize("la,lb", [(0, 1), (1, 0)])
def test_an_infinity_in_the_overlap_stays_one(G, types, inf, la, lb):
    """The elements that both of the first slabs hold become zeros on both operands: an infinity times the other's zero would
    be a NaN."""
    es = np.dtype(O.IN_DTYPE[types]).itemsize
    m, n, k = 256, 256, 3 * (128 // es) + 8
    a, b, _ = O.make_inputs(types, m, n, k, kind=O.FILL_UNIFORM_PM1, seed=4)
    at = 20   # slab 0 holds it, and slab 1, which begins at 8
    flat = a.reshape(-1)
    flat[(5 * k + at) if la == 0 else (at * m + 5)] = inf
    for variant in (5, 6, 11):
        got = G.run_gemm(types, a, b, None, m, n, k, la, lb, 1, 0, MFMA, variant).astype(np.float64)
        assert np.isinf(got[5]).all() and np.isfinite(np.delete(got, 5, axis=0)).all(), (variant, la, lb)
