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
