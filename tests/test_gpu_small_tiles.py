"""The small tiles (variants 12 and 13): 32 x 32 and, from a longer K on, 64 x 64 tiles whose waves share out K, and the
register-staged 64 x 64 ones.  Every number of slabs around a full set of stages, slabs that the end of K cuts, rows and columns
around the edges of a tile and of a 16-byte piece, aligned and unaligned lines (two ways into LDS).  Exact inputs, so a slab or
a piece lost, counted twice or not zeroed shows."""
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


@pytest.mark.parametrize("la,lb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("types", TYPES)
def test_slabs_edges_and_alignment(G, types, la, lb):
    es = np.dtype(O.IN_DTYPE[types]).itemsize
    slab, piece = 128 // es, 16 // es
    kind = O.FILL_INT8_UNIFORM if types == O.S8S8S32 else O.FILL_SMALL_INT
    # aligned lines: whole pieces everywhere
    ks = [piece, slab, slab + piece, 3 * slab, 5 * slab - piece, 8 * slab, 9 * slab, 17 * slab + piece]
    aligned = [(64, 128, k) for k in ks] + [(32 + piece, 16, 4 * slab), (96, 64 + piece, 7 * slab), (16, 208, 2 * slab + piece)]
    # any size: lines that are not whole pieces, and (K alone, lines along M and N) cut slabs of whole lines
    ragged = [(1, 1, 1), (63, 65, slab - 1), (65, 33, 2 * slab + 3), (31, 129, 5 * slab + 1), (17, 3, 9 * slab), (64, 64, 4 * slab + 1),
              (128, 96, 3 * slab + 5)]
    for variant, (m, n, k), (beta, misalign) in itertools.product((12, 13), aligned + ragged, ((1, 0), (0, 1))):
        a, b, c = O.make_inputs(types, m, n, k, kind=kind, seed=k + m)
        print("case", types, la, lb, variant, m, n, k, beta, misalign, flush=True)
        got = G.run_gemm(types, a, b, c, m, n, k, la, lb, 1, beta, MFMA, variant, misalign=misalign)
        assert np.array_equal(got, O.gemm(types, a, b, c, m, n, k, la, lb, 1, beta)), (types, la, lb, variant, m, n, k, beta, misalign)


@pytest.mark.parametrize("la,lb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("types", (O.S8S8S32, O.BF16BF16F32, O.F16F16F16, O.E5M2E5M2F16))
def test_64x64_tiles_with_slabs_of_the_waves_own(G, types, la, lb):
    """A K long enough for the kernel whose four waves have slabs of their own: every number of slabs around full sets of its
    stages, cut last slabs, rows and columns past the edges, rows of D that are no whole vectors; one work-group per compute
    unit (two slabs on their way to each wave) and more (one)."""
    es = np.dtype(O.IN_DTYPE[types]).itemsize
    slab, piece = 128 // es, 16 // es
    kind = O.FILL_INT8_UNIFORM if types == O.S8S8S32 else O.FILL_SMALL_INT
    cases = [(64, 128, (17 + i) * slab) for i in range(9)] + [(96, 64 + piece, 17 * slab + piece), (128, 80, 25 * slab - piece)]
    # (lines along M and N in whole pieces; otherwise any)
    cases += [(64 + (1 if la == 0 else piece), 64 + (5 if lb == 1 else piece), 20 * slab + piece), (1088, 1024, 25 * slab)]
    for (m, n, k), beta in itertools.product(cases, (0, 1)):
        p = G.capi.plan(types, m, n, k, la, lb, MFMA, 12)
        assert (p.wave_m, p.wave_n, p.threads) == (64, 64, 256), "slabs of the waves' own"
        if m > 1000 and beta:
            continue
        a, b, c = O.make_inputs(types, m, n, k, kind=kind, seed=k + m)
        print("case", types, la, lb, m, n, k, beta, p.lds_bytes, flush=True)
        got = G.run_gemm(types, a, b, c, m, n, k, la, lb, 1, beta, MFMA, 12)
        assert np.array_equal(got, O.gemm(types, a, b, c, m, n, k, la, lb, 1, beta)), (types, la, lb, m, n, k, beta)


@pytest.mark.parametrize("variant", (12, 13))
@pytest.mark.parametrize("la,lb", [(0, 1), (1, 0)])
def test_an_infinity_beside_the_end_of_k(G, variant, la, lb):
    """A slab that the end of K cuts holds repeated elements there until they are zeroed, on both operands."""
    types, m, n = O.BF16BF16F32, 64, 64
    for k in (2 * 64 + 8, 20 * 64 + 8):
        a, b, _ = O.make_inputs(types, m, n, k, kind=O.FILL_UNIFORM_PM1, seed=4)
        a.reshape(-1)[5 * k + k - 1 if la == 0 else (k - 1) * m + 5] = 0x7F80
        got = G.run_gemm(types, a, b, None, m, n, k, la, lb, 1, 0, MFMA, variant).astype(np.float64)
        assert np.isinf(got[5]).all() and np.isfinite(np.delete(got, 5, axis=0)).all()
