"""Split K on 64 x 64 tiles, the launcher's own choice for grids that leave the device mostly empty: the K parts' 32-bit
sums through the library's workspace, added by a second launch in the order of the parts.  Bit-exact against the CPU
oracle on integer-valued data, where every summation order gives the same bits."""
import itertools
import threading

import numpy as np
import pytest
import torch

import oracle_lib as O

pytestmark = pytest.mark.gpu

TYPES = (O.S8S8S32, O.BF16BF16F32, O.BF16BF16BF16, O.F16F16F16, O.F32F32F32, O.E4M3E4M3F16, O.E5M2E5M2F16)
LAYOUTS = tuple(itertools.product((O.ROW, O.COL), (O.ROW, O.COL)))


def exact_kind(types):
    return O.FILL_INT8_UNIFORM if types == O.S8S8S32 else O.FILL_SMALL_INT


def k_of(types, slabs, extra):
    """`slabs` whole 128-byte slabs and `extra` elements of K."""
    return slabs * (128 // np.dtype(O.IN_DTYPE[types]).itemsize) + extra


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


@pytest.mark.parametrize("types", TYPES)
@pytest.mark.parametrize("layouts", LAYOUTS)
def test_every_layout_bit_exact(G, types, layouts):
    """Rows and columns on both sides of a tile's and a block's edge, K in whole slabs, in slabs and one element, in
    slabs and all but one, parts of unequal length; C and alpha / beta in the second launch; unaligned operands."""
    la, lb = layouts
    bk = 128 // np.dtype(O.IN_DTYPE[types]).itemsize
    split = 0
    for (m, n, slabs, extra), (al, be) in itertools.product(
            [(200, 64, 60, 0), (129, 100, 61, 1), (160, 33, 67, bk - 1), (193, 257, 80, 5), (140, 31, 50, 1)], [(1, 0), (2, -1)]):
        k = k_of(types, slabs, extra)
        p = G.capi.plan(types, m, n, k, la, lb)
        split += p.split_k > 1
        a, b, c = O.make_inputs(types, m, n, k, kind=exact_kind(types), seed=m + extra)
        print("case", types, la, lb, m, n, k, al, be, p.split_k, flush=True)
        ref = O.gemm(types, a, b, c, m, n, k, la, lb, al, be)
        assert np.array_equal(G.run_gemm(types, a, b, c, m, n, k, la, lb, al, be, -1), ref), (m, n, k, al, be)
        assert np.array_equal(G.run_gemm(types, a, b, c, m, n, k, la, lb, al, be, -1, misalign=1), ref), (m, n, k, al, be)
    assert split >= 6, "these shapes are meant to be split"
    # views whose padding is NaN (or large), rows of D that are not whole 16-byte pieces
    m, n, k = 150, 70, k_of(types, 64, 3)
    a, b, c = O.make_inputs(types, m, n, k, kind=exact_kind(types), seed=4)
    got = G.run_gemm_ld(types, a, b, c, m, n, k, la, lb, 1, 1, -1, 0, (5, 3, 1, 2))
    assert np.array_equal(got, O.gemm(types, a, b, c, m, n, k, la, lb, 1, 1))


def test_normal_data_repeatable(G):
    m, n, k = 150, 200, 2560
    a, b, c = O.make_inputs(O.BF16BF16F32, m, n, k, kind=O.FILL_NORMAL, seed=1)
    assert G.capi.plan(O.BF16BF16F32, m, n, k, O.ROW, O.COL).split_k > 1
    got = [G.run_gemm(O.BF16BF16F32, a, b, c, m, n, k, O.ROW, O.COL, 1, 0.5, -1) for _ in range(3)]
    truth, _ = O.gemm_f64(O.BF16BF16F32, a, b, c, m, n, k, O.ROW, O.COL, 1, 0.5)
    G.assert_within(O.BF16BF16F32, got[0], truth, "split K")
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


def _problem(G, seed, m=192, n=128, k=5120):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randint(-128, 128, (m * k,), generator=gen, device="cuda", dtype=torch.int8)
    b = torch.randint(-128, 128, (k * n,), generator=gen, device="cuda", dtype=torch.int8)
    ref = (a.view(m, k).double() @ b.view(n, k).t().double()).int()
    return a, b, ref, (m, n, k)


def test_threads_that_share_a_stream(G):
    """One workspace serves a stream: the two launches of a call must not be torn apart by another thread's."""
    problems = [_problem(G, s) for s in range(4)]
    assert G.capi.plan(O.S8S8S32, *problems[0][3], O.ROW, O.COL).split_k > 1
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    outs = [[torch.empty(192, 128, dtype=torch.int32, device="cuda") for _ in range(25)] for _ in problems]
    errors = []

    def work(i):
        try:
            a, b, _, (m, n, k) = problems[i]
            for d in outs[i]:
                G.capi.gemm(O.S8S8S32, a, b, None, d, m, n, k, O.ROW, O.COL, 1, 0, -1, 0, stream.cuda_stream)
        except Exception as e:   # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(problems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for (_, _, ref, _), ds in zip(problems, outs):
        for d in ds:
            assert torch.equal(d, ref)


def test_under_capture(G):
    """A captured call takes a plan without the workspace: every replay gives the right result, whatever eager calls on
    the same stream have done to the workspace in between."""
    a, b, ref, (m, n, k) = _problem(G, 7)
    d = torch.empty(m, n, dtype=torch.int32, device="cuda")
    other = _problem(G, 8, 192, 1024, 16384)
    e = torch.empty(192, 1024, dtype=torch.int32, device="cuda")
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        G.capi.gemm(O.S8S8S32, a, b, None, d, m, n, k, O.ROW, O.COL, 1, 0, -1, 0, stream.cuda_stream)
    for _ in range(3):
        d.fill_(-1)
        e.fill_(-1)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(d, ref)
        mo, no, ko = other[3]
        G.capi.gemm(O.S8S8S32, other[0], other[1], None, e, mo, no, ko, O.ROW, O.COL, 1, 0, -1, 0, stream.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(e, other[2])


def test_threads_on_the_per_thread_stream(G):
    """hipStreamPerThread is one handle and another stream in every thread: calls that run side by side on it share no
    partial sums."""
    problems = [_problem(G, 20 + s) for s in range(4)]
    outs = [[torch.empty(192, 128, dtype=torch.int32, device="cuda") for _ in range(25)] for _ in problems]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            a, b, _, (m, n, k) = problems[i]
            for d in outs[i]:
                G.capi.gemm(O.S8S8S32, a, b, None, d, m, n, k, O.ROW, O.COL, 1, 0, -1, 0, 2)
        except Exception as e:   # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(problems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for (_, _, ref, _), ds in zip(problems, outs):
        for d in ds:
            assert torch.equal(d, ref)


def test_the_pool_gives_idle_buffers_back(G):
    """More streams than the pool holds buffers for (68 MiB each, 1 GiB in all): those that have gone longest without a
    call lose theirs, get new ones when they call again, and every result is right."""
    a, b, ref, (m, n, k) = _bf16_problem(1024, 1024, 16384)
    assert 17 * G.capi.plan(O.BF16BF16F32, m, n, k, O.ROW, O.COL).workspace_bytes > 1 << 30
    streams = [torch.cuda.Stream() for _ in range(20)]
    torch.cuda.synchronize()
    free = []
    for part in (streams[:10], streams[10:], streams[:10]):
        outs = [torch.full((m, n), -1.0, device="cuda") for _ in part]
        torch.cuda.synchronize()
        for d, s in zip(outs, part):
            G.capi.gemm(O.BF16BF16F32, a, b, None, d, m, n, k, O.ROW, O.COL, 1, 0, -1, 0, s.cuda_stream)
        torch.cuda.synchronize()
        assert all(torch.equal(d, ref) for d in outs)
        del outs
        free.append(torch.cuda.mem_get_info()[0])
    assert free[2] >= free[1] - (128 << 20), "the third part took the place of the second's buffers"


def _bf16_problem(m, n, k):
    """Small whole numbers: every sum is exact."""
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    a, b = (torch.randint(-1, 2, (rows, k), generator=gen, device="cuda").bfloat16() for rows in (m, n))
    return a.reshape(-1), b.reshape(-1), a.float() @ b.float().t().contiguous(), (m, n, k)


# what cuts K outside a capture: split K on 64 x 64 tiles, stream-K by the launcher's choice and by name, the wide column
# blocks of the streaming rung by choice and by name
CAPTURED = {"split": (O.S8S8S32, (192, 128, 5120), -1, 0), "stream-K": (O.BF16BF16F32, (1024, 1024, 8192), -1, 0),
            "stream-K, named": (O.BF16BF16F32, (1024, 1024, 8192), 4, 7), "wide": (O.BF16BF16F32, (128, 14336, 8192), -1, 0),
            "wide, named": (O.BF16BF16F32, (128, 14336, 8192), 5, 0)}


@pytest.mark.parametrize("what", CAPTURED)
@pytest.mark.parametrize("entry", ("gemm", "gemm_static_scratch"))
def test_every_plan_that_cuts_k_under_capture(G, what, entry):
    """A captured call takes a plan without the pool (the entry point with the static buffer keeps its plan): every replay
    gives the right result, whatever eager calls on the same stream, with more memory than the captured problem would
    take, have done to the pool in between."""
    types, shape, rung, variant = CAPTURED[what]
    a, b, ref, (m, n, k) = _problem(G, 7, *shape) if types == O.S8S8S32 else _bf16_problem(*shape)
    p = G.capi.plan(types, m, n, k, O.ROW, O.COL, rung, variant)
    assert p.workspace_bytes > 0
    d = torch.empty(m, n, dtype=ref.dtype, device="cuda")
    other = _problem(G, 8, 1024, 1536, 16384)
    mo, no, ko = other[3]
    po = G.capi.plan(O.S8S8S32, mo, no, ko, O.ROW, O.COL, 4, 7)
    assert po.workspace_bytes > p.workspace_bytes
    e = torch.empty(mo, no, dtype=torch.int32, device="cuda")
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        getattr(G.capi, entry)(types, a, b, None, d, m, n, k, O.ROW, O.COL, 1, 0, rung, variant, stream.cuda_stream)
    for _ in range(4):
        d.fill_(-1)
        e.fill_(-1)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(d, ref)
        G.capi.gemm(O.S8S8S32, other[0], other[1], None, e, mo, no, ko, O.ROW, O.COL, 1, 0, 4, 7, stream.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(e, other[2])
