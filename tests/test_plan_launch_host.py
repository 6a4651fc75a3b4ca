"""gz_plan says what a call launches: grid, threads and LDS of the first launch, how many launches, on a stand-in for the HIP
runtime (hip_stub.c), without a GPU."""
import random

import pytest

from test_workspace_host import run  # noqa: F401 - the fixture

MFMA = 4
S8, BF16F32, BF16, F16, F32, E4M3, E5M2 = range(7)


def problems(seed, count):
    """Seeded problems of every type bundle and layout: extents of a few tiles to a few thousand, whole and ragged, the
    launcher's choice and every variant of the MFMA rung."""
    rng = random.Random(seed)
    out = []
    while len(out) < count:
        q = rng.choice([1, 1, 8, 16, 64, 128, 256])
        m, n, k = (max(1, int(2 ** rng.uniform(4, 12.5)) // q * q) for _ in range(3))
        if rng.random() < 0.25:
            m = rng.randint(1, 128)
        variant = rng.choice([0, 0, 0] + list(range(1, 14)))
        out.append((rng.randrange(7), m, n, k, rng.randrange(2), rng.randrange(2), MFMA if variant else -1, variant))
    return out


# LDS that depends on the grid, the type and the lines: nine buffers of a lone 128 x 128 tile, two slabs of a lone 64 x 64 one,
# padded rows of unaligned 32 x 32 ones
NAMED = [(BF16F32, 3072, 3072, 4096, 0, 1, MFMA, 11), (BF16F32, 1024, 1024, 1024, 0, 1, MFMA, 11), (F32, 1024, 1024, 1024, 0, 0, MFMA, 11),
         (F16, 2048, 2048, 1024, 0, 0, MFMA, 11), (S8, 2048, 2048, 3072, 0, 1, MFMA, 11), (E4M3, 1024, 1024, 1024, 0, 0, MFMA, 11),
         (BF16, 1024, 1024, 2048, 0, 0, MFMA, 12), (BF16, 2048, 2048, 2048, 0, 0, MFMA, 12), (S8, 130, 70, 96, 0, 1, MFMA, 13),
         (S8, 130, 70, 97, 0, 1, MFMA, 13), (F32, 130, 71, 97, 1, 0, MFMA, 13), (S8, 200, 64, 4096, 0, 0, -1, 0), (BF16F32, 4352, 4096, 4096, 0, 1, -1, 0),
         (F16, 4095, 4097, 1023, 0, 0, -1, 0), (BF16F32, 4096, 4104, 512, 1, 1, -1, 0), (S8, 20, 1280, 11008, 0, 1, -1, 0)]


@pytest.mark.parametrize("batch", [NAMED, problems(1, 250), problems(2, 250)], ids=["named", "seed 1", "seed 2"])
def test_plan_and_launch_agree(run, capi, batch):  # noqa: F811
    calls = [dict(types=t, m=m, n=n, k=k, la=la, lb=lb, rung=rung, variant=v, stream=0x1000) for t, m, n, k, la, lb, rung, v in batch]
    wrong = []
    for problem, step in zip(batch, run(*(["gemm", c] for c in calls))):
        p = capi.plan(*problem)
        assert step["result"][0] == 0, (problem, step)
        launches, groups = ([e for e in step["events"] if e[0] == kind] for kind in ("launch", "group"))
        first = (launches[0][2], groups[0][1], groups[0][2])
        second = bool(p.tail_rows or p.tail_cols) + bool(p.split_k > 1 or p.streamk_tiles)
        lds = first[2] if p.rung == capi.RUNG_SKINNY and p.variant == 1 else p.lds_bytes   # (that rung has static LDS as well)
        if first != (p.grid, p.threads, lds) or len(launches) != 1 + second:
            wrong.append((problem, first, len(launches), p.as_dict()))
        if p.tail_grid and launches[1][2] != p.tail_grid:
            wrong.append((problem, "tail", launches[1][2], p.tail_grid))
    assert not wrong, wrong[:3]


def test_lds_of_the_kernel_that_runs(capi):
    plan = capi.plan
    assert plan(BF16F32, 3072, 3072, 4096, 0, 1, MFMA, 11).lds_bytes == 5 * 256 * 64      # more tiles than compute units
    assert plan(BF16F32, 1024, 1024, 1024, 0, 1, MFMA, 11).lds_bytes == 9 * 256 * 64
    assert plan(F32, 1024, 1024, 1024, 0, 0, MFMA, 11).lds_bytes == 5 * 256 * 64
    assert plan(S8, 256, 256, 1024, 0, 1, MFMA, 13).lds_bytes == 8 * 64 * 128
    assert plan(S8, 256, 256, 1023, 0, 1, MFMA, 13).lds_bytes == 8 * 64 * 144


def test_a_device_with_less_lds_keeps_its_plans(capi):
    """Problems that smaller kernels run are planned on them, not refused."""
    def plan(lds, *a):
        return capi.plan(*a, *([] if len(a) > 6 else [-1, 0]), 256, lds)
    assert plan(64 * 1024, BF16F32, 512, 512, 512, 0, 1).lds_bytes <= 64 * 1024
    assert plan(128 * 1024, BF16F32, 1024, 1024, 1024, 0, 1, MFMA, 11).lds_bytes == 5 * 256 * 64
    p = plan(48 * 1024, BF16F32, 1024, 1024, 4096, 0, 0, MFMA, 12)
    assert (p.lds_bytes, p.threads, p.tile_m) == (2 * 128 * 144, 256, 64)
    assert plan(100 * 1024, BF16F32, 512, 512, 4096, 0, 0, MFMA, 12).lds_bytes == 64 * 1024
    rng = random.Random(3)
    for _ in range(300):
        t, m, n, k = rng.randrange(7), rng.randint(1, 3000), rng.randint(1, 3000), rng.randint(1, 9000)
        p = plan(48 * 1024, t, m, n, k, rng.randrange(2), rng.randrange(2))
        assert p.rung != MFMA or p.lds_bytes <= 48 * 1024, (t, m, n, k)
    with pytest.raises(capi.GzError):
        plan(48 * 1024, BF16F32, 512, 512, 512, 0, 1, MFMA, 13)
    with pytest.raises(capi.GzError):
        plan(48 * 1024, BF16F32, 4096, 4096, 4096, 0, 1, MFMA, 5)
