"""The library's workspace pool on a stand-in for the HIP runtime (hip_stub.c), without a GPU: which calls take memory, from
whom it is kept, and what a call does that cannot have any.  Nothing runs; what is checked is what the runtime is asked
for, call by call."""
import json
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
S8, BF16F32, BF16 = 0, 1, 2
MFMA, SKINNY = 4, 5
STREAM = 0x1000
# problems whose plans cut K: split K on 64 x 64 tiles, stream-K, the wide column blocks of the streaming rung
SPLITK = dict(types=S8, m=192, n=128, k=5120)
STREAMK = dict(types=BF16F32, m=1024, n=1024, k=16384)
WIDE = dict(types=BF16, m=128, n=14336, k=8192)
CUT_K = ("splitk_reduce", "streamk_fixup", "stream_wide_reduce")


@pytest.fixture(scope="module")
def run(tmp_path_factory, capi):
    stub = tmp_path_factory.mktemp("stub") / "libhipstub.so"
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", str(HERE / "hip_stub.c"), "-o", str(stub), "-ldl", "-lpthread"], check=True)

    def steps(*what):
        p = subprocess.run([sys.executable, str(HERE / "hip_stub_run.py"), str(stub), str(capi.LIB_PATH), json.dumps(what)],
                           capture_output=True, text=True, timeout=120)
        assert p.returncode == 0, p.stderr
        return json.loads(p.stdout)
    return steps


def events(step, kind):
    return [e for e in step["events"] if e[0] == kind]


def cuts_k(step):
    return [e for e in events(step, "launch") if any(name in e[3] for name in CUT_K)]


@pytest.mark.parametrize("problem", (SPLITK, STREAMK, WIDE, dict(STREAMK, rung=MFMA, variant=7), dict(STREAMK, rung=MFMA, variant=8),
                                     dict(WIDE, rung=SKINNY)))
@pytest.mark.parametrize("warm", (False, True))
def test_a_captured_call_takes_no_pool_memory(run, problem, warm):
    """A graph keeps the addresses of what it captured, and the pool's buffers are replaced when a call needs more: a call
    on a stream that is being captured runs a plan without a workspace, whether or not the stream has a buffer by then."""
    call = dict(problem, stream=STREAM)
    plain, cap, captured, off, after = run(*((["gemm", call],) if warm else (["stub_capture", 0],)), ["stub_capture", STREAM],
                                           ["gemm", call], ["stub_capture", 0], ["gemm", call])
    assert captured["result"][0] == 0, captured
    assert not events(captured, "malloc") and not events(captured, "refused") and not events(captured, "free"), captured
    assert events(captured, "launch") and not cuts_k(captured), captured
    assert after["result"][0] == 0 and cuts_k(after), "outside the capture the same call cuts K"


def test_static_scratch_cuts_k_under_capture(run):
    """The entry point that allocates nothing has its buffer in the device image: captured calls keep their plan."""
    for problem in (SPLITK, STREAMK, WIDE):
        _, step = run(["stub_capture", STREAM], ["gemm", dict(problem, stream=STREAM, entry="gz_gemm_static_scratch")])
        assert step["result"][0] == 0 and cuts_k(step) and not events(step, "malloc"), step


PER_THREAD = 2   # hipStreamPerThread: one handle, another stream in every thread


@pytest.mark.parametrize("problem", (SPLITK, STREAMK, WIDE, dict(STREAMK, rung=MFMA, variant=7), dict(WIDE, rung=SKINNY)))
def test_the_per_thread_stream_takes_no_pool_memory(run, problem):
    """The pool keeps one buffer per stream handle; the per-thread stream's handle is the same in threads whose streams
    run side by side, so calls on it run plans without a workspace."""
    call = dict(problem, stream=PER_THREAD)
    for step in run(["gemm", call], ["other_thread", call]):
        assert step["result"][0] == 0 and events(step, "launch"), step
        assert not events(step, "malloc") and not cuts_k(step), step


def test_a_pinned_variant_launches_its_kernel(run):
    """What the plan says of a pinned variant is what is launched (the streaming rung's kernels take no variants)."""
    shapes = [dict(types=S8, m=64, n=4096, k=4096), dict(types=BF16, m=8, n=4096, k=1000), dict(types=5, m=1, n=4096, k=4096)]
    for variant in (1, 3, 5, 12):
        for problem, step in zip(shapes, run(*(["gemm", dict(s, variant=variant)] for s in shapes))):
            assert step["result"][0] == 0, (problem, variant, step)
            assert all("mfma" in e[3] for e in events(step, "launch")), (problem, variant, step)


LARGER = dict(types=BF16F32, m=408, n=2560, k=8164, lb=0)   # a split K with 17.5 MiB of partial sums


def test_without_memory_a_split_k_runs_unsplit(run):
    """A problem that needs no workspace but is faster with one must not fail for want of it."""
    _, small, large = run(["stub_memory", 1], ["gemm", dict(SPLITK, stream=STREAM)], ["gemm", dict(LARGER, stream=STREAM)])
    assert cuts_k(small) and large["result"][0] == 0
    assert events(large, "nomemory") and events(large, "launch") and not cuts_k(large)


def test_an_earlier_failure_is_reported(run):
    """Growing the pool waits for the stream, which may report what went wrong in work that was queued before: that is no
    lack of memory, and the caller has to hear of it."""
    _, _, step, _, again = run(["gemm", dict(SPLITK, stream=STREAM)], ["stub_sync_status", 719], ["gemm", dict(LARGER, stream=STREAM)],
                               ["stub_sync_status", 0], ["gemm", dict(LARGER, stream=STREAM)])
    assert step["result"][0] == 3 and "hipStreamSynchronize" in step["result"][1] and not events(step, "launch"), step
    assert again["result"][0] == 0 and cuts_k(again)


def live(steps):
    """Bytes held after each step."""
    sizes, out = {}, []
    for step in steps:
        for e in step["events"]:
            if e[0] == "malloc":
                sizes[e[2]] = e[1]
            elif e[0] == "free":
                assert sizes.pop(e[1], None) is not None, "freed twice"
        out.append(sum(sizes.values()))
    return out


def test_a_small_problem_takes_little(run):
    step, = run(["gemm", dict(SPLITK, stream=STREAM)])
    assert live([step])[0] <= 4 << 20, "1.9 MiB of partial sums"


def test_streams_that_come_and_go_do_not_pile_up(run, capi):
    """A handle is all the pool knows of a stream; the buffers that have gone longest without a call are given back."""
    need = capi.plan(BF16F32, 1024, 1024, 16384, 0, 1).workspace_bytes
    steps = run(*(["gemm", dict(STREAMK, stream=0x1000 + 16 * i)] for i in range(60)), ["gemm", dict(STREAMK, stream=0x1000 + 16 * 59)],
                ["gemm", dict(STREAMK, stream=0x1000)])
    held = live(steps)
    assert max(held) <= 1 << 30 and held[3] >= 4 * need and all(s["result"][0] == 0 and cuts_k(s) for s in steps)
    assert not steps[60]["events"][0][0] == "malloc", "the last stream's buffer is still there"
    assert events(steps[61], "malloc"), "the first stream's is not, and the stream gets another"


def test_a_full_device_is_not_asked_on_every_call(run):
    call = ["gemm", dict(SPLITK, stream=STREAM)]
    _, *calls = run(["stub_memory", 0], *([call] * 300))
    assert all(s["result"][0] == 0 and events(s, "launch") and not cuts_k(s) for s in calls)
    assert 1 <= sum(bool(events(s, "nomemory")) for s in calls) <= 3
    _, _, _, *later = run(["stub_memory", 0], call, ["stub_memory", 9], *([call] * 300))
    assert cuts_k(later[-1]), "memory that comes back is found"
    assert run(["stub_memory", 0], call, ["stub_memory", 9], ["gemm", dict(STREAMK, stream=STREAM)])[3]["result"][0] == 0


def test_idle_buffers_make_room(run):
    """What another stream's idle buffer holds is given back before a call is told that there is no memory."""
    first, _, second = run(["gemm", dict(SPLITK, stream=STREAM)], ["stub_room", 1], ["gemm", dict(SPLITK, stream=STREAM + 16)])
    assert events(second, "nomemory") and events(second, "free") and cuts_k(second), second
