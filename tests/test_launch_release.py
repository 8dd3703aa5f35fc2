"""What a loop of launches without a wait leaves on the host heap.  The runtime keeps the host object of
a launch that carries an event (1.4 KB) until it has processed a record on that stream, or a wait that
found the stream busy.  An executor records its event behind every 64th launch, so that a loop keeps a
bounded number: the heap grows by 2.8 MB at most, however long the loop (by 4.5 MB with the event
recorded behind every launch).  Kept for all of the loop's launches it would grow by 27 MB here."""
import ctypes
import gc
import time

import pytest

from grouped_gemm_gpu_kernel_amd import api
from grouped_gemm_gpu_kernel_amd.api import GroupedGemmExecutor, KernelConfig, ProblemDesc, SortMode
from grouped_gemm_gpu_kernel_amd.torch_ops import MoeGroupedGemmPlan

pytestmark = pytest.mark.gpu

LAUNCHES = 20000
KEPT = 8 << 20


class _Mallinfo2(ctypes.Structure):
    _fields_ = [(n, ctypes.c_size_t) for n in ("arena", "ordblks", "smblks", "hblks", "hblkhd", "usmblks", "fsmblks",
                                               "uordblks", "fordblks", "keepcost")]


def _heap():
    info = ctypes.CDLL(None).mallinfo2
    info.restype = _Mallinfo2
    got = info()
    return got.uordblks + got.hblkhd


def _growth(torch, launch):
    """Heap growth over LAUNCHES launches that have run, with no wait in between or behind them, against
    the same loop's first thousand (the runtime's own pools grow to their size there)."""
    for i in range(1000):
        launch(i)
    torch.cuda.synchronize()
    time.sleep(0.2)
    gc.collect()
    before = _heap()
    for i in range(LAUNCHES):
        launch(i)
    for _ in range(30):  # the launches end, and the runtime processes their records on a thread of its own
        time.sleep(0.1)
        if _heap() - before < KEPT:
            break
    grown = _heap() - before
    torch.cuda.synchronize()
    return grown


@pytest.fixture
def executor(torch_cuda):
    torch = torch_cuda
    a = torch.ones((16, 32), device="cuda", dtype=torch.float16)
    b = torch.ones((32, 16), device="cuda", dtype=torch.float16)
    d = torch.zeros((16, 16), device="cuda")
    cfg = KernelConfig.named("64x64x16")
    prob = ProblemDesc(16, 16, 32, a.data_ptr(), b.data_ptr(), None, d.data_ptr(), 32, 16, 16, 16, 1.0, 0.0)
    with GroupedGemmExecutor() as ex:
        assert ex.build(api.prepare_problem_set([prob], cfg, SortMode.kNone), cfg) == 0
        yield ex, d


@pytest.mark.parametrize("streams, run", [(1, 1), (2, 1), (2, 64), (2, 100)])
def test_run_loop_keeps_a_bounded_number_of_launches(torch_cuda, executor, streams, run):
    """`run` launches in a row on each stream.  The streams are not ordered (an event between them would
    be a record of its own): every launch writes the same one tile."""
    torch = torch_cuda
    ex, d = executor
    on = [torch.cuda.Stream() for _ in range(streams)]
    torch.cuda.synchronize()

    def launch(i):
        assert ex.run(on[(i // run) % streams]) == 0

    grown = _growth(torch, launch)
    print(f"{streams} streams, {run} in a row: heap +{grown >> 10} KB over {LAUNCHES} launches", flush=True)
    assert grown < KEPT
    assert (d == 32.0).all()


def test_moe_loop_keeps_a_bounded_number_of_launches(torch_cuda):
    torch = torch_cuda
    a = torch.ones((32, 64), device="cuda", dtype=torch.float16)
    b = torch.ones((4, 64, 64), device="cuda", dtype=torch.float16)
    d = torch.zeros((32, 64), device="cuda")
    counts = torch.full((4,), 8, device="cuda", dtype=torch.int32)
    plan = MoeGroupedGemmPlan(a, b, d)
    grown = _growth(torch, lambda i: plan.run(counts))
    print(f"moe: heap +{grown >> 10} KB over {LAUNCHES} launches", flush=True)
    assert grown < KEPT
    assert (d == 64.0).all()


def test_a_rebuild_waits_for_launches_that_carried_the_event(torch_cuda):
    """Launches 2 to 64 on a stream signal the event themselves, the 65th has it recorded behind it: a
    rebuild after any of them leaves what they computed alone."""
    torch = torch_cuda
    cfg = KernelConfig.named("64x64x16")
    a = torch.ones((512, 2048), device="cuda", dtype=torch.float16)
    b = torch.ones((2048, 512), device="cuda", dtype=torch.float16)

    def prepared(d):
        p = ProblemDesc(512, 512, 2048, a.data_ptr(), b.data_ptr(), None, d.data_ptr(), 2048, 512, 512, 512, 1.0, 0.0)
        return api.prepare_problem_set([p], cfg, SortMode.kNone)

    with GroupedGemmExecutor() as ex:
        for launches in (1, 2, 63, 64, 65, 66):
            first, second = torch.zeros((512, 512), device="cuda"), torch.zeros((512, 512), device="cuda")
            torch.cuda.synchronize()
            assert ex.build(prepared(first), cfg) == 0
            for _ in range(launches):
                assert ex.run() == 0
            assert ex.build(prepared(second), cfg) == 0  # rewrites the descriptors the launches read
            assert ex.run() == 0
            torch.cuda.synchronize()
            assert (first == 2048.0).all() and (second == 2048.0).all(), launches
