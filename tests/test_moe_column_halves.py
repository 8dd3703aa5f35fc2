"""Device-prepared launches of few work tiles claim each 256 x 256 work tile as its two column halves
(csrc/gg_kernels.hip) when that leaves at most one half per workgroup (256 of them).  Tile counts up to
the line, on it (128), one past it (129) and far past it (whole tiles, at 256 one each, at 264 claimed),
one column, widths that end inside the first half, on it and one past it (an empty second half, a
one-column one), with and without C: D must have the bits of the host-prepared launch of the same
problems, and nothing past it may be written."""
import numpy as np
import pytest

from grouped_gemm_gpu_kernel_amd import api, torch_ops
from grouped_gemm_gpu_kernel_amd.api import KernelConfig, ProblemDesc, SortMode

pytestmark = pytest.mark.gpu


def work_tiles(counts, n):
    return sum(-(-int(m) // 256) for m in counts) * -(-n // 256)


def check(torch, counts, n, with_c):
    experts, k = len(counts), 70
    rows, guard = int(counts.sum()), 3
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    a = (torch.rand((rows, k), device="cuda", generator=g) * 2 - 1).half()
    b = (torch.rand((experts, k, n), device="cuda", generator=g) * 2 - 1).half()
    c = torch.rand((rows, n), device="cuda", generator=g) if with_c else None
    full = torch.full((rows + guard, n), float("nan"), device="cuda")
    want = torch.full((rows, n), float("nan"), device="cuda")
    cfg = KernelConfig.named("128x64x32")
    print(f"moe column halves: {experts} experts, n = {n}, rows {rows}", flush=True)
    plan = torch_ops.MoeGroupedGemmPlan(a, b, full[:rows], c, 1.5, 0.5, config=cfg)
    for _ in range(2):
        full.fill_(float("nan"))
        plan.run(torch.from_numpy(counts).cuda())
    probs, r0 = [], 0
    for e in range(experts):
        m = int(counts[e])
        probs.append(ProblemDesc(m, n, k, a.data_ptr() + 2 * r0 * k, b[e].data_ptr(),
                                 c.data_ptr() + 4 * r0 * n if with_c else None, want.data_ptr() + 4 * r0 * n, k, n, n,
                                 n, 1.5, 0.5))
        r0 += m
    assert api.run_grouped_gemm_once(probs, SortMode.kByTiles, cfg) == 0
    torch.cuda.synchronize()
    assert not torch.isnan(full[:rows]).any() and torch.isnan(full[rows:]).all()
    assert torch.equal(full[:rows].view(torch.int32), want.view(torch.int32))
    grid = plan.moe.grid_ctas()
    plan.close()
    return grid


@pytest.mark.parametrize("with_c", [False, True])
@pytest.mark.parametrize("experts,n,most", [(1, 1, 40), (1, 128, 256), (3, 129, 300), (5, 300, 257), (16, 2048, 100),
                                            (43, 700, 60), (2, 16384, 256), (9, 255, 129)])
def test_column_halves(torch_cuda, experts, n, most, with_c):
    """At most 128 work tiles: column halves."""
    counts = np.random.RandomState(experts * 1000 + n).randint(0, most + 1, experts).astype(np.int32)
    counts[0] = most
    grid = check(torch_cuda, counts, n, with_c)
    assert 2 * work_tiles(counts, n) <= grid


@pytest.mark.parametrize("with_c", [False, True])
@pytest.mark.parametrize("experts,n,tiles", [(16, 2048, 128), (43, 700, 129), (26, 1100, 130), (32, 2048, 256),
                                             (33, 2048, 264)])
def test_both_sides_of_the_line(torch_cuda, experts, n, tiles, with_c):
    counts = np.random.RandomState(experts + n).randint(1, 101, experts).astype(np.int32)
    assert work_tiles(counts, n) == tiles
    grid = check(torch_cuda, counts, n, with_c)
    assert grid == 256 and (2 * tiles <= grid) == (tiles <= 128)
