"""The k-loops while a claim request is in flight: their hand-counted waits differ by one then, and the
next tile's loads follow in the LDS that the tile before has left.  A grid of 3 workgroups claims all
tiles but its first ones, at depths of one to six stages (fewer than the stage buffers, prologue, main
loop, last stages), odd depths and columns (2-byte aligned rows, repaired last pieces), with padding
that holds infinities (nothing past K or N may reach D, nothing past M or N may be written).

Device-prepared launches run 256 x 256 work tiles: the phased loop on full ones, the loop in halves
with three and four buffers on row-edge, column-edge and corner ones.  Host-prepared launches of so few
problems run 128 x 128 work tiles (two buffers), or the path without matrix cores.  D must have the
bits of the per-problem launch, which claims nothing.  Against 64 bits: binary16 products are exact in
binary32, so each of the K additions of an element rounds once, and alpha and beta C add two more
roundings: |error| <= 2^-24 (K + 2) (|alpha| sum |a b| + |beta c|) (1 + 2^-20)."""
import pytest

from grouped_gemm_gpu_kernel_amd import api
from grouped_gemm_gpu_kernel_amd.api import GroupedGemmExecutor, KernelConfig, ProblemDesc, SortMode
from grouped_gemm_gpu_kernel_amd.torch_ops import MoeGroupedGemmPlan

pytestmark = pytest.mark.gpu

DEPTHS = [1, 7, 31, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 256, 257, 321]
GRID = 3


def _source(torch, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return lambda *shape: torch.rand(shape, device="cuda", generator=g) * 2 - 1


@pytest.mark.parametrize("config", ["128x64x32", "64x64x16", "64x128x32"])
@pytest.mark.parametrize("k", DEPTHS)
def test_device_prepared(torch_cuda, config, k):
    torch = torch_cuda
    uniform = _source(torch, 4000 + k)
    # Rows whole, past a half, on it and below it; columns whole and 101 of 256 in the last work tile.
    counts, n, pad = [256, 300, 100, 0, 129, 128, 513, 1], 357, 3
    rows, ld, experts = sum(counts), 357 + pad, len(counts)
    a = torch.full((rows + 1, k + pad), float("inf"), device="cuda", dtype=torch.float16)
    b = torch.full((experts, k + 1, ld), float("inf"), device="cuda", dtype=torch.float16)
    a[:rows, :k] = uniform(rows, k).half()
    b[:, :k, :n] = uniform(experts, k, n).half()
    c = uniform(rows, ld)
    d = [torch.full((rows + 1, ld), float("nan"), device="cuda") for _ in range(2)]
    cfg = KernelConfig.named(config, persistent_ctas=GRID)
    print(f"claims, device-prepared, {config}, K = {k}", flush=True)
    plan = MoeGroupedGemmPlan(a[:rows, :k], b[:, :k, :n], d[0][:rows, :n], c[:, :n], 1.25, -0.5, config=cfg)
    assert plan.moe.grid_ctas() == GRID
    counts_gpu = torch.tensor(counts, dtype=torch.int32, device="cuda")
    for _ in range(2):  # the second from counters that the first has returned to zero
        d[0].fill_(float("nan"))
        plan.run(counts_gpu)
    probs, row = [], 0
    for e, m in enumerate(counts):
        probs.append(ProblemDesc(m, n, k, a[row:].data_ptr(), b[e].data_ptr(), c[row:].data_ptr() if m else None,
                                 d[1][row:].data_ptr(), k + pad, ld, ld, ld, 1.25, -0.5))
        row += m
    assert api.run_baseline_per_problem([p for p in probs if p.m], cfg) == 0
    torch.cuda.synchronize()
    plan.close()
    for got in d:
        assert torch.isnan(got[rows:]).all() and torch.isnan(got[:, n:]).all()
    assert torch.equal(*(x[:rows, :n].contiguous().view(torch.int32) for x in d))
    row = 0
    for e, m in enumerate(counts):
        a64, b64, c64 = a[row:row + m, :k].double(), b[e, :k, :n].double(), c[row:row + m, :n].double()
        want, size = 1.25 * (a64 @ b64) - 0.5 * c64, 1.25 * (a64.abs() @ b64.abs()) + 0.5 * c64.abs()
        error = (d[0][row:row + m, :n].double() - want).abs()
        assert (error <= 2.0 ** -24 * (k + 2) * size * (1 + 2.0 ** -20)).all(), e
        row += m


@pytest.mark.parametrize("mfma", [True, False])
@pytest.mark.parametrize("config", ["128x64x32", "64x64x16", "64x128x32"])
@pytest.mark.parametrize("k", DEPTHS)
def test_host_prepared(torch_cuda, config, k, mfma):
    torch = torch_cuda
    uniform = _source(torch, 5000 + k)
    cfg = KernelConfig.named(config, use_tensor_cores=mfma, persistent_ctas=GRID)
    probs, checks, keep = [], [], []
    for m, n, pad in ((256, 256, 0), (129, 129, 0), (192, 255, 5), (100, 131, 3), (37, 90, 0), (1, 1, 0), (65, 129, 1)):
        a = torch.full((m + 1, k + pad), float("inf"), device="cuda", dtype=torch.float16)
        b = torch.full((k + 1, n + pad), float("inf"), device="cuda", dtype=torch.float16)
        a[:m, :k] = uniform(m, k).half()
        b[:k, :n] = uniform(k, n).half()
        c = uniform(m, n + pad)
        d = [torch.full((m + 1, n + pad), float("nan"), device="cuda") for _ in range(2)]
        for i in range(2):
            probs.append(ProblemDesc(m, n, k, a.data_ptr(), b.data_ptr(), c.data_ptr(), d[i].data_ptr(), k + pad,
                                     n + pad, n + pad, n + pad, 1.25, -0.5))
        checks.append((m, n, d))
        keep.append((a, b, c))
    print(f"claims, host-prepared, {config}, matrix cores {mfma}, K = {k}", flush=True)
    with GroupedGemmExecutor() as ex:
        assert ex.build(api.prepare_problem_set(probs[0::2], cfg, SortMode.kByTiles), cfg) == 0
        assert ex.grid_ctas() == GRID and ex.launched_work_tiles() > GRID
        for _ in range(2):
            for _, _, d in checks:
                d[0].fill_(float("nan"))
            assert ex.run() == 0
        torch.cuda.synchronize()
    assert api.run_baseline_per_problem(probs[1::2], cfg) == 0
    torch.cuda.synchronize()
    for (m, n, (got, single)), (a, b, c) in zip(checks, keep):
        assert torch.isnan(got[m:]).all() and torch.isnan(got[:, n:]).all(), (m, n)
        assert torch.equal(*(x[:m, :n].contiguous().view(torch.int32) for x in (got, single))), (m, n)
        a64, b64, c64 = a[:m, :k].double(), b[:k, :n].double(), c[:, :n].double()
        want, size = 1.25 * (a64 @ b64) - 0.5 * c64, 1.25 * (a64.abs() @ b64.abs()) + 0.5 * c64.abs()
        error = (got[:m, :n].double() - want).abs()
        assert (error <= 2.0 ** -24 * (k + 2) * size * (1 + 2.0 ** -20)).all(), (m, n)
