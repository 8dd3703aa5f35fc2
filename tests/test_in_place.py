"""C and D the same matrix: tiles that ask for C before their k-loop (64-row wave blocks, the 4 x 4 form
of the path without matrix cores) and those that ask for it after theirs read it before any element of
theirs is written, and no tile reads another's.  D must have the bits of the launch with a C of its own."""
import pytest

from grouped_gemm_gpu_kernel_amd import api
from grouped_gemm_gpu_kernel_amd.api import GroupedGemmExecutor, KernelConfig, ProblemDesc, SortMode
from grouped_gemm_gpu_kernel_amd.torch_ops import MoeGroupedGemmPlan

pytestmark = pytest.mark.gpu

SHAPES = [(256, 256, 130, 0), (129, 131, 64, 0), (300, 385, 193, 3), (100, 256, 65, 1), (256, 99, 70, 0),
          (37, 91, 33, 0), (1, 1, 7, 0), (64, 64, 200, 4), (200, 7, 0, 0)]  # m, n, k, padding of C and D


def _sets(torch, launches):
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    sets, out, keep = [[] for _ in range(launches)], [], []
    for m, n, k, pad in SHAPES:
        a = (torch.rand((m, max(k, 1)), device="cuda", generator=g) * 2 - 1).half()
        b = (torch.rand((max(k, 1), n), device="cuda", generator=g) * 2 - 1).half()
        c = torch.rand((m, n + pad), device="cuda", generator=g) * 2 - 1
        d = [torch.full_like(c, float("nan"))] + [c.clone() for _ in range(launches - 1)]
        for i in range(launches):
            probs_c = c if i == 0 else d[i]
            sets[i].append(ProblemDesc(m, n, k, a.data_ptr(), b.data_ptr(), probs_c.data_ptr(), d[i].data_ptr(),
                                       max(k, 1), n, n + pad, n + pad, 1.25, -0.5))
        out.append((m, n, c, d))
        keep.append((a, b))
    return sets, out, keep


@pytest.mark.parametrize("mfma", [True, False])
@pytest.mark.parametrize("config", ["128x64x32", "64x64x16", "64x128x32"])
def test_in_place(torch_cuda, config, mfma):
    torch = torch_cuda
    cfg = KernelConfig.named(config, use_tensor_cores=mfma)
    (apart, single, once, claimed), out, keep = _sets(torch, 4)
    print(f"in place, {config}, matrix cores {mfma}", flush=True)
    assert api.run_grouped_gemm_once(apart, SortMode.kByK, cfg) == 0
    assert api.run_baseline_per_problem(single, cfg) == 0  # MFMA: 256 x 256 work tiles and their edge classes
    assert api.run_grouped_gemm_once(once, SortMode.kByK, cfg) == 0
    few = KernelConfig.named(config, use_tensor_cores=mfma, persistent_ctas=2)
    with GroupedGemmExecutor() as ex:
        assert ex.build(api.prepare_problem_set(claimed, few, SortMode.kByTiles), few) == 0
        assert ex.run() == 0
        torch.cuda.synchronize()
    for m, n, c, d in out:
        want = d[0][:, :n].contiguous().view(torch.int32)
        assert not torch.isnan(d[0][:, :n]).any(), (m, n)
        for got in d[1:]:
            assert torch.equal(got[:, :n].contiguous().view(torch.int32), want), (m, n)
            assert torch.equal(got[:, n:], c[:, n:]), (m, n)  # padding untouched


@pytest.mark.parametrize("persistent", [0, 2])
def test_moe_in_place(torch_cuda, persistent):
    """persistent 0: column halves; 2: whole 256 x 256 work tiles and edge classes."""
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(12)
    counts, k, n = [300, 0, 129, 64, 513], 130, 357
    rows = sum(counts)
    a = (torch.rand((rows, k), device="cuda", generator=g) * 2 - 1).half()
    b = (torch.rand((len(counts), k, n), device="cuda", generator=g) * 2 - 1).half()
    c = torch.rand((rows, n), device="cuda", generator=g) * 2 - 1
    apart, both = torch.full_like(c, float("nan")), c.clone()
    cfg = KernelConfig.named("128x64x32", persistent_ctas=persistent)
    on_gpu = torch.tensor(counts, dtype=torch.int32, device="cuda")
    for src, dst in ((c, apart), (both, both)):
        plan = MoeGroupedGemmPlan(a, b, dst, src, 1.25, -0.5, config=cfg)
        plan.run(on_gpu)
        torch.cuda.synchronize()
        plan.close()
    assert not torch.isnan(apart).any()
    assert torch.equal(apart.view(torch.int32), both.view(torch.int32))
