"""Launches of about as many work tiles as workgroups: with at most one tile per workgroup every tile is
assigned without the claim counters (also those of chunks that hold more tiles than workgroups start
there), with one tile more they are claimed.  D is the same bit for bit as from a small persistent
grid, where all but the first tiles are claimed, and so is D of a second run."""
import pytest

from grouped_gemm_gpu_kernel_amd import api
from grouped_gemm_gpu_kernel_amd.api import GroupedGemmExecutor, KernelConfig, ProblemDesc, SortMode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mfma", [True, False])
@pytest.mark.parametrize("count", [1, 9, 45, 130])
def test_grids_around_the_tile_count(torch_cuda, count, mfma):
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(count)
    probs, ds = [], []
    keep = []
    for i in range(count):
        # a few deep problems among shallow ones: chunks of equal time hold unequal numbers of tiles
        m, n, k = 1 + 37 * i % 150, 1 + 53 * i % 140, 1000 if i % 11 == 0 else 1 + 29 * i % 90
        a = (torch.rand((m, k), device="cuda", generator=g) - 0.5).half()
        b = (torch.rand((k, n), device="cuda", generator=g) - 0.5).half()
        d = torch.empty((m, n), device="cuda")
        probs.append(ProblemDesc(m, n, k, a.data_ptr(), b.data_ptr(), None, d.data_ptr(), k, n, n, n, 1.0, 0.0))
        keep.append((a, b))
        ds.append(d)

    def run(persistent):
        cfg = KernelConfig.named("64x64x16", use_tensor_cores=mfma, persistent_ctas=persistent)
        with GroupedGemmExecutor() as ex:
            assert ex.build(api.prepare_problem_set(probs, cfg, SortMode.kByTiles), cfg) == 0
            for _ in range(2):
                for d in ds:
                    d.fill_(float("nan"))
                assert ex.run() == 0
                torch.cuda.synchronize()
            return ex.launched_work_tiles(), [d.clone() for d in ds]

    tiles, want = run(3)
    for (a, b), d in zip(keep, want):
        torch.testing.assert_close(d.double(), a.double() @ b.double(), rtol=0, atol=2.0 ** -24 * 1001 * 250)
    for persistent in sorted({max(1, tiles - 1), tiles, tiles + 1, tiles + 5, tiles + 8, 2 * tiles + 3, 0}):
        print(f"{count} problems, {tiles} tiles, grid {persistent}", flush=True)
        _, got = run(persistent)
        for x, y in zip(got, want):
            assert torch.equal(x.view(torch.int32), y.view(torch.int32)), persistent
