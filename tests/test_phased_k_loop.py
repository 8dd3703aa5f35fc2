"""The pipelined k-loops at the depths where they can go wrong: the phased one of the full 256 x 256
work tile (csrc/gg_phased.h) and the one in halves of its edge classes (three and four stage buffers)
and of the 128 x 128 work tile (two), csrc/gg_tiles.h.  One to six stages (fewer than the buffers,
prologue, main loop and last stages), depths around the 32-deep half stage and the 16-byte piece, odd
depths and columns (2-byte aligned rows, repaired last pieces), partial tiles, and padding that holds
infinities (nothing past K, M or N may reach D).

run_baseline_per_problem runs 256 x 256 work tiles (more than 128 rows and columns: the phased loop;
else an edge class); the grouped launch of the same few problems runs on 128 x 128 work tiles and
must give the same bits.  Against 64 bits: binary16 products are exact in binary32, so each of the K additions of an
element rounds once, and alpha and beta C add two more roundings: |error| <= 2^-24 (K + 2)
(|alpha| sum |a b| + |beta c|) (1 + 2^-20)."""
import pytest

from grouped_gemm_gpu_kernel_amd import api
from grouped_gemm_gpu_kernel_amd.api import KernelConfig, ProblemDesc, SortMode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config", ["128x64x32", "64x64x16", "64x128x32"])
@pytest.mark.parametrize("k", [1, 7, 8, 31, 32, 33, 63, 64, 65, 72, 127, 128, 129, 191, 192, 193, 256, 257, 321])
def test_depths_and_edges(torch_cuda, config, k):
    torch = torch_cuda
    cfg = KernelConfig.named(config)
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 + k)
    probs, checks, keep = [], [], []
    for m, n, pad in ((256, 256, 0), (129, 129, 0), (192, 255, 5), (300, 385, 3), (257, 131, 0), (100, 256, 0),
                      (256, 100, 1), (37, 90, 0), (128, 128, 0), (1, 1, 0), (65, 129, 0)):
        lda, ldb, ldd = k + pad, n + pad, n + pad
        a = torch.full((m + 1, lda), float("inf"), device="cuda", dtype=torch.float16)
        b = torch.full((k + 1, ldb), float("inf"), device="cuda", dtype=torch.float16)
        c = torch.rand((m, ldd), device="cuda", generator=g) * 2 - 1
        a[:m, :k] = (torch.rand((m, k), device="cuda", generator=g) * 2 - 1).half()
        b[:k, :n] = (torch.rand((k, n), device="cuda", generator=g) * 2 - 1).half()
        d = [torch.full((m + 1, ldd), float("nan"), device="cuda") for _ in range(2)]
        for i in range(2):
            probs.append(ProblemDesc(m, n, k, a.data_ptr(), b.data_ptr(), c.data_ptr(), d[i].data_ptr(), lda, ldb, ldd,
                                     ldd, 1.25, -0.5))
        a64, b64, c64 = a[:m, :k].double(), b[:k, :n].double(), c[:, :n].double()
        checks.append((m, n, d, 1.25 * (a64 @ b64) - 0.5 * c64, 1.25 * (a64.abs() @ b64.abs()) + 0.5 * c64.abs()))
        keep.append((a, b, c))
    print(f"phased k-loop, {config}, K = {k}", flush=True)
    assert api.run_baseline_per_problem(probs[0::2], cfg) == 0
    assert api.run_grouped_gemm_once(probs[1::2], SortMode.kByK, cfg) == 0
    torch.cuda.synchronize()
    for m, n, (single, grouped), want, size in checks:
        got = single[:m, :n]
        assert torch.isnan(single[m:]).all() and torch.isnan(single[:, n:]).all(), (m, n)
        assert ((got.double() - want).abs() <= 2.0 ** -24 * (k + 2) * size * (1 + 2.0 ** -20)).all(), (m, n)
        assert torch.equal(got.contiguous().view(torch.int32), grouped[:m, :n].contiguous().view(torch.int32)), (m, n)
