"""The k-loop and epilogue of the path without matrix cores at the sizes where they can go wrong: depths
around the 8-deep slice and the 64-deep stage, one to five stages (two LDS buffers), tiles with one
row, one column, a vector of four columns or a wave's rows left over, odd depths and columns (2-byte
aligned rows, repaired last pieces), and padding that holds infinities (nothing past K, M or N may
reach D, nothing past M or N may be written).

The single-problem and the grouped launch must give the same bits.  Against 64 bits: binary16 products
are exact in binary32, so each of the K additions of an element rounds once, and alpha and beta C add
two more roundings: |error| <= 2^-24 (K + 2) (|alpha| sum |a b| + |beta c|) (1 + 2^-20)."""
import pytest

from grouped_gemm_gpu_kernel_amd import api
from grouped_gemm_gpu_kernel_amd.api import KernelConfig, ProblemDesc, SortMode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config", ["64x64x16", "128x64x32", "64x128x32"])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 16, 17, 63, 64, 65, 72, 127, 128, 129, 192, 193, 257])
def test_depths_and_edges(torch_cuda, config, k):
    torch = torch_cuda
    cfg = KernelConfig.named(config, use_tensor_cores=False)
    g = torch.Generator(device="cuda")
    g.manual_seed(2000 + k)
    probs, checks, keep = [], [], []
    for i, (m, n, pad) in enumerate(((64, 64, 0), (128, 128, 0), (1, 1, 0), (65, 66, 0), (17, 3, 5), (33, 68, 3),
                                     (127, 129, 1), (16, 131, 0), (200, 63, 0), (5, 4, 0))):
        lda, ldb, ldd = k + pad, n + pad, n + pad
        a = torch.full((m + 1, lda), float("inf"), device="cuda", dtype=torch.float16)
        b = torch.full((k + 1, ldb), float("inf"), device="cuda", dtype=torch.float16)
        c = torch.full((m + 1, ldd), float("inf"), device="cuda") if i % 3 != 2 else None
        a[:m, :k] = (torch.rand((m, k), device="cuda", generator=g) * 2 - 1).half()
        b[:k, :n] = (torch.rand((k, n), device="cuda", generator=g) * 2 - 1).half()
        if c is not None:
            c[:m, :n] = torch.rand((m, n), device="cuda", generator=g) * 2 - 1
        d = [torch.full((m + 1, ldd), float("nan"), device="cuda") for _ in range(2)]
        for j in range(2):
            probs.append(ProblemDesc(m, n, k, a.data_ptr(), b.data_ptr(), c.data_ptr() if c is not None else None,
                                     d[j].data_ptr(), lda, ldb, ldd, ldd, 1.25, -0.5))
        a64, b64 = a[:m, :k].double(), b[:k, :n].double()
        c64 = c[:m, :n].double() if c is not None else torch.zeros((m, n), dtype=torch.float64, device="cuda")
        checks.append((m, n, d, 1.25 * (a64 @ b64) - 0.5 * c64, 1.25 * (a64.abs() @ b64.abs()) + 0.5 * c64.abs()))
        keep.append((a, b, c))
    print(f"FMA k-loop, {config}, K = {k}", flush=True)
    assert api.run_baseline_per_problem(probs[0::2], cfg) == 0
    assert api.run_grouped_gemm_once(probs[1::2], SortMode.kByK, cfg) == 0
    torch.cuda.synchronize()
    for m, n, (single, grouped), want, size in checks:
        got = single[:m, :n]
        assert torch.isnan(single[m:]).all() and torch.isnan(single[:, n:]).all(), (m, n)
        assert ((got.double() - want).abs() <= 2.0 ** -24 * (k + 2) * size * (1 + 2.0 ** -20)).all(), (m, n)
        assert torch.equal(got.contiguous().view(torch.int32), grouped[:m, :n].contiguous().view(torch.int32)), (m, n)
