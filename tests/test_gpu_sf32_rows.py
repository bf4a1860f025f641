"""Small fp32 linear kernel at 33 .. 64 rows (two row chunks): the second
chunk of one row and of 32, columns past a tile, K inside and past a 64-k
block, both sides of the K and N lines; |y - ref| <= 1e-5 (|ref| + RMS(ref))
for fp32 sums of at most 4096 terms."""
import pytest
import torch

from conftest import close
from oracle import eager as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("gamma,bias", [(True, False), (False, True)])
@pytest.mark.parametrize("M", [33, 48, 64])
@pytest.mark.parametrize("N,K", [(1, 16), (257, 80), (970, 1280), (4096, 1536), (4097, 512),
                                 (300, 1552)])
def test_rows_33_to_64(M, N, K, gamma, bias):
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g)
    W = 0.02 * torch.randn(N, K, generator=g)
    gm = 1 + 0.1 * torch.randn(K, generator=g) if gamma else None
    b = 0.1 * torch.randn(N, generator=g) if bias else None
    print(f"case sf32 rows M={M} N={N} K={K}", flush=True)
    y = mk.fused_rmsnorm_linear(x.to(DEV), W.to(DEV), b.to(DEV) if bias else None, 1e-6,
                                gamma=gm.to(DEV) if gamma else None)
    ok, worst = close(y, O.rmsnorm_linear(x, W, b, 1e-6, 1.0, gamma=gm), 1e-5)
    assert ok, f"worst err/bound = {worst:.3g}"


@pytest.mark.parametrize("M", [33, 48])
@pytest.mark.parametrize("N,K,tiled", [(2500, 64, True), (2064, 112, True), (2048, 64, False),
                                       (2500, 128, False)])
def test_short_rows_of_many_columns_keep_the_tiled_kernel(M, N, K, tiled, tune):
    """A second workgroup per CU pays from K 128 on: below, the planned call
    has the bits of the tiled kernel."""
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g)
    W = 0.02 * torch.randn(N, K, generator=g)
    gm = 1 + 0.1 * torch.randn(K, generator=g)
    args = [t.to(DEV) for t in (x, W)]
    print(f"case sf32 short rows M={M} N={N} K={K}", flush=True)
    y = mk.fused_rmsnorm_linear(*args, gamma=gm.to(DEV))
    ok, worst = close(y, O.rmsnorm_linear(x, W, None, 1e-6, 1.0, gamma=gm), 1e-5)
    assert ok, f"worst err/bound = {worst:.3g}"
    tune(sf32=0)
    if tiled:
        assert torch.equal(y, mk.fused_rmsnorm_linear(*args, gamma=gm.to(DEV)))
