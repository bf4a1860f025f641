"""Prompt GEMM (more than 64 rows) against the oracle, every tile shape and
K-split forced at the sizes where it can go wrong: rows and columns one past
a tile, a tile of one row or column, fewer stages than buffers, odd and
unaligned output rows, splits with an uneven last share. Bound |y - ref| <=
2e-2 (|ref| + RMS(ref)): x * gamma and y are each rounded once to 8 (bf16)
or 11 (f16) bits, the sums are fp32."""
import pytest
import torch

from conftest import close
from oracle import eager as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
TYPES = [(torch.bfloat16, "same"), (torch.bfloat16, "fp8"), (torch.float16, "same"),
         (torch.float16, "fp8")]
SHAPES = 14  # tile shapes of the kernel


def _case(M, N, K, dtype, w, gamma=True, bias=True, norm=True, seed=0):
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(seed + M + 3 * N + 7 * K)
    x = torch.randn(M, K, generator=g).to(dtype)
    W = 0.02 * torch.randn(N, K, generator=g)
    gm = 1 + 0.1 * torch.randn(K, generator=g) if gamma else None
    b = (0.1 * torch.randn(N, generator=g)).to(dtype) if bias else None
    dev = [t.to(DEV) if t is not None else None for t in (x, b, gm)]
    if w == "fp8":
        wq, ws = O.quantize_fp8_per_channel(W)
        y = mk.fused_rmsnorm_linear_fp8(dev[0], wq.to(DEV), ws.to(DEV), dev[1], 1e-6,
                                        gamma=dev[2], norm=norm)
        ref = O.rmsnorm_linear_fp8(x, wq, ws, b, 1e-6, gamma=gm, norm=norm)
    else:
        W = W.to(dtype)
        y = mk.fused_rmsnorm_linear(dev[0], W.to(DEV), dev[1], 1e-6, gamma=dev[2], norm=norm)
        ref = O.rmsnorm_linear(x, W, b, 1e-6, 1.0, gamma=gm, norm=norm)
    assert y.dtype == dtype and y.shape == (M, N)
    ok, worst = close(y, ref, 2e-2)
    assert ok, f"worst err/bound = {worst:.3g}"
    return y


@pytest.mark.parametrize("dtype,w", TYPES)
@pytest.mark.parametrize("shape", range(1, SHAPES + 1))
def test_every_tile_shape(shape, dtype, w, tune):
    tune(pg=shape)
    for M, N, K in ((65, 1, 64), (257, 257, 128), (193, 451, 192), (300, 520, 448)):
        print(f"case pg shape={shape} {dtype} {w} M={M} N={N} K={K}", flush=True)
        _case(M, N, K, dtype, w)


@pytest.mark.parametrize("dtype,w", TYPES)
@pytest.mark.parametrize("shape", range(10, SHAPES + 1))
def test_k_splits(shape, dtype, w, tune):
    for S in (2, 3, 8):
        tune(pg=shape, pg_splits=S)
        for M, N, K in ((65, 70, 64 * 4 * S), (130, 300, 64 * (4 * S + 3))):
            print(f"case pg split shape={shape} S={S} {dtype} {w} M={M} N={N} K={K}", flush=True)
            a = _case(M, N, K, dtype, w)
            assert torch.equal(a, _case(M, N, K, dtype, w))  # fixed order of the sums


@pytest.mark.parametrize("gamma,bias,norm", [(False, False, True), (False, True, False),
                                             (True, False, False)])
@pytest.mark.parametrize("dtype,w", TYPES)
@pytest.mark.parametrize("M,N,K", [(65, 513, 1024), (517, 2049, 512), (1000, 96, 2112)])
def test_planned(M, N, K, dtype, w, gamma, bias, norm):
    print(f"case pg {dtype} {w} M={M} N={N} K={K} {gamma} {bias} {norm}", flush=True)
    _case(M, N, K, dtype, w, gamma, bias, norm)


def _planned_splits(M, N, K, wcode):
    """Whether the plan of a bf16 call splits K: its partials are then part of
    the workspace asked for."""
    from mtp_hip import _lib as L
    lib = L.load()
    planned = lib.mtp_rmsnorm_linear_workspace_bytes(L.BF16, wcode, M, N, K)
    with L.tuning(pg_splits=1):
        return planned > lib.mtp_rmsnorm_linear_workspace_bytes(L.BF16, wcode, M, N, K)


@pytest.mark.parametrize("w", ["same", "fp8"])
def test_planned_splits(w):
    """A size whose plan splits K, with the same bits on a repeat."""
    from mtp_hip import _lib as L
    assert _planned_splits(128, 1000, 4096, L.FP8E4M3 if w == "fp8" else L.BF16)
    print(f"case pg planned splits {w}", flush=True)
    a = _case(128, 1000, 4096, torch.bfloat16, w)
    assert torch.equal(a, _case(128, 1000, 4096, torch.bfloat16, w))


@pytest.mark.parametrize("M,N,K,splits", [(70, 300, 2048, False), (128, 1000, 4096, True)])
def test_graph_replay(M, N, K, splits):
    """Prep and GEMM replay, without K-splits and with their partials and
    arrival counts; eager calls in between."""
    import mtp_kernels as mk
    from mtp_hip import _lib as L
    assert _planned_splits(M, N, K, L.BF16) == splits
    g = torch.Generator().manual_seed(9)
    W = (0.02 * torch.randn(N, K, generator=g)).to(torch.bfloat16).to(DEV)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    gm = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
    mk.fused_rmsnorm_linear(x, W, gamma=gm)
    torch.cuda.synchronize()
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr):
        y = mk.fused_rmsnorm_linear(x, W, gamma=gm)
    for i in range(4):
        x.copy_(torch.randn(M, K, generator=g).to(torch.bfloat16))
        ref = mk.fused_rmsnorm_linear(x, W, gamma=gm)
        gr.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref)


@pytest.mark.parametrize("dtype,w", TYPES)
@pytest.mark.parametrize("splits", [1, 4])
def test_non_finite_x_and_gamma(splits, dtype, w, tune):
    """inf and NaN in x stay in their rows, an infinite gamma reaches every
    row, as in the oracle."""
    import mtp_kernels as mk
    tune(pg=13, pg_splits=splits)
    g = torch.Generator().manual_seed(12)
    M, N, K = 90, 70, 1024
    x = torch.randn(M, K, generator=g).to(dtype)
    x[3, 5], x[64, 1000], x[89, 0] = float("inf"), float("nan"), float("-inf")
    W = 0.02 * torch.randn(N, K, generator=g)
    gm = 1 + 0.1 * torch.randn(K, generator=g)
    inf_gamma = gm.clone()
    inf_gamma[77] = float("inf")
    if w == "fp8":
        wq, ws = O.quantize_fp8_per_channel(W)
        dev = [t.to(DEV) for t in (x, wq, ws)]
    else:
        dev = [x.to(DEV), W.to(dtype).to(DEV)]
    for gamma in (gm, inf_gamma):
        print(f"case pg non-finite {dtype} {w} S={splits}", flush=True)
        if w == "fp8":
            y = mk.fused_rmsnorm_linear_fp8(*dev, gamma=gamma.to(DEV)).cpu()
            ref = O.rmsnorm_linear_fp8(x, wq, ws, None, 1e-6, gamma=gamma)
        else:
            y = mk.fused_rmsnorm_linear(*dev, gamma=gamma.to(DEV)).cpu()
            ref = O.rmsnorm_linear(x, W.to(dtype), None, 1e-6, 1.0, gamma=gamma)
        assert torch.equal(torch.isnan(y), torch.isnan(ref))
        assert torch.equal(torch.isinf(y), torch.isinf(ref))
        f = torch.isfinite(ref)
        assert bool((y[~f & ~torch.isnan(ref)] == ref[~f & ~torch.isnan(ref)]).all())
        if bool(f.any()):
            ok, worst = close(y[f], ref[f], 2e-2)
            assert ok, f"worst err/bound = {worst:.3g}"


@pytest.mark.parametrize("dtype,w", TYPES)
def test_long_prompt_in_passes(dtype, w):
    """x * gamma above 128 MiB goes in passes of whole 256-row tiles, the last
    one shorter and ragged: rows around the seams, against the oracle (K 512:
    two passes, of 66048 rows and 65953)."""
    import mtp_kernels as mk
    M, N, K = 132001, 40, 512
    g = torch.Generator().manual_seed(11)
    x = torch.randn(M, K, generator=g).to(dtype)
    W = 0.02 * torch.randn(N, K, generator=g)
    gm = 1 + 0.1 * torch.randn(K, generator=g)
    print(f"case pg passes {dtype} {w} M={M}", flush=True)
    if w == "fp8":
        wq, ws = O.quantize_fp8_per_channel(W)
        y = mk.fused_rmsnorm_linear_fp8(x.to(DEV), wq.to(DEV), ws.to(DEV), gamma=gm.to(DEV)).cpu()
        ref = O.rmsnorm_linear_fp8(x, wq, ws, None, 1e-6, gamma=gm)
    else:
        y = mk.fused_rmsnorm_linear(x.to(DEV), W.to(dtype).to(DEV), gamma=gm.to(DEV)).cpu()
        ref = O.rmsnorm_linear(x, W.to(dtype), None, 1e-6, 1.0, gamma=gm)
    for rows in (slice(0, 64), slice(66000, 66100), slice(M - 64, M), slice(0, M)):
        ok, worst = close(y[rows], ref[rows], 2e-2)
        assert ok, f"rows {rows}: worst err/bound = {worst:.3g}"


@pytest.mark.parametrize("dtype,w", TYPES)
@pytest.mark.parametrize("M,N,K,gamma", [(1000, 100, 3200, True), (999, 100, 3264, True),
                                         (1100, 113, 3200, True), (2500, 16, 4096, False),
                                         (1300, 257, 2496, True)])
def test_many_rows_of_few_columns(M, N, K, gamma, dtype, w):
    """Both sides of the line to the row-chunk kernel."""
    print(f"case pg narrow {dtype} {w} M={M} N={N} K={K} {gamma}", flush=True)
    _case(M, N, K, dtype, w, gamma=gamma)
