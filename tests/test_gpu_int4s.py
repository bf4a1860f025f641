"""Skinny INT4 kernel (at most 16 rows of 16-bit x) against the oracle, where
it can go wrong: one and two row halves, columns that end inside a tile and
inside a workgroup's tiles, K of one unit, odd units, fewer chunks than waves
and several per wave, every group the lane layout distinguishes, scales whose
rows are whole pieces and not, both nibble codes. Bound |y - ref| <= rtol
(|ref| + RMS(ref)): bf16 y 2e-2 (8 bits), f16 5e-3 (x * gamma rounded to 11
bits, 2^-12 of each term, and y to 11 bits; the sums are fp32)."""
import pytest
import torch

from conftest import close
from oracle import eager as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
RTOL = {torch.bfloat16: 2e-2, torch.float16: 5e-3}


def _case(M, N, K, group, dtype, sdt, nibble="ref", gamma=True, norm=True, scale_by=1.0):
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(M + 3 * N + K + group)
    x = torch.randn(M, K, generator=g).to(dtype)
    packed = torch.randint(0, 256, (N, K // 2), generator=g).to(torch.uint8)
    ng = -(-K // group)
    sc = (scale_by * (0.005 + 0.01 * torch.rand(N, ng, generator=g))).to(sdt)
    gm = 1 + 0.1 * torch.randn(K, generator=g) if gamma else None
    print(f"case int4s {dtype} {sdt} M={M} N={N} K={K} group={group} {nibble} {gamma} {norm}",
          flush=True)
    y = mk.fused_int4_matmul(x.to(DEV), packed.to(DEV), sc.to(DEV), K, group, nibble=nibble,
                             gamma=gm.to(DEV) if gamma else None, norm=norm)
    ref = O.int4_matmul(x, packed, sc, K, group, nibble=nibble, gamma=gm, norm=norm)
    assert y.shape == (M, N) and y.dtype == dtype
    ok, worst = close(y, ref, RTOL[dtype])
    assert ok, f"worst err/bound = {worst:.3g}"
    return y


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sdt", [torch.float16, torch.float32])
@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (8, 9, 384), (9, 65, 256), (16, 2100, 1152),
                                   (5, 4111, 4096), (13, 100, 8192), (7, 300, 8320)])
def test_sizes(M, N, K, group, dtype, sdt):
    _case(M, N, K, group, dtype, sdt, gamma=K <= 4096)


@pytest.mark.parametrize("nibble", ["ref", "twos"])
@pytest.mark.parametrize("gamma,norm", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("M", [8, 16])
def test_options(M, gamma, norm, nibble):
    for sdt in (torch.float16, torch.float32):
        _case(M, 777, 1280, 64, torch.bfloat16, sdt, nibble, gamma, norm)


@pytest.mark.parametrize("M", [3, 12])
def test_matches_the_tiled_kernel(M, tune):
    """Same call on the kernel of more rows, and the same bits on a repeat."""
    a = _case(M, 600, 2048, 128, torch.float16, torch.float16)
    assert torch.equal(a, _case(M, 600, 2048, 128, torch.float16, torch.float16))
    tune(int4s=0)
    b = _case(M, 600, 2048, 128, torch.float16, torch.float16)
    ok, worst = close(a, b.float().cpu(), 5e-3)
    assert ok, f"worst err/bound = {worst:.3g}"


def test_large_rows_and_small_scales():
    """Rows far above fp16's range are scaled per unit; scales are not rounded."""
    import mtp_kernels as mk
    _case(4, 200, 512, 32, torch.bfloat16, torch.float32, norm=False, scale_by=1e-12)
    g = torch.Generator().manual_seed(0)
    x = torch.randn(4, 512, generator=g)
    x[0] *= 1e30
    x[1, :128] *= 1e8
    x[2] *= 1e-30
    x = x.to(torch.bfloat16)
    packed = torch.randint(0, 256, (50, 256), generator=g).to(torch.uint8)
    sc = 0.01 * torch.rand(50, 4, generator=g)
    y = mk.fused_int4_matmul(x.to(DEV), packed.to(DEV), sc.to(DEV), 512, 128)
    ref = O.int4_matmul(x, packed, sc, 512, 128)
    for r in range(4):  # each row against its own scale
        ok, worst = close(y[r], ref[r], 2e-2)
        assert ok, f"row {r}: worst err/bound = {worst:.3g}"


def test_non_finite_scales_and_x_stay_in_their_columns_and_rows():
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(1)
    x = torch.randn(3, 384, generator=g).to(torch.float16)
    x[1, 5] = float("nan")
    packed = torch.randint(0, 256, (40, 192), generator=g).to(torch.uint8)
    sc = 0.01 + 0.01 * torch.rand(40, 3, generator=g)
    sc[7, 2] = float("inf")
    sc[8, 0] = float("nan")
    y = mk.fused_int4_matmul(x.to(DEV), packed.to(DEV), sc.to(DEV), 384, 128).cpu()
    ref = O.int4_matmul(x, packed, sc, 384, 128)
    assert torch.equal(torch.isfinite(y), torch.isfinite(ref))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,group", [(17, 130, 256, 32), (40, 257, 384, 64), (71, 300, 512, 128),
                                         (97, 129, 256, 32), (200, 700, 256, 128),
                                         (257, 40, 256, 64)])
def test_smaller_tiles_of_few_workgroups(M, N, K, group, dtype, tune):
    """The tiled kernel's tile per launch, planned and forced to each size."""
    for mt in (-1, 1, 2, 4):
        tune(int4_mt=mt)
        import mtp_kernels as mk
        g = torch.Generator().manual_seed(M + N)
        x = torch.randn(M, K, generator=g).to(dtype)
        packed = torch.randint(0, 256, (N, K // 2), generator=g).to(torch.uint8)
        sc = 0.005 + 0.01 * torch.rand(N, -(-K // group), generator=g)
        gm = 1 + 0.1 * torch.randn(K, generator=g)
        print(f"case int4 tiles mt={mt} {dtype} M={M} N={N} K={K}", flush=True)
        y = mk.fused_int4_matmul(x.to(DEV), packed.to(DEV), sc.to(DEV), K, group,
                                 gamma=gm.to(DEV), norm=True)
        ok, worst = close(y, O.int4_matmul(x, packed, sc, K, group, gamma=gm, norm=True), 2e-2)
        assert ok, f"mt={mt}: worst err/bound = {worst:.3g}"


@pytest.mark.parametrize("M,N,K,group,sdt", [(8, 1029, 1024, 128, torch.float16),
                                             (3, 20000, 3072, 128, torch.float32),
                                             (16, 2053, 2560, 32, torch.float16),
                                             (9, 8, 1024, 256, torch.float32),
                                             (1, 4099, 8192, 64, torch.float16)])
def test_scales_through_lds_change_no_bit(M, N, K, group, sdt, tune):
    """Whole 16-byte scale rows go through LDS: the same sums in the same
    order as with one load per tile, also where columns end inside a tile, a
    chunk has one unit and a wave several chunks."""
    y = _case(M, N, K, group, torch.bfloat16, sdt)
    tune(int4s=2)
    assert torch.equal(y, _case(M, N, K, group, torch.bfloat16, sdt))


@pytest.mark.parametrize("gamma", [None, 1.0, 1e30])
@pytest.mark.parametrize("M", [6, 13])
def test_rows_whose_sums_leave_fp32_under_the_norm(M, gamma, tune):
    """The sums hold x * gamma before the row factor: rows whose squares
    overflow are 0 (inf in x: NaN) and a huge gamma is finite, as in the
    oracle (and, but for the huge gamma, in the kernel of more rows)."""
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, 512, generator=g).to(torch.bfloat16)
    for r, mag in enumerate((1e12, 1e20, 1e35, 1e36)):
        x[r] *= mag
    x[4, ::7] = 3.3e38
    x[5, 3] = float("inf")
    packed = torch.randint(0, 256, (50, 256), generator=g).to(torch.uint8)
    sc = 0.01 * torch.rand(50, 4, generator=g)
    gm = gamma * (1 + 0.1 * torch.randn(512, generator=g)) if gamma else None
    ref = O.int4_matmul(x, packed, sc, 512, 128, gamma=gm, norm=True)
    args = [t.to(DEV) for t in (x, packed, sc)]
    gd = gm.to(DEV) if gamma else None
    for keys in ({}, {"int4s": 2}, {"int4s": 0}):
        if keys == {"int4s": 0} and gamma == 1e30:
            continue
        tune(**keys)
        print(f"case int4s large rows M={M} gamma={gamma} {keys}", flush=True)
        y = mk.fused_int4_matmul(*args, 512, 128, gamma=gd, norm=True).cpu()
        assert torch.equal(torch.isfinite(y), torch.isfinite(ref))
        for r in (0, 1, 2, 3, 4, *range(6, M)):
            ok, worst = close(y[r], ref[r], 2e-2)
            assert ok, f"{keys} row {r}: worst err/bound = {worst:.3g}"


@pytest.mark.parametrize("M", [3, 12])
def test_large_rows_without_the_norm(M):
    """A unit's power of two reaches every finite x."""
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, 256, generator=g)
    x[0] *= 1e35
    x[1] *= 1e36
    x[2, :128] *= 1e37
    x = x.to(torch.bfloat16)
    packed = torch.randint(0, 256, (50, 128), generator=g).to(torch.uint8)
    sc = 0.01 * torch.rand(50, 2, generator=g)
    y = mk.fused_int4_matmul(x.to(DEV), packed.to(DEV), sc.to(DEV), 256, 128).cpu()
    ref = O.int4_matmul(x, packed, sc, 256, 128)
    for r in range(M):
        ok, worst = close(y[r], ref[r], 2e-2)
        assert ok, f"row {r}: worst err/bound = {worst:.3g}"
