"""Decode attention kernel (one query per batch row and head; fp32, 16-bit
and fp8 K / V) against the oracle and against the kernels it replaces, where
it can go wrong: key counts around a step (8 .. 64 keys), a block (64) and a
chunk, every row width, chunked and whole contexts, both key sources, masks
of every dtype, rows with no key. Bound |y - ref| <= rtol (|ref| + RMS(ref)):
fp32 1e-5 (sums of up to some thousand fp32 terms and exp of fp32 scores),
16-bit outputs 2e-2 (the oracle rounds probabilities to the type)."""
import pytest
import torch

from conftest import close
from oracle import eager as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
RTOL = {torch.bfloat16: 2e-2, torch.float16: 2e-2, torch.float32: 1e-5}


def _check(out, ref, dtype):
    assert torch.equal(torch.isnan(out.cpu()), torch.isnan(ref.cpu()))
    ok, worst = close(torch.nan_to_num(out.cpu()), torch.nan_to_num(ref.cpu()), RTOL[dtype])
    assert ok, f"worst err/bound = {worst:.3g}"


@pytest.mark.parametrize("chunk_blocks", [-1, 1, 3])
@pytest.mark.parametrize("dtype,kv", [(torch.float32, "same"), (torch.bfloat16, "same"),
                                      (torch.float16, "same"), (torch.float32, "fp8"),
                                      (torch.bfloat16, "fp8"), (torch.float16, "fp8")])
@pytest.mark.parametrize("B,H,L,D", [(1, 1, 1, 64), (2, 3, 63, 256), (1, 2, 65, 64),
                                     (3, 1, 129, 128), (2, 2, 1601, 128), (1, 2, 4097, 64)])
def test_dense(B, H, L, D, dtype, kv, chunk_blocks, tune):
    import mtp_kernels as mk
    tune(attn_chunk_blocks=chunk_blocks)
    g = torch.Generator().manual_seed(B * L + D)
    q = torch.randn(B, H, D, generator=g).to(dtype)
    k, v = torch.randn(B, H, L, D, generator=g), torch.randn(B, H, L, D, generator=g)
    print(f"case decode dense {dtype} {kv} B={B} H={H} L={L} D={D} cb={chunk_blocks}", flush=True)
    if kv == "fp8":
        ks, vs = 0.01 + 0.01 * torch.rand(H, generator=g), 0.01 + 0.01 * torch.rand(H, generator=g)
        k = (k / ks[None, :, None, None]).to(torch.float8_e4m3fn)
        v = (v / vs[None, :, None, None]).to(torch.float8_e4m3fn)
        ref = O.causal_attention_fp8(q, k, v, ks, vs)
        args = [t.to(DEV) for t in (q, k, v, ks, vs)]
        out = mk.fused_causal_attention_fp8(*args)
    else:
        k, v = k.to(dtype), v.to(dtype)
        ref = O.causal_attention(q, k, v)
        args = [t.to(DEV) for t in (q, k, v)]
        out = mk.fused_causal_attention(*args)
    _check(out, ref, dtype)
    # the kernel of every other shape gives the same within the bound
    tune(attn_dec=0)
    old = (mk.fused_causal_attention_fp8 if kv == "fp8" else mk.fused_causal_attention)(*args)
    _check(out, old, dtype)


@pytest.mark.parametrize("mdtype", [torch.float32, torch.bfloat16, torch.float16, torch.bool,
                                    torch.uint8])
@pytest.mark.parametrize("dtype,D,L", [(torch.float32, 64, 300), (torch.float32, 128, 64),
                                       (torch.bfloat16, 256, 77), (torch.float16, 128, 500)])
def test_masks(dtype, D, L, mdtype, tune):
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(L)
    B, H = 2, 3
    q = torch.randn(B, H, D, generator=g).to(dtype)
    k = torch.randn(B, H, L, D, generator=g).to(dtype)
    v = torch.randn(B, H, L, D, generator=g).to(dtype)
    for mask in (torch.rand(L, generator=g) > 0.9, torch.zeros(L, dtype=torch.bool),
                 torch.arange(L) == L - 1):
        m = mask.to(mdtype)
        for cb in (-1, 1):
            tune(attn_chunk_blocks=cb)
            print(f"case decode mask {dtype} {mdtype} D={D} L={L} cb={cb}", flush=True)
            out = mk.fused_tree_attention(q.to(DEV), k.to(DEV), v.to(DEV), m.to(DEV))
            _check(out, O.tree_attention(q, k, v, mask.float()), dtype)


@pytest.mark.parametrize("dtype,B,H,L,D,ps", [(torch.bfloat16, 2, 3, 130, 128, 16),
                                              (torch.float16, 1, 2, 777, 64, 5),
                                              (torch.float32, 3, 2, 1100, 128, 32),
                                              (torch.bfloat16, 2, 2, 64, 256, 7)])
def test_paged(dtype, B, H, L, D, ps, tune):
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(L + ps)
    n = -(-L // ps)
    P = n + 2
    q = torch.randn(B, H, D, generator=g).to(dtype)
    kp = torch.randn(P, B, H, ps, D, generator=g).to(dtype)
    vp = torch.randn(P, B, H, ps, D, generator=g).to(dtype)
    table = torch.stack([torch.randperm(P, generator=g)[:n].repeat_interleave(ps)[:L]
                         for _ in range(B)]).to(torch.int32)
    ref = O.paged_attention(q, kp, vp, table, ps)
    args = [t.to(DEV) for t in (q, kp, vp, table)]
    for cb in (-1, 1, 4):
        tune(attn_chunk_blocks=cb)
        print(f"case decode paged {dtype} L={L} D={D} ps={ps} cb={cb}", flush=True)
        _check(mk.fused_paged_attention(*args, ps), ref, dtype)
    # pages outside the cache are keys that are not there
    bad = table.clone()
    bad[:, ::3] = -1
    bad[0, 1::3] = P
    out = mk.fused_paged_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), bad.to(DEV), ps)
    tune(attn_dec=0)
    _check(out, mk.fused_paged_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), bad.to(DEV), ps), dtype)


@pytest.mark.parametrize("N,H,Lc,D", [(5, 2, 100, 128), (70, 2, 65, 64), (3, 4, 0, 64)])
def test_tree_verify_fp32(N, H, Lc, D, tune):
    """Several fp32 queries per head over both key sources and a 2-D mask."""
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(N)
    ps, n = 16, -(-Lc // 16)
    q, kt, vt = (torch.randn(N, H, D, generator=g) for _ in range(3))
    kp, vp = (torch.randn(n + 1, 1, H, ps, D, generator=g) for _ in range(2))
    table = torch.randperm(n + 1, generator=g)[:n].repeat_interleave(ps)[:Lc].to(torch.int32)[None]
    tm = torch.tril((torch.rand(N, N, generator=g) > 0.5).float())
    tm.fill_diagonal_(1.0)
    ref = O.tree_verify_attention(q, kp, vp, table, ps, kt, vt, tm)
    for cb in (-1, 1):
        tune(attn_chunk_blocks=cb)
        print(f"case decode tree-verify fp32 N={N} H={H} Lc={Lc} D={D} cb={cb}", flush=True)
        out = mk.tree_verify_attention(*(t.to(DEV) for t in (q, kp, vp, table)), ps,
                                       *(t.to(DEV) for t in (kt, vt, tm)))
        _check(out, ref, torch.float32)


def test_infinite_and_nan_scores():
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(1)
    q = torch.randn(1, 1, 64, generator=g)
    k = torch.randn(1, 1, 200, 64, generator=g)
    v = torch.randn(1, 1, 200, 64, generator=g)
    for val in (float("inf"), float("nan"), -1e38):
        k2 = k.clone()
        k2[0, 0, 150, 3] = val
        out = mk.fused_causal_attention(q.to(DEV), k2.to(DEV), v.to(DEV))
        _check(out, O.causal_attention(q, k2, v), torch.float32)


def test_unaligned_rows_take_the_general_kernel():
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(2)
    q = torch.randn(1, 2, 64, generator=g)
    buf = torch.randn(2 * 50 * 64 + 1, generator=g).to(DEV)
    k = buf[1:].view(1, 2, 50, 64)
    out = mk.fused_causal_attention(q.to(DEV), k, k)
    _check(out, O.causal_attention(q, k.cpu(), k.cpu()), torch.float32)


def test_fp8_entry_without_workspace():
    """The C entry that takes no workspace reads every key in one workgroup."""
    from mtp_hip import _lib as L
    from mtp_hip import ops
    g = torch.Generator().manual_seed(4)
    B, H, N, D = 1, 2, 1000, 128
    q = torch.randn(B, H, D, generator=g).to(torch.bfloat16).to(DEV)
    k = torch.randn(B, H, N, D, generator=g).to(torch.float8_e4m3fn).to(DEV)
    v = torch.randn(B, H, N, D, generator=g).to(torch.float8_e4m3fn).to(DEV)
    s = torch.ones(H, device=DEV)
    out = torch.empty_like(q)
    st = L.load().mtp_fused_causal_attention_fp8(
        q.data_ptr(), L.BF16, B, H, D, k.data_ptr(), v.data_ptr(), N, s.data_ptr(), s.data_ptr(),
        D ** -0.5, out.data_ptr(), L.stream_handle(q.device))
    assert st == L.OK
    _check(out, ops.causal_attention_fp8(q, k, v, s, s), torch.bfloat16)


def test_16bit_needs_no_more_workspace_than_the_mfma_kernel():
    """A 16-bit call whose MFMA plan has one chunk needs no workspace; where
    the decode plan would split the keys it then keeps them whole."""
    from mtp_hip import _lib as L
    import mtp_kernels as mk
    B, H, D, N = 24, 12, 64, 512
    lib = L.load()
    with L.tuning(attn_dec=0):
        mfma = lib.mtp_attention_workspace_bytes(L.BF16, B, 1, H, D, 0, N)
    if mfma:
        pytest.skip("the MFMA kernel splits these keys on this device")
    g = torch.Generator().manual_seed(5)
    q = torch.randn(B, H, D, generator=g).to(torch.bfloat16).to(DEV)
    k, v = (torch.randn(B, H, N, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    out = torch.empty_like(q)
    st = lib.mtp_fused_causal_attention(q.data_ptr(), L.BF16, B, H, D, k.data_ptr(), v.data_ptr(),
                                        N, D ** -0.5, out.data_ptr(), None, 0,
                                        L.stream_handle(q.device))
    assert st == L.OK
    _check(out, mk.fused_causal_attention(q, k, v), torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("which", ["q", "out"])
def test_unaligned_query_or_output_needs_no_workspace(which, dtype):
    """q or out off a 16-byte boundary is none of the MFMA kernel's calls:
    with no workspace the keys stay in one workgroup, with one they split."""
    from mtp_hip import _lib as L
    import mtp_kernels as mk
    B, H, D, N = 1, 2, 128, 1000
    lib = L.load()
    code = L.BF16 if dtype == torch.bfloat16 else L.F16
    need = lib.mtp_attention_workspace_bytes(code, B, 1, H, D, 0, N)
    assert need > 0
    g = torch.Generator().manual_seed(6)
    k, v = (torch.randn(B, H, N, D, generator=g).to(dtype).to(DEV) for _ in range(2))
    bufs = [torch.zeros(B * H * D + 1, dtype=dtype, device=DEV) for _ in range(2)]
    q, out = (b[1:] if name == which else b[:-1] for b, name in zip(bufs, ("q", "out")))
    q = q.view(B, H, D).copy_(torch.randn(B, H, D, generator=g))
    ref = O.causal_attention(q.cpu(), k.cpu(), v.cpu())
    ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
    for w, n in ((None, 0), (ws.data_ptr(), need)):
        print(f"case decode unaligned {which} {dtype} workspace={n}", flush=True)
        st = lib.mtp_fused_causal_attention(q.data_ptr(), code, B, H, D, k.data_ptr(), v.data_ptr(),
                                            N, D ** -0.5, out.data_ptr(), w, n,
                                            L.stream_handle(q.device))
        assert st == L.OK
        _check(out.view(B, H, D), ref, dtype)
    _check(mk.fused_causal_attention(q, k, v), ref, dtype)


@pytest.mark.parametrize("B,H,D,L,N,dtype", [(1, 2, 128, 1000, 512, torch.float32),
                                             (24, 12, 64, 512, 600, torch.bfloat16),
                                             (5, 70, 64, 130, 130, torch.float16)])
def test_monolith_needs_no_more_workspace_than_without_the_faster_plans(B, H, D, L, N, dtype):
    """Key chunks of the decode kernel and the prompt GEMM's x * gamma are
    taken where the workspace has room; any size from the one without them on
    runs, a smaller one is refused."""
    from mtp_hip import _lib as LB
    lib = LB.load()
    code = LB.code(dtype)
    with LB.tuning(attn_dec=0, pg=0):
        least = lib.mtp_tree_attn_rmsnorm_linear_workspace_bytes(code, B, H, D, L, code, N)
    best = lib.mtp_tree_attn_rmsnorm_linear_workspace_bytes(code, B, H, D, L, code, N)
    assert best > least
    g = torch.Generator().manual_seed(N)
    q = torch.randn(B, H, D, generator=g).to(dtype)
    k, v = (torch.randn(B, H, L, D, generator=g).to(dtype) for _ in range(2))
    W = (0.05 * torch.randn(N, D, generator=g)).to(dtype)
    mask = (torch.rand(L, generator=g) > 0.4).float()
    gm = 1 + 0.1 * torch.randn(D, generator=g)
    ref = O.tree_attn_rmsnorm_linear(q, k, v, mask, W, gm)
    dev = [t.to(DEV) for t in (q, k, v, mask, W, gm)]
    qd, kd, vd, md, Wd, gd = (t.data_ptr() for t in dev)
    out = torch.empty(B, H, N, dtype=dtype, device=DEV)
    ws = torch.zeros(best + 4096, dtype=torch.uint8, device=DEV)
    for n in (best + 4096, best, best - 1, (least + best) // 2, least, least - 1):
        print(f"case monolith {dtype} B={B} H={H} workspace={n}", flush=True)
        st = lib.mtp_fused_tree_attn_rmsnorm_linear(
            qd, code, B, H, D, kd, vd, L, md, LB.F32, Wd, code, N, gd, LB.F32, None, 0, None,
            D ** -0.5, 1e-6, out.data_ptr(), ws.data_ptr(), n, LB.stream_handle(out.device))
        if n < least:
            assert st == LB.ERR_WORKSPACE
            continue
        assert st == LB.OK
        _check(out, ref, dtype)


@pytest.mark.parametrize("kv", ["same", "fp8"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_no_keys(D, dtype, kv, tune):
    """An empty context runs on every K / V type, with the rows of the
    general kernel (0 / 0)."""
    import mtp_kernels as mk
    q = torch.randn(2, 3, D, generator=torch.Generator().manual_seed(D)).to(dtype).to(DEV)
    k = torch.zeros(2, 3, 0, D, dtype=torch.float8_e4m3fn if kv == "fp8" else dtype, device=DEV)
    s = torch.ones(3, device=DEV)
    outs = []
    for dec in (-1, 0):
        tune(attn_dec=dec)
        print(f"case decode no keys {dtype} {kv} D={D} attn_dec={dec}", flush=True)
        outs.append(mk.fused_causal_attention_fp8(q, k, k, s, s) if kv == "fp8" else
                    mk.fused_causal_attention(q, k, k))
    assert torch.equal(torch.isnan(outs[0]), torch.isnan(outs[1])) and bool(outs[0].isnan().all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,L,D", [(2, 8, 448, 64), (12, 1, 192, 128), (48, 8, 96, 64),
                                     (1, 3, 3000, 128), (9, 11, 700, 128), (520, 8, 130, 64)])
def test_planned_waves_and_chunks(B, H, L, D, dtype):
    """Few and many heads at some hundred keys: workgroups of 4, 8 and 16
    waves, in one chunk and several."""
    import mtp_kernels as mk
    g = torch.Generator().manual_seed(L)
    q = torch.randn(B, H, D, generator=g).to(dtype)
    k, v = (torch.randn(B, H, L, D, generator=g).to(dtype) for _ in range(2))
    print(f"case decode planned {dtype} B={B} H={H} L={L} D={D}", flush=True)
    out = mk.fused_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV))
    _check(out, O.causal_attention(q, k, v), dtype)
