"""Streaming verify at K that is not a whole number of ring rounds (the last
stages of a tile are zeros): one, two and three padded stages, tiles past V,
one and several tiles per workgroup, row chunks, the fp32 forms and a bias.
Tokens equal the oracle's argmax wherever the two best logits are 1e-3 apart,
and the column-group kernel's."""
import pytest
import torch

from oracle import eager as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("dtype,K", [(torch.bfloat16, 576), (torch.float16, 640),
                                     (torch.bfloat16, 704), (torch.float16, 1984),
                                     (torch.float32, 288), (torch.float32, 320),
                                     (torch.float32, 352)])
@pytest.mark.parametrize("B,D,V", [(1, 1, 130), (5, 7, 20001), (16, 7, 70000)])
def test_padded_stages(dtype, K, B, D, V, bias, tune):
    from mtp_hip import ops
    g = torch.Generator().manual_seed(K + V)
    h = torch.randn(B, D + 1, K, generator=g).to(dtype)
    W = (0.05 * torch.randn(V, K, generator=g)).to(dtype)
    b = (0.1 * torch.randn(V, generator=g)).to(dtype) if bias else None
    top, gap = O.logits_top(h.reshape(-1, K), W, b)
    draft = top.reshape(B, D + 1)[:, 1:].clone().to(torch.int32)
    draft[0, 0] = (draft[0, 0] + 1) % V
    hd, Wd, dd = h.to(DEV), W.to(DEV), draft.to(DEV)
    bd = b.to(DEV) if bias else None
    assert ops.verify_route(hd, Wd, bd) == "stream"
    print(f"case padded verify {dtype} K={K} B={B} D={D} V={V} bias={bias}", flush=True)
    a, n, c, t = ops.multi_verify(hd, Wd, dd, bd, return_top=True)
    sure = gap > 1e-3
    assert torch.equal(t.cpu().reshape(-1)[sure], top[sure].to(torch.int32))
    tune(verify_wstream=1)
    a2, n2, c2, t2 = ops.multi_verify(hd, Wd, dd, bd, return_top=True)
    assert torch.equal(t2.cpu().reshape(-1)[sure], t.cpu().reshape(-1)[sure])
    if bool(sure.all()):
        assert torch.equal(a, a2) and torch.equal(n, n2) and torch.equal(c, c2)


def test_non_finite_weights_stay_in_their_rows():
    """The zero stages multiply nothing of the next row."""
    from mtp_hip import ops
    g = torch.Generator().manual_seed(3)
    K, V = 576, 5000
    h = torch.randn(4, K, generator=g).to(torch.bfloat16)
    W = (0.05 * torch.randn(V, K, generator=g)).to(torch.bfloat16)
    W[77, 0] = float("nan")
    top, _ = O.logits_top(h, W)
    d = torch.zeros(4, dtype=torch.int32, device=DEV)
    _, t = ops.verify(h.to(DEV), W.to(DEV), d)
    assert t.cpu().tolist() == top.tolist() == [77] * 4


def test_workspace_refused_as_before():
    """A shape that needed the column-group kernel's workspace still does."""
    from mtp_hip import _lib as L
    lib = L.load()
    need = lib.mtp_verify_workspace_bytes(L.BF16, 4, 1, 5000, 576)
    fake = 4096
    assert lib.mtp_fused_verify(fake, L.BF16, 4, 576, fake, L.BF16, 5000, None, 0, fake, fake,
                                fake, fake, need - 1, None) == L.ERR_WORKSPACE
