"""NorMuon and the parameter update in one pass against the two operators it
stands for, bit for bit: wide, tall, square and single-line shapes, a last
dimension that is no multiple of 8 and an unaligned parameter (both take the
two operators), a parameter of other leading dimensions, and the C entry
writing over the parameter it reads."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 64, 192), (3, 192, 64), (1, 128, 128), (2, 8, 8), (1, 1, 24),
                                   (5, 24, 8), (2, 12, 10), (2, 6, 28)])
def test_update_equals_rescale_then_apply(shape):
    from attention_nn_amd import optim as G
    g = torch.Generator().manual_seed(sum(shape))
    v = torch.randn(shape, generator=g).bfloat16().cuda()
    p = torch.randn(shape, generator=g).cuda()
    M, N = shape[-2:]
    line = (shape[0], M, 1) if M >= N else (shape[0], 1, N)
    sm = (torch.rand(line, generator=g) * 0.1).cuda()
    buf = torch.empty(p.numel() + 1, device="cuda")
    odd = buf[1:].view(shape)
    odd.copy_(p)
    u, rsm = G.normuon_rescale(v, sm, 0.9)
    ref = G.muon_apply(p, u, 0.02, 1.2)
    for q in (p, odd):
        got, gsm = G._normuon_update(v, sm, 0.9, q, 0.02, 1.2)
        assert torch.equal(got, ref) and torch.equal(gsm, rsm)
    flat, _ = G._normuon_update(v, sm, 0.9, p.reshape(-1, N), 0.02, 1.2)
    assert flat.shape == (p.numel() // N, N) and torch.equal(flat.view(shape), ref)
    with pytest.raises(ValueError):
        G._normuon_update(v, sm, 0.9, p[..., :N // 2].contiguous(), 0.02, 1.2) if N % 8 == 0 \
            else G.normuon_rescale(v, sm.reshape(-1)[1:], 0.9)


@pytest.mark.parametrize("shape", [(2, 64, 192), (3, 192, 64), (1, 1, 24), (1, 768, 3072)])
def test_update_in_place(shape):
    from attention_nn_amd import _lib, optim as G
    from attention_nn_amd._stream import current_stream
    batch, M, N = shape
    g = torch.Generator().manual_seed(sum(shape))
    v = torch.randn(shape, generator=g).bfloat16().cuda()
    p = torch.randn(shape, generator=g).cuda()
    sm = (torch.rand((batch, max(M, N)), generator=g) * 0.1).cuda()
    ref, _ = G._normuon_update(v, sm, 0.9, p, 0.02, 1.2)
    nws = _lib.lib().ann_op_normuon_ws_bytes(batch, M, N)
    ws = torch.empty(nws, dtype=torch.uint8, device="cuda")
    _lib.check(_lib.lib().ann_op_normuon_update(G._ptr(v), G._ptr(sm), batch, M, N, 0.9, G._ptr(p),
                                                0.02, 1.2, G._ptr(p), G._ptr(ws), nws,
                                                current_stream()))
    assert torch.equal(p, ref)
