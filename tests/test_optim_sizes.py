"""The optimizer's host checks: tensors that do not belong together are refused
before anything is launched (the library raises on any use here), and a matrix
beyond the one-pass update's range takes the two operators."""

import pytest
import torch

from attention_nn_amd import optim as G


class _NoLaunch:
    def __getattr__(self, name):
        raise AssertionError(f"{name} reached")


@pytest.fixture(autouse=True)
def host_only(monkeypatch):
    monkeypatch.setattr(G, "_f32", lambda t: t.to(torch.float32).contiguous())
    monkeypatch.setattr(G._lib, "lib", lambda: _NoLaunch())


def _unaligned(shape):
    n = torch.Size(shape).numel()
    return torch.zeros(n + 1)[1:].view(shape)


@pytest.mark.parametrize("op", [
    lambda a, b: G.adam_step(b, a, b, b, 0.9, 0.95, 1e-8, 1e-3, 1e-4),
    lambda a, b: G.adam_step(b, b, a, b, 0.9, 0.95, 1e-8, 1e-3, 1e-4),
    lambda a, b: G.adam_step(b, b, b, a, 0.9, 0.95, 1e-8, 1e-3, 1e-4),
    lambda a, b: G.muon_momentum(b, a, 0.95),
    lambda a, b: G.muon_apply(b, a, 0.02, 1.2),
], ids=["adam_g", "adam_m", "adam_v", "momentum_buf", "apply_u"])
def test_operand_shorter_than_what_is_read(op):
    with pytest.raises(ValueError, match="elements"):
        op(torch.zeros(15), torch.zeros(16))


@pytest.mark.parametrize("N,param", [(16, torch.zeros), (16, _unaligned), (12, torch.zeros)],
                         ids=["one_pass", "unaligned", "columns_not_of_8"])
def test_update_of_another_size_than_the_parameter(N, param):
    v = torch.zeros((2, 8, N), dtype=torch.bfloat16)
    sm = torch.zeros((2, 1, N))
    for shape in ((3, 8, N), (2, 4, N)):
        with pytest.raises(ValueError, match="belong together"):
            G._normuon_update(v, sm, 0.9, param(shape), 0.02, 1.2)
    with pytest.raises(ValueError, match="belong together"):
        G._normuon_update(v, sm[:1], 0.9, param((2, 8, N)), 0.02, 1.2)


def test_matrix_beyond_the_one_pass_update_takes_the_two_operators(monkeypatch):
    v = torch.empty((1, 1 << 17, 1 << 16), dtype=torch.bfloat16, device="meta")
    p, sm = torch.empty(v.shape, device="meta"), torch.empty((1, 1 << 17, 1), device="meta")
    monkeypatch.setattr(G, "normuon_rescale", lambda v, sm, beta2: ("u", sm))
    monkeypatch.setattr(G, "muon_apply", lambda p, u, lr, wd: (u, lr, wd))
    got, gsm = G._normuon_update(v, sm, 0.9, p, 0.02, 1.2)
    assert got == ("u", 0.02, 1.2) and gsm is sm
