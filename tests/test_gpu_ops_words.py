"""The row operators on whole 16-byte words and beside them: dimensions around
a wave's words (64 words of 4 fp32 or 8 bf16 values), remainders, row counts
that do not fill a work-group, rotated halves that are no whole words, and
buffers that are not 16-byte aligned."""

import numpy as np
import pytest
import torch

import oracle.ref_model as R

pytestmark = pytest.mark.gpu

DT = [torch.float32, torch.bfloat16]


def _x(dtype, *shape):
    g = torch.Generator().manual_seed(sum(shape))
    return torch.randn(shape, generator=g).to(dtype)


def _shifted(x):
    """x on the GPU one element past an aligned address."""
    buf = torch.empty(x.numel() + 1, dtype=x.dtype, device="cuda")
    v = buf[1:].view(x.shape)
    v.copy_(x)
    assert v.data_ptr() % 16
    return v


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("dim", [4, 8, 100, 129, 256, 260, 512, 520, 1024, 1028, 2048, 2056, 5000])
def test_rms_dims(dtype, dim):
    """fp32: sums of up to 5000 squares in another order, 1e-6 relative; bf16:
    one rounding of the result, 2^-8."""
    from attention_nn_amd import kernels as K
    for rows in (1, 3, 6):
        x = _x(dtype, rows, dim)
        ref = R.rms_f32(x.float())
        tol = 2e-6 if dtype == torch.float32 else 2.0 ** -8
        for xg in (x.cuda(), _shifted(x)):
            got = K.rms(xg).float().cpu()
            assert ((got - ref).abs() <= tol * ref.abs() + 1e-7).all()


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 255, 2048, 2051, 1 << 20])
def test_relu2_sizes(dtype, n):
    """Exact: one product in fp32, one rounding.  NaN and -inf give 0, inf inf."""
    from attention_nn_amd import kernels as K
    x = _x(dtype, n)
    x[0] = float("nan")
    x[-1] = float("inf") if n > 1 else float("nan")
    ref = torch.where(x.float() > 0, x.float(), 0.0) ** 2
    for xg in (x.cuda(), _shifted(x)):
        assert torch.equal(K.relu2(xg).cpu(), ref.to(dtype))


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("D", [4, 8, 16, 24, 32, 36, 64, 128])
def test_rope_dims(dtype, D):
    """fp32: two products and a sum per value, 1e-6 of the pair's size; bf16:
    one rounding of the result, 2^-8 of it."""
    from attention_nn_amd import kernels as K
    x = _x(dtype, 2, 7, 3, D)
    cs, sn = (t.cuda() for t in R.rope_tables(12, D))
    for pos0, inverse in ((0, False), (5, False), (2, True)):
        ref = R.rope_ht_f32(x, cs.cpu(), -sn.cpu() if inverse else sn.cpu(),
                            torch.arange(pos0, pos0 + 7))
        tol = 1e-6 * x.float().abs().max().item() * 2
        for xg in (x.cuda(), _shifted(x)):
            got = K.rope_ht(xg, cs, sn, pos0, inverse).float().cpu()
            bound = tol + (0.0 if dtype == torch.float32 else 2.0 ** -8) * ref.abs()
            assert ((got - ref).abs() <= bound).all()
