"""The RMSNorm quantizer from 16 rows up (a reduction of 32 virtual threads, whole in every wave)
at the edges of its reads and loads, against the oracle."""

import numpy as np
import pytest
import torch

import oracle
from _helpers import bits16, codes
from minillm_amd import mi355x_fp8 as fp8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_residual", [False, True])
@pytest.mark.parametrize("rows,width", [
    # Vectors short of, at and past the 32 threads and the ten reads ahead (32 x 10 x 4 = 1280);
    # widths of 2, 5 and 8 16-byte loads per lane and of more than one batch; both row layouts.
    (16, 128), (17, 132), (33, 1276), (16, 1280), (40, 1284), (16, 2560), (512, 2560), (513, 2560), (1025, 2564),
    (16, 5120), (700, 5128), (31, 9728), (520, 8192), (16, 16128),
])
def test_rmsnorm_quant_wide_rows_match_oracle(rows, width, with_residual):
    gen = torch.Generator().manual_seed(rows * 31 + width)
    x = torch.randn((rows, width), generator=gen).bfloat16()
    r = torch.randn((rows, width), generator=gen).bfloat16() if with_residual else None
    w = (1 + 0.1 * torch.randn(width, generator=gen)).bfloat16()
    outs = fp8.rmsnorm_quant_mi355x_fp8(x.cuda(), w.cuda(), 1e-6, None if r is None else r.cuda(), scale_layout="row",
                                        return_intermediate=True)
    y_ref, summed_ref = oracle.rmsnorm(bits16(x), bits16(w), 1e-6, None if r is None else bits16(r))
    assert np.array_equal(bits16(outs[0].cpu()), y_ref)
    q_ref, s_ref = oracle.act_quant(y_ref)
    assert np.array_equal(codes(outs[1].cpu()), q_ref)
    assert np.array_equal(outs[2].cpu().numpy().view(np.uint32), s_ref.view(np.uint32))
    if with_residual:
        assert np.array_equal(bits16(outs[3].cpu()), summed_ref)


def test_rmsnorm_quant_infinite_and_zero_rows():
    """Rows whose mean square is infinite, NaN or zero (eps 0) keep what 1 / sqrt gives there: 0,
    NaN and infinity, so NaN where an infinity meets a zero."""

    x = torch.ones((20, 256), dtype=torch.bfloat16)
    x[3, 7] = float("inf")
    x[5, 9] = float("nan")
    x[8] = 0
    x[11] = 3e38  # the sum of squares overflows
    w = torch.ones(256, dtype=torch.bfloat16)
    y = fp8.rmsnorm_quant_mi355x_fp8(x.cuda(), w.cuda(), 0.0, scale_layout="row", return_intermediate=True)[0].cpu().float()
    ref = x.float() * torch.rsqrt(x.float().square().mean(dim=1, keepdim=True))
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    keep = ~torch.isnan(ref)
    assert torch.equal(y[keep], ref[keep])
