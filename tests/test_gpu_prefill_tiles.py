"""The LDS-DMA prefill kernel at its tile edges: 96-row tiles, the register-buffered K step at
every remainder of its four-stage ring, and depths that end inside a 128-wide K group.

Every kernel folds the same MFMA partials in the same K order, so each case is compared bit for
bit with the register-staged kernel (row-major activation scales select it)."""

import pytest
import torch

from minillm_amd import mi355x_fp8 as fp8
from minillm_amd.validation import ModelShape, bit_mismatch_details, bitwise_equal, make_activations, make_weights

pytestmark = pytest.mark.gpu
TILE128 = next(c for c in fp8.GEMM_CONFIGS if c.name == "tile128")


def _reference(x, w, ws, out_dtype):
    q, s = fp8.quantize_mi355x_fp8_activation(x)  # row-major scales: the register-staged kernel
    out = torch.empty((x.shape[0], w.shape[0]), device=x.device, dtype=out_dtype)
    fp8.launch_block_gemm(q, w, out, s, ws, TILE128)
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("m,n,k", [
    # 96-row tiles (128-row picks whose 96-row form fits one per CU), rows at their edges.
    (512, 2560, 512), (536, 2560, 384), (385, 2500, 640), (577, 2560, 128), (97, 6144, 1024), (1024, 2560, 256),
    (1056, 2560, 896),
    # K ending inside a group (16 to 112 columns of it), one group and several, every tile height.
    (333, 2880, 2880), (96, 320, 16), (65, 192, 112), (128, 129, 144), (300, 2560, 400), (700, 3000, 1200),
    (2048, 2560, 656), (1500, 6144, 336), (40, 12800, 272),
])
def test_linear_equals_register_kernel(m, n, k, dtype):
    shape = ModelShape("tiles", n, k)
    x = make_activations(m, k, 7, dtype).cuda()
    w, ws = make_weights(shape, 7, "cuda")
    got = fp8.mi355x_fp8_linear(x, w, ws, [128, 128])
    ref = _reference(x, w, ws, dtype)
    assert bitwise_equal(got, ref), bit_mismatch_details(got, ref)


@pytest.mark.parametrize("k", [144, 400])
def test_k_tail_keeps_a_nan_code_in_its_own_column(k):
    """The tail's out-of-range weight chunks read other chunks of the same row: a NaN code there
    must stay in its own output column, and the rows behind the weight are never read."""

    m, n = 200, 256
    x = make_activations(m, k, 11).cuda()
    w, ws = make_weights(ModelShape("tail", n, k), 11, "cuda")
    codes = w.view(torch.uint8).clone()
    first = k // 128 * 128
    codes[5, first] = 0x7F
    codes[17, 0] = 0x7F
    w = codes.view(torch.float8_e4m3fn)
    got = fp8.mi355x_fp8_linear(x, w, ws, [128, 128])
    ref = _reference(x, w, ws, torch.bfloat16)
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.isnan(got).all(dim=0).nonzero().flatten().tolist() == [5, 17]
    keep = [c for c in range(n) if c not in (5, 17)]
    assert bitwise_equal(got[:, keep], ref[:, keep])
