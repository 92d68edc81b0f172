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
    # 96-row tiles (128-row picks whose 96-row form fits one per CU), rows at their edges, and beside
    # them one size each that a 128x64 (577 rows) and a 64x64 tile (97 rows) takes.
    (512, 2560, 512), (536, 2560, 384), (385, 2500, 640), (577, 2560, 128), (97, 6144, 1024), (1024, 2560, 256),
    (1056, 2560, 896),
    # 96-wide tiles at every tile height, whose column halves straddle weight-scale blocks; one row and
    # ten columns on, a 96x128 tile.
    (200, 6144, 384), (32, 19456, 256), (63, 19400, 128), (128, 19456, 640), (100, 11008, 512), (864, 2560, 256),
    (865, 2570, 384),
    # K ending inside a group (16 to 112 columns of it), one group and several, every tile height.
    (333, 2880, 2880), (96, 320, 16), (65, 192, 112), (128, 129, 144), (300, 2560, 400), (700, 3000, 1200),
    (2048, 2560, 656), (1500, 6144, 336), (40, 12800, 272), (200, 6144, 400), (864, 2500, 176), (128, 19456, 208),
])
def test_linear_equals_register_kernel(m, n, k, dtype):
    shape = ModelShape("tiles", n, k)
    x = make_activations(m, k, 7, dtype).cuda()
    w, ws = make_weights(shape, 7, "cuda")
    got = fp8.mi355x_fp8_linear(x, w, ws, [128, 128])
    ref = _reference(x, w, ws, dtype)
    assert bitwise_equal(got, ref), bit_mismatch_details(got, ref)


@pytest.mark.parametrize("m,n,tile,depths", [
    (96, 320, "64x64", (128, 256, 384, 512, 640, 16, 272, 400)), (257, 6144, "64x128", (128, 384, 512, 640, 208, 528)),
    (600, 6144, "128x128", (128, 256, 384, 512, 3584, 3712, 144, 3472)),
])
def test_three_stage_ring_equals_register_kernel(m, n, tile, depths):
    """Single-wave tiles over few K groups: one group, every remainder of the three-stage ring and
    both sides of the depth where the ring gets its fourth stage; whole and ending in a tail; the
    plain output and, where K is whole, SiLU*up."""

    for k in depths:
        assert fp8.dispatch_name(m, n, k) == f"tile {tile}"
        x = make_activations(m, k, 13).cuda()
        w, ws = make_weights(ModelShape("shallow", n, k), 13, "cuda")
        got, ref = fp8.mi355x_fp8_linear(x, w, ws, [128, 128]), _reference(x, w, ws, torch.bfloat16)
        assert bitwise_equal(got, ref), (k, bit_mismatch_details(got, ref))
        if k % 128 == 0:
            q, s = fp8.quantize_mi355x_fp8_activation(x, scale_layout="kgroup")
            h = fp8.silu_mul_quant_mi355x_fp8(ref[:, :n // 2], ref[:, n // 2:], return_intermediate=True)[0]
            got = fp8._gemm_silu(q, s, w, ws)
            assert bitwise_equal(got, h), (k, bit_mismatch_details(got, h))


@pytest.mark.parametrize("m", [65, 104, 105, 128])
def test_six_stage_ring_equals_register_kernel(m):
    """64x64 tiles over many K groups, with a last row tile on both sides of the six-stage ring's
    bound and a full one: every remainder of the ring and the depth below its first, whole and ending
    in a tail; the plain output and, where K is whole, SiLU*up."""

    n = 320
    for k in (2944, 3072, 3200, 3328, 3456, 3584, 3712, 2960, 3184, 3440):
        assert fp8.dispatch_name(m, n, k) == "tile 64x64"
        x = make_activations(m, k, 17).cuda()
        w, ws = make_weights(ModelShape("deep", n, k), 17, "cuda")
        got, ref = fp8.mi355x_fp8_linear(x, w, ws, [128, 128]), _reference(x, w, ws, torch.bfloat16)
        assert bitwise_equal(got, ref), (k, bit_mismatch_details(got, ref))
        if k % 128 == 0:
            q, s = fp8.quantize_mi355x_fp8_activation(x, scale_layout="kgroup")
            h = fp8.silu_mul_quant_mi355x_fp8(ref[:, :n // 2], ref[:, n // 2:], return_intermediate=True)[0]
            got = fp8._gemm_silu(q, s, w, ws)
            assert bitwise_equal(got, h), (k, bit_mismatch_details(got, h))


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


@pytest.mark.parametrize("m,inter,k", [
    # The Qwen3-4B width at row counts that pick each tile shape; halves that end inside a tile or
    # inside a weight-scale block; one K group.
    (17, 9728, 256), (100, 9728, 128), (160, 9728, 384), (300, 9728, 256), (512, 9728, 256), (536, 9728, 640),
    (864, 9728, 128), (1024, 9728, 256), (2048, 9728, 384), (2208, 9728, 256), (200, 1040, 256), (333, 3008, 384),
    (1000, 1616, 128), (65, 16, 256), (2500, 4880, 256),
])
def test_silu_epilogue_equals_gemm_then_silu(m, inter, k):
    """h of the gate/up GEMM's epilogue against the GEMM followed by the SiLU*up kernel, bit for
    bit, and through the two public calls that use it."""

    x = make_activations(m, k, 3).cuda()
    w, ws = make_weights(ModelShape("gate_up", 2 * inter, k), 3, "cuda")
    q, s = fp8.quantize_mi355x_fp8_activation(x, scale_layout="kgroup")
    gate_up = torch.empty((m, 2 * inter), device="cuda", dtype=torch.bfloat16)
    fp8.launch_block_gemm(q, w, gate_up, s, ws)
    ref = fp8.silu_mul_quant_mi355x_fp8(gate_up[:, :inter], gate_up[:, inter:], return_intermediate=True)[0]
    h = fp8._gemm_silu(q, s, w, ws)
    if h is None:  # the decode kernel takes these rows
        assert fp8.dispatch_name(m, 2 * inter, k).startswith("stream")
    else:
        assert bitwise_equal(h, ref), bit_mismatch_details(h, ref)
    down, down_s = make_weights(ModelShape("down", 256, inter), 5, "cuda")
    out = fp8.mlp_forward_mi355x_fp8(x, w, ws, down, down_s)
    expect = torch.empty((m, 256), device="cuda", dtype=torch.bfloat16)
    hq, hs = fp8.quantize_mi355x_fp8_activation(ref, scale_layout="kgroup")
    fp8.launch_block_gemm(hq, down, expect, hs, down_s)
    assert bitwise_equal(out, expect), bit_mismatch_details(out, expect)


def test_silu_epilogue_refuses_what_it_cannot_take():
    """Decode rows, K inside a group, an odd number of 16-column tiles and row-major scales go to the
    separate kernels."""

    k = 256
    w, ws = make_weights(ModelShape("gate_up", 512, k), 1, "cuda")
    assert not fp8._gemm_silu_takes(16, k, w, ws, w.device)
    assert not fp8._gemm_silu_takes(200, k, w[:496], ws, w.device)
    assert not fp8._gemm_silu_takes(200, 240, w[:, :240], ws, w.device)
    q, s = fp8.quantize_mi355x_fp8_activation(make_activations(200, k, 1).cuda())
    assert fp8._gemm_silu(q, s, w, ws) is None


@pytest.mark.parametrize("m,inter,offset", [(24, 3072, 0), (48, 2048, 0), (200, 512, 8), (200, 512, 0)])
def test_mlp_quantizes_its_input_once(monkeypatch, m, inter, offset):
    """Where the epilogue does not take the gate/up GEMM (streamed sizes, a weight that is not
    16-byte aligned) the linear quantizes the input, and nothing else does."""

    k = 256
    w, ws = make_weights(ModelShape("gate_up", 2 * inter, k), 2, "cuda")
    down, down_s = make_weights(ModelShape("down", 256, inter), 5, "cuda")
    x = make_activations(m, k, 2).cuda()
    takes = offset == 0 and not fp8.dispatch_name(m, 2 * inter, k).startswith("stream")
    expect = fp8.mlp_forward_mi355x_fp8(x, w, ws, down, down_s)
    held = torch.empty(w.numel() + 16, device="cuda", dtype=torch.uint8)
    held[offset:offset + w.numel()] = w.view(torch.uint8).flatten()
    w = held[offset:offset + w.numel()].view(torch.float8_e4m3fn).view(2 * inter, k)
    seen = []
    quantize = fp8.quantize_mi355x_fp8_activation
    monkeypatch.setattr(fp8, "quantize_mi355x_fp8_activation",
                        lambda t, **kw: (seen.append(tuple(t.shape)), quantize(t, **kw))[1])
    assert bitwise_equal(fp8.mlp_forward_mi355x_fp8(x, w, ws, down, down_s), expect)
    assert seen == ([(m, k), (m, inter)] if takes else [])


def test_silu_over_every_bf16_gate():
    """silu(g) for all 65536 bf16 gates (up = 1): the short form within half a bf16 place of the
    exact value plus its own fp32 error (below 2^-20, so 2^-10 of the half place is ample); the
    separate kernel and the GEMM epilogue's form share it.  Infinities, NaN and gates whose
    exponential overflows keep the long form's values."""

    gate = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda().view(512, 128)
    h = fp8.silu_mul_quant_mi355x_fp8(gate, torch.ones_like(gate), return_intermediate=True)[0]
    g64, h64 = gate.double().cpu().flatten(), h.double().cpu().flatten()
    exact = g64 / (1 + torch.exp(-g64))
    inside = torch.isfinite(g64) & (g64 > -80) & (exact.abs() > 2.0 ** -120)
    half_place = torch.exp2(torch.floor(torch.log2(exact[inside].abs()))) * 2.0 ** -8
    assert ((h64[inside] - exact[inside]).abs() <= half_place * (1 + 2.0 ** -10)).all()
    assert h64[g64 == float("inf")].item() == float("inf")
    assert torch.isnan(h64[torch.isnan(g64)]).all() and torch.isnan(h64[g64 == -float("inf")]).all()
    deep = torch.isfinite(g64) & (g64 < -89)
    assert (h64[deep] == 0).all() and torch.signbit(h64[deep]).all()
    zero = h.flatten()[gate.flatten() == 0].cpu()
    assert torch.signbit(zero).tolist() == torch.signbit(gate.flatten()[gate.flatten() == 0].cpu()).tolist()
