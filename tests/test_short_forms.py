"""The kernels' short forms of a division and of a reciprocal square root, over every value they
can meet: on the CPU for every estimate within the hardware's stated accuracy
(tests/c/short_forms_check.c), and on the GPU through the quantizer and SiLU*up."""

import os
import shutil
import subprocess

import numpy as np
import pytest
import torch

import oracle
from _helpers import bits16, codes

HERE = os.path.dirname(os.path.abspath(__file__))


def test_short_forms_match_ieee_exhaustively(tmp_path):
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("gcc not available")
    exe = str(tmp_path / "short_forms_check")
    subprocess.run([gcc, "-O2", "-ffp-contract=off", "-fopenmp", "-o", exe,
                    os.path.join(HERE, "c", "short_forms_check.c"), "-lm"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert run.returncode == 0, run.stdout + run.stderr
    assert run.stdout.count(" 0 mismatches") == 3


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_quantizer_over_every_amax(dtype):
    """One group per finite amax of the format, holding the 16-bit values next to every midpoint of
    two e4m3 codes: codes and scales are the oracle's, bit for bit."""

    from minillm_amd import mi355x_fp8 as fp8

    amax = torch.arange(0x8000, dtype=torch.int32).to(torch.int16).view(dtype)
    amax = amax[torch.isfinite(amax)]
    grid = torch.arange(127, dtype=torch.uint8).view(torch.float8_e4m3fn).float()  # 0 .. 448
    mid = (grid[1:] + grid[:-1]) / 2
    scale = amax.float() / torch.full((1,), 448.0)
    x = torch.zeros((amax.numel(), 128), dtype=dtype)
    x[:, 0] = amax
    x[:, 1:127] = torch.minimum(mid * scale.clamp_min(1e-12)[:, None], amax.float()[:, None]).to(dtype)
    x[:, 2::3] *= -1
    q, s = fp8.quantize_mi355x_fp8_activation(x.cuda())
    q_ref, s_ref = oracle.act_quant(bits16(x), is_fp16=dtype == torch.float16)
    assert np.array_equal(s.cpu().numpy().view(np.uint32), s_ref.view(np.uint32))
    assert np.array_equal(codes(q.cpu()), q_ref)


@pytest.mark.gpu
def test_silu_equals_its_long_form_over_every_bf16_gate():
    """bf16(g / (1 + exp(-g))) of all 65536 gates, up = 1, against the same expression in torch on
    the GPU (ROCm's expf and IEEE division), bit for bit but for a NaN's payload: in order, where
    whole groups of eight take one form, and shuffled, where a group mixes both ranges."""

    from minillm_amd import mi355x_fp8 as fp8

    ordered = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda()
    shuffled = ordered[torch.randperm(65536, generator=torch.Generator().manual_seed(0)).cuda()]
    for gate in (ordered, shuffled):
        g = gate.float()
        ref = (g / (1.0 + torch.exp(-g))).bfloat16()
        h = fp8.silu_mul_quant_mi355x_fp8(gate.view(512, 128), torch.ones_like(gate).view(512, 128),
                                          return_intermediate=True)[0].flatten()
        assert torch.equal(torch.isnan(h), torch.isnan(ref))
        number = ~torch.isnan(ref)
        assert torch.equal(h[number].view(torch.int16), ref[number].view(torch.int16))
