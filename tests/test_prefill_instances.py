"""Every prefill kernel instance that the dispatch reaches on 256 CUs (tile, ring depth, and the
plain, K-tail and SiLU*up forms): the list below is checked against the planner on the CPU, and each
instance against the register-staged kernel on the GPU, bit for bit."""

import ctypes

import pytest
import torch

from minillm_amd import _lib
from minillm_amd import mi355x_fp8 as fp8
from minillm_amd.validation import ModelShape, bit_mismatch_details, bitwise_equal, make_activations, make_weights

CUS = 256
TILE128 = next(c for c in fp8.GEMM_CONFIGS if c.name == "tile128")

# (rows, width, ring) -> (M, N, K groups).  The ring: its stages where the tiles fit one per CU,
# "many" where they do not; the 192- and 256-row tiles have one ring each.
CASES = {
    (64, 64, 3): (65, 96, 4), (64, 64, 4): (65, 96, 5), (64, 64, 6): (65, 96, 29), (64, 64, "many"): (17, 16800, 5),
    (64, 96, 4): (17, 17632, 5),
    (64, 128, 3): (17, 24832, 4), (64, 128, 4): (17, 24832, 5), (64, 128, "many"): (17, 33280, 5),
    (96, 64, 4): (65, 8480, 6), (96, 96, 4): (65, 16800, 7), (96, 128, 4): (65, 24832, 5),
    (128, 64, 4): (98, 12544, 5), (128, 64, "many"): (5442, 672, 5),
    (128, 96, 4): (98, 16800, 5),
    (128, 128, 3): (98, 24832, 5), (128, 128, 4): (98, 24832, 29), (128, 128, "many"): (263, 21440, 5),
    (128, 160, 3): (65, 33280, 5), (128, 160, "many"): (263, 22528, 5),
    (192, 128, ""): (131, 22528, 5), (192, 160, ""): (131, 31712, 5), (192, 256, ""): (263, 27392, 5),
    (256, 128, ""): (196, 21440, 5), (256, 160, ""): (196, 33280, 5), (256, 192, ""): (395, 21440, 5),
    (256, 224, ""): (395, 24832, 5), (256, 256, ""): (395, 28768, 5),
}
TAIL_CASES = {key: case for key, case in CASES.items() if key[0] <= 128}
TAIL_CASES[128, 128, "many"] = (131, 22528, 5)
TAIL_CASES[128, 160, "many"] = (131, 33280, 5)


def _tile(m, n, k):
    kernel, rows, bn = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert _lib.load().mi355x_fp8_dispatch_choice(m, n, k, CUS, kernel, rows, bn) == _lib.OK
    return None if kernel.value == _lib.CONFIG_STREAM else (rows.value, bn.value)


def _instance(m, n, k):
    """The instance that an aligned M x N x K call launches (launch_tile_dma's choice of the ring),
    or None for the decode kernel."""

    tile = _tile(m, n, k)
    if tile is None or tile[0] > 128:
        return tile and (*tile, "")
    if -(-m // tile[0]) * -(-n // tile[1]) > CUS:
        return (*tile, "many")
    groups = -(-k // 128)
    if tile == (64, 64) and groups >= 24 and 1 <= m % 64 <= 40:
        return (*tile, 6)
    three = tile == (128, 160) or (tile == (128, 128) and groups <= 28) or (tile in ((64, 64), (64, 128)) and groups <= 4)
    return (*tile, 3 if three else 4)


def _tail_k(key, groups):
    """A depth of ``groups`` K groups whose last one holds 16, or 112, columns."""

    return 128 * (groups - 1) + (16 if key[0] == 128 else 112)


def _reachable(depths):
    rows = sorted({int(round(17 * 1.06 ** i)) for i in range(100)} | {128 * i for i in range(1, 33)})
    widths = [32 * i for i in range(1, 20)] + [32 * int(20 * 1.05 ** i) for i in range(82)]
    return {_instance(m, n, k) for k in depths for m in rows for n in widths} - {None}


def test_the_list_holds_every_reachable_instance():
    for key, (m, n, groups) in CASES.items():
        assert _instance(m, n, 128 * groups) == key
        assert _lib.load().mi355x_fp8_block_gemm_silu_fits(0x10000000, 128 * groups, m, n, 128 * groups) == 1
    for key, (m, n, groups) in TAIL_CASES.items():
        assert _instance(m, n, _tail_k(key, groups)) == key
    assert _reachable((128, 640, 3712)) == set(CASES)
    assert _reachable((144, 656, 3600)) == set(TAIL_CASES)


def _operands(m, n, k, dtype=torch.bfloat16):
    w, ws = make_weights(ModelShape("instance", n, k), 21, "cuda")
    x = make_activations(m, k, 21, dtype).cuda()
    q, s = fp8.quantize_mi355x_fp8_activation(x)  # row-major scales: the register-staged kernel
    ref = torch.empty((m, n), device="cuda", dtype=dtype)
    fp8.launch_block_gemm(q, w, ref, s, ws, TILE128)
    return x, w, ws, ref


def _ids(key):
    return "x".join(map(str, key[:2])) + (f"-{key[2]}" if key[2] else "")


@pytest.mark.gpu
@pytest.mark.parametrize("key", CASES, ids=_ids)
def test_whole_k_instances(key):
    m, n, groups = CASES[key]
    for dtype in (torch.bfloat16, torch.float16):
        x, w, ws, ref = _operands(m, n, 128 * groups, dtype)
        got = fp8.mi355x_fp8_linear(x, w, ws, [128, 128])
        assert bitwise_equal(got, ref), (dtype, bit_mismatch_details(got, ref))


@pytest.mark.gpu
@pytest.mark.parametrize("key", TAIL_CASES, ids=_ids)
def test_k_tail_instances(key):
    m, n, groups = TAIL_CASES[key]
    for dtype in (torch.bfloat16, torch.float16):
        x, w, ws, ref = _operands(m, n, _tail_k(key, groups), dtype)
        got = fp8.mi355x_fp8_linear(x, w, ws, [128, 128])
        assert bitwise_equal(got, ref), (dtype, bit_mismatch_details(got, ref))


@pytest.mark.gpu
@pytest.mark.parametrize("key", CASES, ids=_ids)
def test_silu_instances(key):
    m, n, groups = CASES[key]
    x, w, ws, gate_up = _operands(m, n, 128 * groups)
    q, s = fp8.quantize_mi355x_fp8_activation(x, scale_layout="kgroup")
    ref = fp8.silu_mul_quant_mi355x_fp8(gate_up[:, :n // 2], gate_up[:, n // 2:], return_intermediate=True)[0]
    got = fp8._gemm_silu(q, s, w, ws)
    assert got is not None and bitwise_equal(got, ref), bit_mismatch_details(got, ref)
