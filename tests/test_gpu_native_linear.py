"""The native common case of mi355x_fp8_linear against the wrapper's own path, over the forms it
accepts and the ones it leaves to the wrapper."""

import ctypes

import pytest
import torch

from minillm_amd import _lib
from minillm_amd import mi355x_fp8 as fp8
from minillm_amd.build import LIB_PATH
from minillm_amd.validation import ModelShape, bitwise_equal, make_activations, make_weights

pytestmark = pytest.mark.gpu
N, K = 384, 256


def _operands(m, dtype=torch.bfloat16):
    w, ws = make_weights(ModelShape("native", N, K), 9, "cuda")
    return make_activations(m, K, 9, dtype).cuda(), w, ws


def _wrapper(monkeypatch, *args, **kwargs):
    with monkeypatch.context() as patch:
        patch.setattr(_lib.load_native(), "linear", lambda *a: None)
        return fp8.mi355x_fp8_linear(*args, **kwargs)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("m", [1, 8, 9, 33, 200])
def test_native_equals_wrapper(monkeypatch, m, dtype):
    x, w, ws = _operands(m, dtype)
    wide = torch.zeros((m, K + 64), dtype=dtype, device="cuda")
    wide[:, :K] = x
    other = torch.float16 if dtype == torch.bfloat16 else torch.bfloat16
    wt = w.view(torch.uint8).t().contiguous().t().view(torch.float8_e4m3fn)  # column-major weight: the wrapper copies it
    bias = torch.ones(N, device="cuda", dtype=dtype)
    for args, kw in (((x, w, ws, [128, 128]), {}), ((wide[:, :K], w, ws, (128, 128)), {}),
                     ((x.view(1, m, K), w, ws, [128, 128]), {}), ((x, w, ws, [128, 128]), {"output_dtype": other}),
                     ((x, w, ws.t().contiguous().t(), [128, 128]), {"path": "split"}), ((x, wt, ws, [128, 128]), {}),
                     ((x.t().contiguous().t(), w, ws, [128, 128]), {}), ((x, w, ws, [128, 128]), {"bias": bias}),
                     ((wide.view(1, m, K + 64)[..., :K], w, ws, [128, 128]), {})):
        got = fp8.mi355x_fp8_linear(*args, **kw)
        assert bitwise_equal(got, _wrapper(monkeypatch, *args, **kw)), (args[0].shape, kw)
        assert bitwise_equal(got, fp8.mi355x_fp8_linear(*args, **kw))


def test_native_leaves_the_rest_to_the_wrapper():
    x, w, ws = _operands(4)
    native = _lib.load_native().linear
    fp8.mi355x_fp8_linear(x, w, ws, [128, 128])
    buffers = fp8._workspace._buffers
    assert native(x, w, ws, None, buffers) is not None
    assert native(x, w, ws, None, {}) is None                       # no workspace yet on this stream
    assert native(x, w, ws, torch.float32, buffers) is None
    assert native(x.float(), w, ws, None, buffers) is None
    assert native(x[:, :-1], w, ws, None, buffers) is None
    assert native(x[:0], w, ws, None, buffers) is None
    assert native(x, w, ws[:1], None, buffers) is None
    assert native(x.cpu(), w, ws, None, buffers) is None
    with pytest.raises(TypeError):
        fp8.mi355x_fp8_linear(x, w, ws, [128, 128], output_dtype=torch.float32)
    with pytest.raises(RuntimeError):
        fp8.mi355x_fp8_linear(x, w, ws[:1], [128, 128])
    with pytest.raises(ValueError):
        fp8.mi355x_fp8_linear(x, w, ws, [128, 128], path="typo")


def test_native_on_other_streams_and_after_clear():
    """A new stream, a larger call than any before on it, and a cleared workspace all go through the
    wrapper once and natively afterwards, with the same bits."""

    x, w, ws = _operands(300)
    ref = fp8.mi355x_fp8_linear(x, w, ws, [128, 128])
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        outs = [fp8.mi355x_fp8_linear(x[:m], w, ws, [128, 128]) for m in (20, 20, 300, 300, 7)]
    stream.synchronize()
    for m, out in zip((20, 20, 300, 300, 7), outs):
        assert bitwise_equal(out, ref[:m])
    fp8._workspace.clear()
    assert bitwise_equal(fp8.mi355x_fp8_linear(x, w, ws, [128, 128]), ref)


def test_native_reports_a_failed_launch(monkeypatch):
    """A HIP error that the launch check finds (here one left behind by a refused host call) is
    raised by the native call as by the wrapper, once, and not covered up by a second launch."""

    x, w, ws = _operands(33)
    ref = fp8.mi355x_fp8_linear(x, w, ws, [128, 128])
    torch.cuda.synchronize()
    hip_set_device = ctypes.CDLL(LIB_PATH).hipSetDevice
    args = (x, w, ws, [128, 128])
    for call in (lambda: _wrapper(monkeypatch, *args), lambda: fp8.mi355x_fp8_linear(*args)):
        assert hip_set_device(4096) != 0
        with pytest.raises(RuntimeError, match=r"launch failed \(status 4\)"):
            call()
        assert bitwise_equal(call(), ref)
