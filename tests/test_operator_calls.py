"""The Python side of an operator call: where its outputs live, and the stream it asks torch for."""
import importlib
import types

import pytest

torch = pytest.importorskip("torch")
mynn = importlib.import_module("my-nn-engine_amd")


@pytest.fixture
def calls(monkeypatch):
    """operator calls with the library's side replaced: they return what they would hand to it"""
    class Lib:
        def __getattr__(self, name):
            return lambda *a: 0

    monkeypatch.setattr(mynn, "lib", Lib)
    monkeypatch.setattr(mynn, "_ptr", lambda t: 0)
    monkeypatch.setattr(mynn, "_stream", lambda: 0)
    return mynn


def test_outputs_live_with_the_operand_they_are_made_from(calls):
    """the weight of DequantMatMul, the left operand of QuantizedMatMul; never the scale ("meta": another device)"""
    wq, scale = torch.empty((6, 32), dtype=torch.int8, device="meta"), torch.empty(6, dtype=torch.float16)
    for out in (calls.dequant_gemv(torch.empty(32), wq, scale), calls.dequant_matmul(torch.empty((2, 3, 32)), wq, scale)):
        assert out.device.type == "meta" and out.dtype == torch.float16
    assert calls.dequant_matmul(torch.empty((2, 3, 32)), wq, scale).shape == (2, 3, 6)
    out, acc = calls.quantized_matmul(wq, scale, torch.empty((5, 32), dtype=torch.int8), torch.empty(5, dtype=torch.bfloat16))
    assert out.device.type == acc.device.type == "meta" and (out.dtype, acc.dtype) == (torch.bfloat16, torch.int32)


def test_stream_without_the_raw_handle(monkeypatch):
    public = types.SimpleNamespace(_C=types.SimpleNamespace(), cuda=types.SimpleNamespace(current_stream=lambda: types.SimpleNamespace(cuda_stream=41)))
    monkeypatch.setattr(mynn, "_t", lambda: public)
    assert mynn._stream() == 41
