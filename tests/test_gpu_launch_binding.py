"""The native operand checks of device.dense_launch (csrc/torch_launch.cpp)
against its Python checks: the same calls are taken, with the same results, and
the same ones refused, with the same error."""
import pytest
import torch

from mlir_edsl_hip import device

CASES = ["plain", "no_bias", "strided_rows", "parameter", "one_column", "empty_rows", "int", "int_alpha_none",
         "stream", "transposed", "bias_strided", "bias_shape", "w_shape", "y_shape", "dtype_mix", "half", "host",
         "vector", "subclass", "alpha_text", "epilogue_text", "epilogue_unknown"]
REFUSED = {"transposed", "bias_strided", "bias_shape", "w_shape", "y_shape", "dtype_mix", "half", "host", "vector",
           "alpha_text", "epilogue_text", "epilogue_unknown"}


class Sub(torch.Tensor):
    pass


def call(case, dev):
    g = torch.Generator().manual_seed(3)
    t = lambda *s: torch.randint(-9, 10, s, generator=g).float().to(dev)
    x, w, b, y = t(5, 7), t(7, 6), t(6), torch.zeros(5, 6, device=dev)
    kw = {"epilogue": 3, "alpha": 0.5}
    if case == "no_bias":
        b, kw["epilogue"] = None, 2
    elif case == "strided_rows":
        x, w = t(5, 12)[:, 3:10], t(7, 9)[:, :6]
        y = torch.zeros(5, 11, device=dev)[:, 2:8]
    elif case == "parameter":
        w = torch.nn.Parameter(w)
    elif case == "one_column":
        w, b, y = t(7, 3)[:, 1:2], t(1), torch.zeros(5, 1, device=dev)
    elif case == "empty_rows":
        x, y = t(0, 7), torch.zeros(0, 6, device=dev)
    elif case.startswith("int"):
        x, w, b, y = x.int(), w.int(), b.int(), y.int()
        if case == "int_alpha_none":
            kw["alpha"] = None
    elif case == "stream":
        kw["stream"] = torch.cuda.current_stream() if dev == "cuda" else None
    elif case == "transposed":
        x = t(7, 5).t()
    elif case == "bias_strided":
        b = t(12)[::2]
    elif case == "bias_shape":
        b = t(5)
    elif case == "w_shape":
        w = t(8, 6)
    elif case == "y_shape":
        y = torch.zeros(6, 5, device=dev)
    elif case == "dtype_mix":
        w = w.int()
    elif case == "half":
        x, w, b, y = x.half(), w.half(), b.half(), y.half()
    elif case == "host":
        w = w.cpu()
    elif case == "vector":
        x = t(7)
    elif case == "subclass":
        x = x.as_subclass(Sub)
    elif case == "alpha_text":
        kw["alpha"] = "1"
    elif case == "epilogue_text":
        kw["epilogue"] = "3"
    elif case == "epilogue_unknown":
        kw["epilogue"] = 99
    try:
        device.dense_launch(x, w, b, y, **kw)
    except Exception as e:
        return type(e), str(e)
    return y.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_native_checks_agree_with_python(case, monkeypatch):
    device._torch_module()
    assert device._native_launch is not None, "the torch launch module is not built"
    native = call(case, "cuda")
    monkeypatch.setattr(device, "_native_launch", None)
    python = call(case, "cuda")
    assert isinstance(native, tuple) == (case in REFUSED), native
    if case in REFUSED:
        assert native == python
    else:
        assert torch.equal(native, python)
        assert case == "empty_rows" or native.abs().max() > 0


@pytest.mark.parametrize("case", ["plain", "no_bias", "int", "vector", "w_shape", "half", "subclass"])
def test_host_tensors_are_refused_without_the_gpu(case, monkeypatch):
    device._torch_module()
    assert device._native_launch is not None, "the torch launch module is not built"
    native = call(case, "cpu")
    monkeypatch.setattr(device, "_native_launch", None)
    assert isinstance(native, tuple) and native == call(case, "cpu")
