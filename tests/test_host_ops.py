"""The module that four operators' calls go through (csrc/host_ops.cpp): what it does not take it leaves to the long way, and what
it takes has the long way's results, shapes, types, errors and stream."""
import importlib

import pytest

torch = pytest.importorskip("torch")
mynn = importlib.import_module("my-nn-engine_amd")


class Nothing:
    def __getattr__(self, name):
        return lambda *a: None


class Sub(torch.Tensor):
    pass


def test_what_is_not_a_plain_gpu_tensor_is_left_alone():
    ops = mynn._host_ops()
    x, w, s = torch.ones(2, 32), torch.ones((4, 32), dtype=torch.int8), torch.ones(4)
    q = torch.ones(1, 2, 1, 64)
    for a in ((x, w, s), (x.as_subclass(Sub), w, s), (x.to("meta"), w.to("meta"), s.to("meta")), (x, w, None), (x.numpy(), w, s), (x, w), ()):
        assert ops.dequant_matmul(*a) is None
    for a in ((w, s, w, s), (w, s, w), (1, 2, 3, 4)):
        assert ops.quantized_matmul(*a) is None
    assert ops.dynamic_quantize_linear(x) is None and ops.dynamic_quantize_linear("x") is None
    for a in ((q, q, q, 0.1, False, None, None, None, None), (q,), (None,) * 9):
        assert ops.attention(*a) is None
    with pytest.raises(TypeError):
        ops.bind()
    with pytest.raises(ValueError):
        ops.bind(mynn.MynnError, 0, 0, 0, 0, 0)


def make_nothing(path, monkeypatch):
    pass


def make_garbage(path, monkeypatch):
    (path / "lib").mkdir()
    (path / "lib" / "_host_ops.so").write_bytes(b"not a module")


def make_one_for_another_torch(path, monkeypatch):
    (path / "lib").mkdir()
    import os
    import shutil

    shutil.copy(os.path.join(mynn._HERE, "lib", "_host_ops.so"), path / "lib" / "_host_ops.so")
    monkeypatch.setattr(torch, "__version__", "2.3.1+other")


@pytest.mark.parametrize("make", [make_nothing, make_garbage, make_one_for_another_torch])
def test_without_the_module_the_long_way_stays_open(make, tmp_path, monkeypatch):
    import warnings

    make(tmp_path, monkeypatch)
    mynn.lib()
    monkeypatch.setattr(mynn, "_HERE", str(tmp_path))
    monkeypatch.setattr(mynn, "_ops", None)
    with pytest.warns(RuntimeWarning, match="ctypes"):
        ops = mynn._host_ops()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert mynn._host_ops() is ops  # said once
    assert ops.dequant_matmul(1, 2, 3) is None and ops.attention() is None


@pytest.mark.gpu
def test_operators_work_without_the_module(tmp_path, monkeypatch):
    w, s = torch.ones((8, 64), dtype=torch.int8, device="cuda"), torch.ones(8, device="cuda")
    x = torch.ones((2, 64), device="cuda")
    monkeypatch.setattr(mynn, "_HERE", str(tmp_path))
    monkeypatch.setattr(mynn, "_ops", None)
    with pytest.warns(RuntimeWarning, match="ctypes"):
        assert torch.equal(mynn.dequant_matmul(x, w, s), torch.full((2, 8), 64.0, device="cuda"))


@pytest.fixture
def both(monkeypatch):
    """f -> (its result through the module, its result without)"""
    def run(f):
        fast = f()
        with monkeypatch.context() as m:
            m.setattr(mynn, "_ops", Nothing())
            return fast, f()

    return run


def same(a, b):
    if isinstance(a, tuple):
        return type(b) is tuple and len(a) == len(b) and all(same(x, y) for x, y in zip(a, b))
    return (a is None and b is None) or (a.dtype == b.dtype and a.shape == b.shape and a.device == b.device and a.stride() == b.stride()
                                         and not a.requires_grad and torch.equal(a, b))


@pytest.mark.gpu
@pytest.mark.parametrize("T", [torch.float16, torch.bfloat16, torch.float32])
def test_results_are_those_of_the_long_way(both, T):
    gen = torch.Generator(device="cuda").manual_seed(5)
    w = torch.randint(-127, 128, (48, 64), generator=gen, dtype=torch.int8, device="cuda")
    s = (torch.rand(48, generator=gen, device="cuda") * 1e-2).to(T)
    for shape in ((64,), (1, 64), (5, 64), (2, 3, 64), (33, 64)):
        x = torch.randn(shape, generator=gen, device="cuda").to(T).requires_grad_()
        assert same(*both(lambda: mynn.dequant_matmul(x, w, s)))
        if len(shape) > 1:
            assert same(*both(lambda: mynn.dynamic_quantize_linear(x.detach())))
    assert same(*both(lambda: mynn.dequant_matmul(torch.ones(3, 64, device="cuda").to(T), w, torch.nn.Parameter(s))))
    y, ys, _ = mynn.dynamic_quantize_linear(torch.randn((7, 64), generator=gen, device="cuda").to(T))
    for acc in (False, True):
        assert same(*both(lambda: mynn.quantized_matmul(y, ys, w, s, want_acc=acc)))
    k = torch.randn((2, 2, 70, 64), generator=gen, device="cuda").to(T)
    for sq, causal, active, off in ((1, False, None, None), (1, False, 33, None), (20, True, 60, None), (20, True, 60, 40), (70, True, 70, None)):
        q = torch.randn((2, 8, sq, 64), generator=gen, device="cuda").to(T)
        assert same(*both(lambda: mynn.attention(q, k, k, 0.125, causal, active, q_pos_offset=off)))
    if T != torch.float32:
        codes = torch.randint(-127, 128, (2, 2, 70, 64), generator=gen, dtype=torch.int8, device="cuda")
        ks = (torch.rand((2, 2, 70), generator=gen, device="cuda") * 1e-2).to(T)
        q = torch.randn((2, 8, 1, 64), generator=gen, device="cuda").to(T)
        assert same(*both(lambda: mynn.attention(q, codes, codes, 0.125, active=50, k_scale=ks, v_scale=ks)))
        assert same(*both(lambda: mynn.attention(q, k, k, 1, active=torch.tensor(50).item())))


@pytest.mark.gpu
def test_errors_are_those_of_the_long_way(monkeypatch):
    w, s, x = torch.ones((8, 64), dtype=torch.int8, device="cuda"), torch.ones(8, device="cuda"), torch.ones((2, 64), device="cuda")
    calls = [lambda: mynn.dequant_matmul(x.repeat(1, 2)[:, ::2], w, s),          # not contiguous
             lambda: mynn.dequant_matmul(x, w, s.cpu()),                         # another device
             lambda: mynn.dequant_matmul(x.double(), w, s),                      # no such type
             lambda: mynn.dequant_matmul(x[:0], w, s),                           # no rows: the library's own error
             lambda: mynn.quantized_matmul(w[:, :24].contiguous(), s, w[:, :24].contiguous(), s, want_acc=False),  # K % 32
             lambda: mynn.dynamic_quantize_linear(x[:0]),
             lambda: mynn.attention(x, x, x, 1.0),
             lambda: mynn.attention(x.view(1, 2, 1, 64), x.view(1, 2, 1, 64), x.view(1, 2, 1, 64), 1.0, active=7)]
    for i, f in enumerate(calls):
        seen = []
        for ops in (mynn._host_ops(), Nothing()):
            monkeypatch.setattr(mynn, "_ops", ops)
            try:
                r = f()
                seen.append(("result", None if r is None else "value"))
            except Exception as e:
                seen.append((type(e), str(e)))
        assert seen[0] == seen[1], (i, seen)


@pytest.mark.gpu
def test_the_current_stream_is_the_one_used():
    w, s = torch.ones((64, 64), dtype=torch.int8, device="cuda"), torch.ones(64, device="cuda").half()
    x = torch.zeros((1, 64), device="cuda").half()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):  # (a launch on another stream would not be recorded)
            out = mynn.dequant_matmul(x, w, s)
    x.fill_(1.0)
    for _ in range(2):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, torch.full_like(out, 64.0))
