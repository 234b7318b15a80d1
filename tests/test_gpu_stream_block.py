"""The library's own scratch memory of the stand-alone operators: a captured graph keeps what it was captured with when a
larger call makes the stream's block grow, graphs replayed on several streams at once share nothing, and two host threads
may call on one stream."""
import threading

import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


def linear(g, rng, M, N, K, dt=orc.F16, aligned=True):
    """operands; aligned=False: weights 8 bytes off, which the call dequantises into the stream's block"""
    import torch

    act = g.to_dev(orc.to_storage(rng.standard_normal((M, K)), dt), dt)
    flat = torch.empty(N * K + 8, dtype=torch.int8, device="cuda")
    W = flat[0 if aligned else 8:][:N * K].view(N, K)
    W.copy_(g.to_dev(rng.integers(-127, 128, (N, K)).astype(np.int8)))
    return act, W, g.to_dev(orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt), dt)


def attention(g, rng, B, L, dt=orc.F16):
    D, Hq, Hkv = 64, 32, 4
    return [g.to_dev(orc.to_storage(rng.standard_normal(s), dt), dt) for s in ((B, Hq, 1, D), (B, Hkv, L, D), (B, Hkv, L, D))]


def calls(g, rng):
    """(name, a small call whose graph is kept, a call that needs a larger block)"""
    m = g.mynn
    s, b = linear(g, rng, 32, 64, 256, aligned=False), linear(g, rng, 32, 4096, 4096, aligned=False)
    yield "dequantised weights", lambda: m.dequant_matmul(*s), lambda: m.dequant_matmul(*b)
    s2, b2 = linear(g, rng, 6, 256, 8192), linear(g, rng, 12, 4096, 14336)
    yield "K ranges of few rows", lambda: m.dequant_matmul(*s2), lambda: m.dequant_matmul(*b2)
    q = [g.to_dev(rng.integers(-127, 128, sh).astype(np.int8)) for sh in ((40, 8192), (256, 8192), (200, 8192), (4096, 8192))]
    sc = [g.to_dev(orc.to_storage(rng.uniform(1e-3, 1e-2, n), orc.F16), orc.F16) for n in (40, 256, 200, 4096)]
    yield "K ranges of int8", lambda: m.quantized_matmul(q[0], sc[0], q[1], sc[1])[0], lambda: m.quantized_matmul(q[2], sc[2], q[3], sc[3])[0]
    a, c = attention(g, rng, 1, 2304), attention(g, rng, 8, 4096)
    yield "key ranges", lambda: m.attention(*a, 0.125), lambda: m.attention(*c, 0.125)
    yield "ring rows", lambda: m.attention_streaming(*a, 0.125, False, 2304, 4, 2300, 7), lambda: m.attention_streaming(*c, 0.125, False, 4004, 4, 4000, 7)


def test_growth_between_capture_and_replay(g):
    import torch

    rng = np.random.default_rng(0)
    for name, small, large in calls(g, rng):
        print(name, flush=True)
        side = torch.cuda.Stream()  # (a stream of its own: its block begins with this call)
        with torch.cuda.stream(side):
            want = small()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                out = small()
            ref = large()
            torch.cuda.synchronize()
            # whatever was given back by now belongs to somebody else
            others = [torch.full((1 << 20,), float("nan"), device="cuda") for _ in range(64)]
            for _ in range(3):
                out.zero_()
                graph.replay()
                again = large()
                torch.cuda.synchronize()
                assert torch.equal(out, want), name
                assert torch.equal(again, ref), name
            del others


def test_graphs_of_split_products_on_two_streams(g):
    """the K ranges of a captured product use no memory that another call could meet"""
    import torch

    rng = np.random.default_rng(1)
    sides = [torch.cuda.Stream(), torch.cuda.Stream()]
    cases = list(calls(g, rng))[1:3]
    for name, one, two in cases:
        graphs, outs, wants = [], [], []
        for call in (one, two):
            with torch.cuda.stream(sides[0]):  # (captured on one stream, replayed on two)
                wants.append(call())
                torch.cuda.synchronize()
                graphs.append(torch.cuda.CUDAGraph())
                with torch.cuda.graph(graphs[-1], stream=sides[0]):
                    outs.append(call())
        for _ in range(20):
            for side, graph in zip(sides, graphs):
                with torch.cuda.stream(side):
                    graph.replay()
        torch.cuda.synchronize()
        for out, want, call in zip(outs, wants, (one, two)):
            assert torch.equal(out, want), name
            with torch.cuda.stream(sides[0]):  # ... and left nothing behind
                assert torch.equal(call(), want), name
        torch.cuda.synchronize()


def test_two_threads_on_one_stream(g):
    """both dequantise into the stream's block, one of them making it grow"""
    import torch

    rng = np.random.default_rng(2)
    side = torch.cuda.Stream()
    jobs = [[linear(g, rng, 32, 64 * (i + 1), 256, aligned=False) for i in range(4)], [linear(g, rng, 48, 512 * (i + 1), 512, aligned=False) for i in range(4)]]
    wants = [[g.mynn.dequant_matmul(*a) for a in job] for job in jobs]
    torch.cuda.synchronize()
    wrong = []

    def work(job, want):
        try:
            with torch.cuda.stream(side):
                for rep in range(25):
                    outs = [g.mynn.dequant_matmul(*a) for a in job]
                    side.synchronize()
                    wrong.extend(i for i, (o, w) in enumerate(zip(outs, want)) if not torch.equal(o, w))
        except Exception as e:  # noqa: BLE001
            wrong.append(e)

    threads = [threading.Thread(target=work, args=a) for a in zip(jobs, wants)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not wrong and not any(t.is_alive() for t in threads), wrong[:5]
