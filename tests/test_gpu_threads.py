"""Several Python threads: native calls let the others run, and calls of two threads on one stream keep their scratch apart."""

import sys
import threading
import time

import pytest
import torch

from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


def _other_thread_runs_during(call, rounds):
    """Whether another thread's counter moves inside ``call``: with an endless switch interval the interpreter lock changes
    hands only where a thread gives it up. (Results are kept: freeing a tensor gives it up too.)"""
    count, stop, kept = [0], threading.Event(), []

    def spin():
        while not stop.is_set():
            count[0] += 1
            time.sleep(0)

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=spin)
    try:
        sys.setswitchinterval(1000.0)
        thread.start()
        for i in range(rounds):
            before = count[0]
            kept.append(call(i))
            if count[0] != before:
                return True
        return False
    finally:
        stop.set()
        sys.setswitchinterval(interval)
        thread.join()


def test_native_calls_give_up_the_interpreter_lock(gpu):
    w, b = torch.randn(3072, 8192, device=gpu).bfloat16(), torch.zeros(3072, device=gpu).bfloat16()
    xs = [torch.randn(1100 + i, 8192, device=gpu).bfloat16() for i in range(24)]
    nat = kernels.native()
    kernels.linear(xs[0][:1099], w, b)
    # a problem seen for the first time: the library ranks its kernels
    assert _other_thread_runs_during(lambda i: nat.linear(xs[i], w, b, False, None, None, None, False, None, 0), len(xs))


@pytest.mark.parametrize("kind", ["qwen", "flux", "wan"])
def test_native_blocks_give_up_the_interpreter_lock(gpu, kind):
    from test_gpu_native_path import _flux, _qwen, _wan

    model, call = {"qwen": _qwen, "flux": _flux, "wan": _wan}[kind](gpu, torch.bfloat16, 64, False)
    name = {"qwen": "qwen_block", "flux": "flux_single_block", "wan": "wan_block"}[kind]
    args = []
    real = getattr(kernels.native(), name)

    class Recorder:
        def __getattr__(self, n):
            if n != name:
                return getattr(nat, n)
            return lambda *a: (args.append(a), real(*a))[1]

    nat = kernels.native()
    with torch.inference_mode():
        kernels._nat = Recorder()
        try:
            call()
        finally:
            kernels._nat = nat
        assert args and _other_thread_runs_during(lambda i: real(*args[0]), 2000)


def test_two_threads_on_one_stream_keep_their_scratch_apart(gpu):
    """Each thread's scratch is its own; what both compute on one stream, with launches that hand partial results to each
    other through scratch, is what one computes alone."""
    # 520 units of 128 rows, eight more than run at once: their keys are split and merged by two more launches
    g = torch.Generator(device=gpu).manual_seed(0)
    qkv = [tuple(torch.randn(1, s, 4, 64, device=gpu, generator=g).bfloat16() for s in (16640, 1100, 1100)) for _ in range(2)]
    lin = [tuple(torch.randn(s, device=gpu, generator=g).bfloat16() for s in ((80, 12288), (3072, 12288))) for _ in range(2)]
    assert ";" in kernels.attn_plan(1, 16640, 1100, 4, 64)
    want = [(kernels.attn_fwd(*qkv[i], 0.125), kernels.linear(*lin[i], engine="handwritten")) for i in range(2)]
    torch.cuda.synchronize()
    addresses, results, errors = [None, None], [None, None], []
    ready = threading.Barrier(2, timeout=60)

    def work(i):
        try:
            ready.wait()
            out = [(kernels.attn_fwd(*qkv[i], 0.125), kernels.linear(*lin[i], engine="handwritten")) for _ in range(20)]
            addresses[i] = {ws.data_ptr() for pool in (kernels._ATTN_SCRATCH, kernels._LINEAR_SCRATCH) for ws in pool.values()}
            ready.wait()   # (so that neither ends, and gives its buffers back, before the other has its own)
            torch.cuda.synchronize()
            results[i] = out
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert len(addresses[0]) == len(addresses[1]) == 2 and not addresses[0] & addresses[1]
    for i in range(2):
        for attn, y in results[i]:
            assert torch.equal(attn, want[i][0]) and torch.equal(y, want[i][1])


def test_scratch_is_given_back_when_a_thread_ends_and_kept_for_graphs(gpu):
    x, w = torch.randn(80, 12288, device=gpu).bfloat16(), torch.randn(3072, 12288, device=gpu).bfloat16()
    kernels.linear(x, w, engine="handwritten")
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    thread = threading.Thread(target=lambda: kernels.linear(x, w, engine="handwritten"))
    thread.start()
    thread.join()
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before

    want = kernels.linear(x, w, engine="handwritten")
    graphs = []

    def record():
        torch.cuda.set_device(gpu)
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            kernels.linear(x, w, engine="handwritten")
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = kernels.linear(x, w, engine="handwritten")
        graphs.append((graph, y))

    thread = threading.Thread(target=record)
    thread.start()
    thread.join()
    graph, y = graphs[0]
    for _ in range(3):
        y.zero_()
        junk = [torch.full((1 << 26,), -1, dtype=torch.int32, device=gpu) for _ in range(4)]   # would land in freed scratch
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert all(bool((j == -1).all()) for j in junk)
        kernels.linear(x, w, engine="handwritten")
