"""The operators' native host side (csrc/host.cpp) under threads, and what it does for torch around the launches.

The tests that need a library call of a known length bind the module to a stand-in library (every entry point of the C ABI
the module resolves, doing nothing or waiting on the host): no kernel runs there.
"""
import ctypes
import importlib.util
import os
import re
import subprocess
import threading
import time

import pytest
import torch

from llm_kernels_amd import _lib
from llm_kernels_amd.fast_dequant.simple_marlin.marlin import mul
from llm_kernels_amd.fast_dequant.simple_marlin.utils import QuantUtils
from llm_kernels_amd.quantization import fp8_kernel
from helpers import announce

pytestmark = pytest.mark.gpu

STAND_IN = r"""
#include <stdint.h>
#include <unistd.h>
int in_call, most_in_call, shared;
static int lock;
static void* seen[8];
static void enter(void) { while (__sync_lock_test_and_set(&lock, 1)) usleep(10); }
static void leave(void) { __sync_lock_release(&lock); }
const char* llmk_last_error(void) { return ""; }
int64_t llmk_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) { return 4096; }
int llmk_gemm_fp8_block(const void* a, const float* as, const void* b, const float* bs, void* c, int dt, int64_t M, int64_t N,
                        int64_t K, void* ws, int64_t bytes, void* stream) {
    int slot = 0;
    enter();
    for (int i = 0; i < 8; ++i) if (seen[i] == ws) shared = 1;      /* another call under way has this scratch */
    while (seen[slot]) ++slot;
    seen[slot] = ws;
    if (++in_call > most_in_call) most_in_call = in_call;
    leave();
    usleep(300000);
    enter();
    seen[slot] = 0;
    --in_call;
    leave();
    return 0;
}
"""


@pytest.fixture
def stand_in(tmp_path):
    """A second instance of the host module, bound to the stand-in library: (module, library, its scratch dictionary)."""
    text = open(os.path.join(os.path.dirname(_lib.__file__), "csrc", "host.cpp")).read()
    names = set(re.findall(r"X\((llmk_\w+)\)", text)) - set(re.findall(r"\b(llmk_\w+)\(", STAND_IN))
    src, so = tmp_path / "stand_in.c", tmp_path / "stand_in.so"
    src.write_text(STAND_IN + "".join("int %s(void) { return 0; }\n" % n for n in sorted(names)))
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-w", "-o", str(so), str(src)], check=True)
    spec = importlib.util.spec_from_file_location("llmk_host", _lib.HOST_PATH)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    kept = {}
    mod.bind(str(so), _lib.LlmkError, kept)
    return mod, ctypes.CDLL(str(so)), kept


def _fp8_operands(dev, M=4, N=128, K=128):
    z = torch.zeros
    return (z(M, K, device=dev).to(torch.float8_e4m3fn), z(M, K // 128, device=dev), z(N, K, device=dev).to(torch.float8_e4m3fn),
            z(N // 128, K // 128, device=dev))


def test_other_threads_run_during_a_library_call(dev, stand_in):
    """A launch that has to wait (a full queue, code loaded on first use) stops its own thread only."""
    announce("host calls and the interpreter's lock")
    mod, lib, _ = stand_in
    in_call = ctypes.c_int.in_dll(lib, "in_call")
    ops = _fp8_operands(dev)
    saw, stop = threading.Event(), threading.Event()

    def watch():
        while not stop.is_set():
            if in_call.value:
                saw.set()
            time.sleep(0.005)

    t = threading.Thread(target=watch)
    t.start()
    mod.fp8_gemm(*ops)
    stop.set()
    t.join()
    assert saw.is_set()


def test_calls_under_way_share_no_scratch(dev, stand_in):
    """Two threads on one stream: their launches may alternate, so each call has scratch of its own while it lasts, and one
    buffer is kept afterwards."""
    announce("host scratch under threads")
    mod, lib, kept = stand_in
    ops = _fp8_operands(dev)
    for _ in range(2):                                   # without and with a kept buffer
        threads = [threading.Thread(target=mod.fp8_gemm, args=ops) for _ in range(3)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert ctypes.c_int.in_dll(lib, "most_in_call").value > 1
        assert ctypes.c_int.in_dll(lib, "shared").value == 0
        assert len(kept) == 1 and next(iter(kept.values())).numel() >= 4096
    first = next(iter(kept.values())).data_ptr()
    mod.fp8_gemm(*ops)
    assert next(iter(kept.values())).data_ptr() == first         # one call after the other: the same buffer


def test_threads_on_one_stream_get_the_serial_results(dev):
    """Operators whose launches hand partial sums over in the scratch, from four threads: bit for bit what one thread gets."""
    announce("threads, same stream and own streams")
    torch.manual_seed(0)
    jobs = []
    for M, N, K in ((16, 1024, 8192), (48, 512, 4096), (16, 2048, 4096)):
        _, q, s = QuantUtils.fake_quantize((torch.randn(K, N, device=dev) * 0.02).half(), 128)
        B, sp = QuantUtils.pack(q, s, 128)
        A = torch.randn(M, K, device=dev).half()

        def marlin(A=A, B=B, sp=sp, M=M, N=N):
            out = torch.empty(M, N, dtype=torch.half, device=dev)
            mul(A, B, out, sp, None)
            return out
        jobs.append(marlin)
        w = fp8_kernel.weight_quant(torch.randn(N, K, device=dev) * 0.02)
        x = torch.randn(M, K, device=dev).bfloat16()
        jobs.append(lambda x=x, w=w: fp8_kernel.fp8_gemm(*fp8_kernel.act_quant(x), *w))
    want = [j() for j in jobs]
    torch.cuda.synchronize()
    for own_streams in (False, True):
        wrong = []

        def work(seed):
            stream = torch.cuda.Stream() if own_streams else torch.cuda.current_stream()
            with torch.cuda.stream(stream):
                for i in range(40):
                    k = (seed + i) % len(jobs)
                    got = jobs[k]()
                    if i % 8 == 7:
                        stream.synchronize()
                        if not torch.equal(got, want[k]):
                            wrong.append(k)

        threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert not wrong


def test_outputs_are_filled_under_deterministic_algorithms(dev):
    """torch.use_deterministic_algorithms fills new tensors, so rows that an operator leaves unwritten are the same in every
    run: the tokens of experts outside the local range here."""
    announce("deterministic fill")
    from llm_kernels_amd.moe import group_gemm_kernel as gk
    torch.manual_seed(0)
    T, E, H = 16, 4, 256
    ids = torch.arange(T, device=dev).remainder(E).view(T, 1)
    x = torch.randn(T, H, device=dev).bfloat16()
    _, src2dst, seg = gk.run_moe_ep_preproess(ids, E)
    first = seg.tolist()[2]                              # rows of experts 0 and 1: not local below
    assert torch.utils.deterministic.fill_uninitialized_memory
    torch.use_deterministic_algorithms(True)
    try:
        q, s = gk.pre_reorder_quant(x, src2dst, ids, None, 2, 3, 1, H, torch.int8)
        qf, sf = gk.pre_reorder_quant(x, src2dst, ids, None, 2, 3, 1, H, torch.float8_e4m3fn)
    finally:
        torch.use_deterministic_algorithms(False)
    assert (q[:first] == 127).all() and s[:first].isnan().all()          # what torch.empty holds then
    assert qf[:first].float().isnan().all() and sf[:first].isnan().all()
    q1, s1 = gk.pre_reorder_quant(x, src2dst, ids, None, 2, 3, 1, H, torch.int8)
    assert torch.equal(q[first:], q1[first:]) and torch.equal(s[first:], s1[first:])


def test_dispatch_modes_see_the_allocations(dev):
    announce("dispatch mode")
    from torch.utils._python_dispatch import TorchDispatchMode

    class Log(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.sizes = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            out = func(*args, **(kwargs or {}))
            if "empty" in func.__name__:
                self.sizes.append((tuple(out.shape), out.dtype))
            return out

    torch.manual_seed(0)
    x = torch.randn(3, 256, device=dev).bfloat16()
    with Log() as log:
        y, s = fp8_kernel.act_quant(x)
    assert ((3, 256), torch.float8_e4m3fn) in log.sizes and ((3, 2), torch.float32) in log.sizes
    y1, s1 = fp8_kernel.act_quant(x)
    assert torch.equal(y.view(torch.uint8), y1.view(torch.uint8)) and torch.equal(s, s1)


def test_the_profiler_sees_the_allocations(dev):
    announce("profiler")
    x = torch.randn(3, 256, device=dev).bfloat16()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        fp8_kernel.act_quant(x)
    assert sum(e.name == "aten::empty" for e in prof.events()) == 2


def test_a_captured_call_keeps_its_scratch(dev):
    """A graph goes on using the scratch it was captured with: a later call on its stream that needs more must not hand that
    memory to anyone else.  Replays, with eager calls between, give the eager result and write nothing of other tensors."""
    announce("scratch of a captured call")
    torch.manual_seed(0)

    def operands(M, N, K):
        w = fp8_kernel.weight_quant(torch.randn(N, K, device=dev) * 0.02)
        return (*fp8_kernel.act_quant(torch.randn(M, K, device=dev).bfloat16()), *w)

    small, large = operands(16, 1024, 8192), operands(16, 8192, 16384)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        want = fp8_kernel.fp8_gemm(*small)               # keeps scratch for this stream
        stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = fp8_kernel.fp8_gemm(*small)
    with torch.cuda.stream(stream):
        fp8_kernel.fp8_gemm(*large)                      # replaces it by a larger one
        others = [torch.full((1 << 18,), 0x5A, dtype=torch.uint8, device=dev) for _ in range(64)]
        others += [torch.full((1 << 20,), 0x5A, dtype=torch.uint8, device=dev) for _ in range(16)]
        for _ in range(3):
            got.zero_()
            graph.replay()
            fp8_kernel.fp8_gemm(*large)
            stream.synchronize()
            assert torch.equal(got, want)
            assert all((t == 0x5A).all() for t in others)
