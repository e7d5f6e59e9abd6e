"""The scratch a chunked prefill takes to split its keys is a means to speed
only: a call that cannot have it runs unsplit, as every call did without one."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import emelk

ROOT = os.path.normpath(os.path.join(os.path.dirname(__file__), ".."))
G = (1, 32, 8, 128, 32, 64)


def _need(g, n_seq, n_q, stride):
    out = ctypes.c_uint64(0)
    assert emelk.lib.emelk_attn_prefill_workspace_size(ctypes.byref(g), n_seq, n_q, stride,
                                                       ctypes.byref(out)) == emelk.ERR_NONE
    return out.value


def test_no_memory_for_the_scratch_means_none(monkeypatch):
    """On a full card the allocator raises; the call must not."""
    import torch
    g = emelk.geometry(*G)
    asked = []

    def full(n, **kw):
        asked.append(n)
        raise torch.OutOfMemoryError("no memory left")

    monkeypatch.setattr(torch, "empty", full)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert emelk._prefill_workspace(g, 1, 6, 64, None) is None
    assert asked == [_need(g, 1, 6, 64)] and asked[0] > 0


def test_executor_without_memory_for_the_scratch(tmp_path):
    """The executor is made with the workspace decode needs where there is no
    room for the prefill's, and refuses only without the former."""
    exe = str(tmp_path / "batch_decoder_memory")
    subprocess.run(["g++", "-std=c++20", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "emel.cpp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "batch_decoder_memory.cpp"),
                    os.path.join(ROOT, "emel.cpp_amd", "csrc", "batch_decoder.cpp"), "-o", exe],
                   check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and res.stdout.strip() == "ok", res.stdout + res.stderr


def _case(device, n_q=6, ctx=1900):
    import torch
    from kvsetup import Scenario
    sc = Scenario(n_layer=1, n_head=32, n_kv=8, head_dim=128, block_tokens=32, lens=[ctx + n_q],
                  seed=5)
    q = torch.from_numpy(np.random.default_rng(6).standard_normal((1, n_q, 32, 128))
                         .astype(np.float32)).to(device)
    start = torch.tensor([ctx], dtype=torch.int32, device=device)
    scale = 1.0 / np.sqrt(128)
    whole = torch.full_like(q, float("nan"))
    e = emelk.lib.emelk_attn_prefill_chunk(
        ctypes.byref(sc.g), sc.k_pool.data_ptr(), sc.v_pool.data_ptr(), 0, q.data_ptr(),
        whole.data_ptr(), 1, n_q, start.data_ptr(), sc.tables.data_ptr(), int(sc.tables.shape[1]),
        scale, torch.cuda.current_stream().cuda_stream)
    assert e == emelk.ERR_NONE
    torch.cuda.synchronize()
    assert _need(sc.g, 1, n_q, int(sc.tables.shape[1])) > 0
    return lambda out: emelk.prefill_chunk(sc.g, sc.k_pool, sc.v_pool, 0, q, out, start, sc.tables,
                                           scale), q, whole


@pytest.mark.gpu
def test_prefill_on_a_full_card(device):
    """torch's allocator at its limit: the call runs unsplit, bit for bit."""
    import torch
    print("\n[gpu-case] prefill chunk without memory for its scratch", flush=True)
    call, q, whole = _case(device)
    out = torch.full_like(q, float("nan"))
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
    try:
        hold = []  # what the reserved blocks still have free, in ever smaller pieces
        for size in (256 << 20, 16 << 20, 4 << 20, 2 << 20, (1 << 20) + 512, 64 << 10):
            try:
                while len(hold) < 20000:
                    hold.append(torch.empty(size, dtype=torch.uint8, device=device))
            except torch.OutOfMemoryError:
                pass
        assert len(hold) < 20000
        call(out)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    torch.cuda.synchronize()
    assert torch.equal(out, whole)


@pytest.mark.gpu
def test_prefill_while_another_thread_captures(device):
    """Another thread's graph capture in its default (global) mode forbids new
    device memory to every thread that has not relaxed it; a chunk call beside
    it runs, split, and the captured graph is what it would be."""
    import threading

    import torch
    print("\n[gpu-case] prefill chunk beside another thread's graph capture", flush=True)
    call, q, _ = _case(device)
    side, work = torch.cuda.Stream(), torch.cuda.Stream()
    want, out = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    x = torch.arange(1000, dtype=torch.float32, device=device)
    with torch.cuda.stream(work):
        call(want)
    torch.cuda.synchronize()
    begun, done, failed = threading.Event(), threading.Event(), []

    def chunk():
        begun.wait(60)
        try:
            with torch.cuda.stream(work):
                call(out)
        except Exception as e:  # noqa: BLE001
            failed.append(e)
        done.set()

    t = threading.Thread(target=chunk)
    t.start()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):  # empties the allocator's cache first
        y = x * 2.0
        begun.set()
        assert done.wait(60)
        y = y + 1.0
    t.join()
    assert not failed, failed
    for i in range(3):
        x.fill_(float(i))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, x * 2.0 + 1.0)
    assert torch.equal(out, want)
