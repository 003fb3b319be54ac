"""The K-split workspace of the W4A16 GEMM (gemm_workspace): one buffer per
stream that no later shape replaces, and one per graph captured on a stream
without one."""
from types import SimpleNamespace

import numpy as np
import pytest

from helpers import f16_normal, synth_w4a16


def test_bound_covers_every_shape(mcv):
    L = mcv.lib()
    need = [L.mcv_w4a16_gemm_workspace_bytes(M, K, N) for K in (1152, 1792, 2048, 2688, 3584, 3968, 8192, 16384)
            for N in (8, 64, 136, 520, 1024, 2048, 3584, 6144) for M in range(1, 600, 3)]
    assert 1 << 20 < max(need) <= mcv.GEMM_WORKSPACE_BYTES


def test_one_buffer_per_stream(mcv, monkeypatch):
    monkeypatch.setattr(mcv, "_stream", lambda stream=None: 0)
    monkeypatch.setattr(mcv, "_GEMM_WS", {})
    small = mcv.gemm_workspace(1 << 18, "cpu:0")
    large = mcv.gemm_workspace(4096 + 48 * 4 * 8192, "cpu:0")     # 77 rows after 40 of K=3584 N=1024
    assert small.data_ptr() == large.data_ptr() and int(small.max()) == 0
    assert mcv.gemm_workspace(mcv.GEMM_WORKSPACE_BYTES + 1, "cpu:0").numel() > mcv.GEMM_WORKSPACE_BYTES
    assert mcv.gemm_workspace(1, "cpu:0").data_ptr() == small.data_ptr()


def test_one_buffer_per_capture(mcv, monkeypatch):
    capture = [0]
    monkeypatch.setattr(mcv, "_stream", lambda stream=None: 0)
    monkeypatch.setattr(mcv, "lib", lambda: SimpleNamespace(mcv_stream_capture_id=lambda handle: capture[0]))
    monkeypatch.setattr(mcv, "_GEMM_WS", {})
    monkeypatch.setattr(mcv, "_GEMM_WS_CAPTURE", {})
    kept = []
    for capture[0] in (5, 6):
        ws = mcv.gemm_workspace(1, "cpu:0")
        assert all(ws.data_ptr() != k.data_ptr() for k in kept) and int(ws[:4096].max()) == 0
        assert mcv.gemm_workspace(1 << 20, "cpu:0").data_ptr() == ws.data_ptr()
        kept.append(ws)
    capture[0] = 0
    eager = mcv.gemm_workspace(1, "cpu:0")
    assert all(eager.data_ptr() != k.data_ptr() for k in kept)
    capture[0] = 7                                     # a stream that has one
    assert mcv.gemm_workspace(1 << 20, "cpu:0").data_ptr() == eager.data_ptr()


@pytest.mark.gpu
def test_capture_ids(mcv, cuda):
    import torch
    L, s, ids = mcv.lib(), torch.cuda.Stream(), set()
    assert L.mcv_stream_capture_id(None) == 0 and L.mcv_stream_capture_id(s.cuda_stream) == 0
    for _ in range(2):
        g, x = torch.cuda.CUDAGraph(), torch.zeros(4, device="cuda")
        with torch.cuda.graph(g, stream=s):
            ids.add(L.mcv_stream_capture_id(s.cuda_stream))
            x.add_(1)
        assert L.mcv_stream_capture_id(s.cuda_stream) == 0
    assert len(ids) == 2 and 0 not in ids


@pytest.mark.gpu
def test_graphs_keep_their_workspace(mcv, cuda):
    """Graphs of split calls captured without a call before them: the second
    replayed first, both at once on two streams, with larger eager calls (and
    the memory they could reuse) in between; every replay gives the eager bits."""
    import torch
    rng = np.random.default_rng(3)
    cases = []
    for M, K, N in ((40, 3584, 1024), (128, 3584, 1024)):
        _, qw, qz, sc = synth_w4a16(rng, K, N)
        w = mcv.W4A16QuantizedWeight.from_awq(qw, qz, sc)
        x = torch.from_numpy(f16_normal(rng, (M, K), 1.0).view(np.int16)).cuda().view(torch.float16)
        assert mcv.lib().mcv_w4a16_gemm_workspace_bytes(M, K, N) > 0
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = mcv.matmul_w4a16(x, w)
            out2 = mcv.matmul_w4a16(x, w)
        cases.append((x, w, graph, out, out2))
    streams = [torch.cuda.Stream() for _ in cases]
    for rep in range(3):
        want = [mcv.matmul_w4a16(x, w).clone() for x, w, *_ in cases]
        junk = [torch.full((1 << 20,), -1, dtype=torch.int32, device="cuda") for _ in range(4)]
        torch.cuda.synchronize()
        for (_, _, graph, _, _), s in zip(cases[::-1], streams):
            with torch.cuda.stream(s):
                graph.replay()
        torch.cuda.synchronize()
        for (_, _, _, out, out2), ref in zip(cases, want):
            assert torch.equal(out.view(torch.int16), ref.view(torch.int16)), rep
            assert torch.equal(out2.view(torch.int16), ref.view(torch.int16)), rep
        assert all(int(j.max()) == -1 for j in junk)


@pytest.mark.gpu
def test_workspace_of_another_stream(mcv, cuda):
    """`stream` given and not current: allocated and cleared on it."""
    import torch
    rng = np.random.default_rng(4)
    _, qw, qz, sc = synth_w4a16(rng, 3584, 1024)
    w = mcv.W4A16QuantizedWeight.from_awq(qw, qz, sc)
    x = torch.from_numpy(f16_normal(rng, (96, 3584), 1.0).view(np.int16)).cuda().view(torch.float16)
    want = mcv.matmul_w4a16(x, w)
    torch.cuda.synchronize()
    for s in (torch.cuda.Stream(), SimpleNamespace(cuda_stream=torch.cuda.Stream().cuda_stream)):
        got = mcv.matmul_w4a16(x, w, out=torch.empty_like(want), stream=s)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
