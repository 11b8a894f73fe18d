"""One runtime used on several streams: its workspaces and graph capture.

Calls of one runtime on different streams share the runtime's workspaces, so
the library puts a call that uses them behind the uses on the streams it was
used on before; here such calls are enqueued on streams in turn and compared
with the same calls alone, bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from gpu_util import assert_bf16_close, bf16_dev_to_f32, empty_bf16, to_dev, tuned
from qm38 import synth

pytestmark = pytest.mark.gpu


def _job(mat, dev):
    import qm38
    return qm38.Runtime.job(*(to_dev(a, dev) for a in mat), mat[0].shape[0])


@pytest.mark.parametrize("M,N,K,env", [
    (12, 700, 2048, {"QM38_Q4_LANES_SLICES": 4}),  # K slices of few rows
    (16, 5120, 17408, {}),                         # ... as the planner cuts them
    (40, 700, 4096, {"QM38_Q4_ROWS_SLICES": 4}),   # a short prompt's, and its converted rows
    (300, 300, 2048, {"QM38_GEMM_SPLITS": 3}),     # the GEMM's pieces and counters
    (3, 512, 9216, {}),                            # K parts of the MFMA streaming kernel
])
def test_workspaces_on_streams_in_turn(torch_dev, M, N, K, env):
    import torch
    rng = np.random.default_rng(M + N)
    with tuned(**env) as rt:
        mat = synth.q4_matrix(rng, N, K)
        job = _job(mat, torch_dev)
        streams = [torch.cuda.Stream() for _ in range(3)]
        xs = [to_dev(synth.bf16_normal(rng, (M, K)), torch_dev) for _ in streams]
        alone = []
        for x in xs:
            y = empty_bf16((M, N), torch_dev)
            rt.q4_project([job], x, K, M, [y])
            alone.append(y)
        busy = torch.randn(2048, 2048, device=torch_dev)
        outs = [[empty_bf16((M, N), torch_dev) for _ in range(8)] for _ in streams]
        torch.cuda.synchronize()
        for s in streams:  # the calls queue up behind work of each stream
            with torch.cuda.stream(s):
                busy @ busy
        for i in range(8):
            for s, x, o in zip(streams, xs, outs):
                rt.set_stream(s)
                rt.q4_project([job], x, K, M, [o[i]])
        torch.cuda.synchronize()
        rt.set_stream(torch.cuda.current_stream())
        assert_bf16_close(bf16_dev_to_f32(alone[0]),
                          oracle.q4_project(xs[0].cpu().numpy().view(np.uint16), *mat), what=f"M{M} N{N} K{K}")
        for ref, o in zip(alone, outs):
            for y in o:
                assert torch.equal(y, ref)


@pytest.mark.parametrize("D,H,KVH,M", [(256, 24, 4, 5), (128, 16, 2, 8), (64, 8, 8, 40), (256, 24, 4, 300)])
def test_prefill_partials_are_sized_once(torch_dev, D, H, KVH, M):
    """A split prefill's partials do not grow with the cache (growing waits for
    the stream), nor with the streams that the runtime is used on."""
    import torch
    rng = np.random.default_rng(D + M)
    with tuned() as rt:
        cache = rt.create_q8_kv_state(KVH, D, 9000)
        cache.reserve(9000)
        f32 = [to_dev(rng.standard_normal((4200, KVH, D)).astype(np.float32), torch_dev) for _ in range(2)]
        q = to_dev(synth.bf16_normal(rng, (4200, H, D)), torch_dev)
        o = empty_bf16((4200, H, D), torch_dev)
        rt.gqa_attention_q8_prefill(cache, q, None, *f32, H, 1100, o)
        streams = [torch.cuda.Stream() for _ in range(5)]
        free = []
        for i in range(20):
            rt.set_stream(streams[i % 5])
            rt.gqa_attention_q8_prefill(cache, q, None, *f32, H, M, o)
            torch.cuda.synchronize()
            free.append(torch.cuda.mem_get_info()[0])
            rt.gqa_attention_q8_prefill(cache, q, None, *f32, H, 90, o)  # a longer cache
        torch.cuda.synchronize()
        rt.set_stream(torch.cuda.current_stream())
        assert len(set(free[5:])) == 1  # a stream's first launch takes memory of its own


@pytest.mark.parametrize("M,specs,K", [
    (12, [(10000, False)], 1536),              # medium matrices
    (9, [(3200, False)], 9216),                # long K
    (16, [(3000, False), (4000, True)], 1536), # a set
])
def test_few_rows_capture_without_a_warm_call(torch_dev, M, specs, K):
    """A fresh runtime's first projection of a few rows may be a captured one:
    where the kernel's K slices have no workspace another kernel takes the call.
    Replayed with eager work in between."""
    import torch
    rng = np.random.default_rng(M)
    with tuned() as rt, tuned() as eager:
        mats = [synth.q4_matrix(rng, n, K) for n, _ in specs]
        ups = [synth.q4_matrix(rng, n, K) if pair else None for n, pair in specs]
        jobs, upj = [_job(m, torch_dev) for m in mats], [_job(u, torch_dev) if u else None for u in ups]
        x = to_dev(synth.bf16_normal(rng, (M, K)), torch_dev)
        outs = [empty_bf16((M, n), torch_dev) for n, _ in specs]
        refs = [empty_bf16((M, n), torch_dev) for n, _ in specs]
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            rt.set_stream(torch.cuda.current_stream())
            rt.q4_project_set(jobs, upj, x, K, M, outs)
        rt.set_stream(torch.cuda.current_stream())
        for i in range(3):
            xb = synth.bf16_normal(rng, (M, K))
            x.copy_(to_dev(xb, torch_dev))
            eager.q4_project_set(jobs, upj, x, K, M, refs)
            graph.replay()
            torch.cuda.synchronize()
            for o, r, m, u in zip(outs, refs, mats, ups):
                ref = oracle.q4_project(xb, *m)
                if u is not None:
                    ref = oracle.swiglu(ref, oracle.q4_project(xb, *u))
                assert_bf16_close(bf16_dev_to_f32(o), ref, what=f"replay {i}")
                assert_bf16_close(bf16_dev_to_f32(r), ref, what=f"eager {i}")
                o.fill_(-1)


@pytest.mark.parametrize("M,N,K,env", [(40, 700, 4096, {"QM38_Q4_ROWS_SLICES": 4}), (300, 300, 2048, {"QM38_GEMM_SPLITS": 3}),
                                       (3, 512, 9216, {})])
def test_capture_after_a_warm_call_elsewhere(torch_dev, M, N, K, env):
    """A call warmed on one stream may be captured on another (the stream that
    is left has used a workspace), and the runtime goes on after it: every
    replay, and eager calls between them, equal the call before the capture."""
    import torch
    rng = np.random.default_rng(M)
    with tuned(**env) as rt:
        mat = synth.q4_matrix(rng, N, K)
        job = _job(mat, torch_dev)
        x = to_dev(synth.bf16_normal(rng, (M, K)), torch_dev)
        want, got, eager = (empty_bf16((M, N), torch_dev) for _ in range(3))
        rt.q4_project([job], x, K, M, [want])
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            rt.set_stream(torch.cuda.current_stream())
            rt.q4_project([job], x, K, M, [got])
        rt.set_stream(torch.cuda.current_stream())
        for _ in range(3):
            got.fill_(-1)
            eager.fill_(-1)
            graph.replay()
            rt.q4_project([job], x, K, M, [eager])
            torch.cuda.synchronize()
            assert torch.equal(got, want) and torch.equal(eager, want)
    assert_bf16_close(bf16_dev_to_f32(want), oracle.q4_project(x.cpu().numpy().view(np.uint16), *mat))
