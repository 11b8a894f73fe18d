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
