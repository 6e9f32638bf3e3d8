"""mxs_nf4_linear_fwd_noalloc's one call before a capture: of a few tokens (a kernel that needs no
partial sums), it still looks up the library's device array for a captured call that splits."""

import ctypes
import shutil

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_a_few_token_call_prepares_a_captured_split_plan(cuda, tmp_path):
    from mindxsoup_amd import _lib, kernels
    from mindxsoup_amd.quant import quantize_4bit

    print("case noalloc lookup by a few-token call", flush=True)
    shutil.copy(_lib.LIB_PATH, tmp_path / "fresh.so")  # a library that has looked nothing up yet
    fn = ctypes.CDLL(str(tmp_path / "fresh.so")).mxs_nf4_linear_fwd_noalloc
    fn.argtypes = _lib._SIGNATURES["mxs_nf4_linear_fwd_noalloc"]
    n, k = 1536, 8960
    packed, st = quantize_4bit((torch.randn((n, k), device=cuda) * 0.02).half())
    assert kernels.gemm_workspace_bytes(300, n, k) > 0  # the captured plan splits

    def call(x, y):
        return fn(_lib.ptr(x), x.shape[0], k, n, *kernels._nf4_args(packed, st), None, None, None,
                  0, _lib.ptr(y), -1, 1, _lib.stream_of(x.device))

    few, many = (torch.randn((m, k), device=cuda).half() for m in (4, 300))
    y4, y = (torch.empty((m, n), dtype=torch.float16, device=cuda) for m in (4, 300))
    assert call(few, y4) == 0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rc = call(many, y)
    assert rc == 0
    want = kernels.nf4_linear_fwd_noalloc(many, packed, st, torch.empty_like(y))
    for rep in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), rep
        assert call(few, y4) == 0  # eager work between the replays
    assert torch.equal(y4, kernels.nf4_linear_fwd(few, packed, st))
    del graph
