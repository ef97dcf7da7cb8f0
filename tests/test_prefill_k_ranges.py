"""K ranges of the prefill stream kernel (long K, tiles that cover at most a third of the CUs): range edges inside a
group's stage pair and a K that ends on half a stage, strides, bias, the converting epilogue, replays of a capture
and a workspace that does not hold the ranges.  Every output within one ulp (of max(|y|, 1)) of the float64
product with the weights rounded once."""
import ctypes

import numpy as np
import pytest
import torch

from litevllm_amd import _lib as L
from oracle import awq_oracle as O
from oracle.gen import make_awq_problem

DEV = torch.device("cuda:0")
STREAM = L.LAYOUT_DECODE_STREAM


def _route(M, N, K, G, ws=None, split_k=0):
    lib, tile, ranges = L.load(), ctypes.c_int32(), ctypes.c_int32()
    if ws is None:
        ws = int(lib.awq_w4a16_gemm_workspace_bytes(M, N, K, G, split_k, STREAM))
    return lib.awq_w4a16_gemm_kernel(M, N, K, G, split_k, STREAM, ws, tile, ranges), ranges.value


def test_calls_that_take_ranges():
    """Where the middle-batch kernel measured slower; never on a forced split or a workspace without room."""
    for M, N, K, G in ((256, 16896, 12288, 128), (512, 8192, 14336, 32), (1024, 4096, 12288, 32), (1931, 2152, 8128, 32)):
        kernel, ranges = _route(M, N, K, G)
        assert kernel == L.KERNEL_PREFILL_STREAM and ranges >= 3, (M, N, K, G)
        assert _route(M, N, K, G, split_k=1)[1] <= 1 and _route(M, N, K, G, split_k=3)[1] <= 1
        assert _route(M, N, K, G, ws=65536 + 4 * ranges * M * N - 1) == (L.KERNEL_MID, 1)
    for M, N, K, G in ((256, 4096, 12288, 128), (1000, 4096, 4096, 128), (64, 16896, 12288, 32)):
        assert _route(M, N, K, G)[0] == L.KERNEL_MID


def _problem(M, K, N, G, dt):
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + N, with_bias=True)
    t = {k: torch.from_numpy(p[k]).to(DEV) for k in ("qweight", "scales", "qzeros", "bias")}
    x = torch.from_numpy(p["x"]).to(dt)
    half = "float16" if dt == torch.float16 else "bfloat16"
    w = O.dequant_awq(p["qweight"], p["scales"], p["qzeros"], G, out_dtype=half)
    w = O.bf16_bits_to_f32(w) if half == "bfloat16" else w
    return t, x, x.double().numpy() @ w.astype(np.float64) + p["bias"].astype(np.float64)


def _ulps(y, ye, dt):
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - (10 if dt == torch.float16 else 7))
    return (np.abs(y.double().cpu().numpy() - ye) / ulp).max()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,G", [(129, 6176, 16632, 32), (200, 6208, 16640, 64), (256, 6144, 16776, 128), (1931, 6176, 1800, 32)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_ranges_vs_oracle(M, K, N, G, dt):
    from litevllm_amd import ops
    kernel, ranges = _route(M, N, K, G)
    print(f"prefill ranges M={M} K={K} N={N} G={G} {dt}: {ranges}", flush=True)
    assert kernel == L.KERNEL_PREFILL_STREAM and ranges >= 3
    t, x, ye = _problem(M, K, N, G, dt)
    a = (x.to(DEV), t["qweight"], t["scales"], t["qzeros"], G)
    y = ops.gemm(*a, bias=t["bias"], layout="autoawq")
    assert torch.equal(y, ops.gemm(*a, bias=t["bias"], layout="autoawq"))
    assert _ulps(y, ye, dt) <= 1.0


@pytest.mark.gpu
def test_ranges_strides_capture_conversion_and_workspace():
    from litevllm_amd import ops
    M, K, N, G = 1931, 6176, 1800, 32
    print("prefill ranges: strides, capture, conversion, workspace", flush=True)
    t, x, ye = _problem(M, K, N, G, torch.float16)
    w = (t["qweight"], t["scales"], t["qzeros"], G)
    x = x.to(DEV)
    y = ops.gemm(x, *w, bias=t["bias"], layout="autoawq")
    xb, ob = torch.zeros((M, K + 64), dtype=x.dtype, device=DEV), torch.full((M, N + 64), 7.0, dtype=x.dtype, device=DEV)
    xb[:, :K] = x
    ops.gemm(xb[:, :K], *w, bias=t["bias"], layout="autoawq", out=ob[:, :N])
    assert torch.equal(ob[:, :N], y) and bool((ob[:, N:] == 7.0).all())
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        yg = ops.gemm(x, *w, bias=t["bias"], layout="autoawq")
    for _ in range(3):
        yg.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(yg, ops.gemm(x, *w, bias=t["bias"], layout="autoawq"))
    nw = torch.ones(K, dtype=torch.float16, device=DEV)
    xn = ops.rmsnorm(x.to(torch.bfloat16), nw, 1e-6)
    assert torch.equal(ops.rmsnorm_gemm(x.to(torch.bfloat16), nw, 1e-6, *w, layout="autoawq"),
                       ops.gemm(xn, *w, layout="autoawq").to(torch.bfloat16))
    lib, qk = L.load(), ops.pack_decode_stream(t["qweight"])
    out = torch.empty_like(y)
    ws = torch.zeros(65536, dtype=torch.uint8, device=DEV)
    rc = lib.awq_w4a16_gemm(x.data_ptr(), K, qk.data_ptr(), t["scales"].data_ptr(), t["qzeros"].data_ptr(), t["bias"].data_ptr(),
                            out.data_ptr(), N, M, N, K, G, 0, STREAM, L.DTYPE_F16, L.DTYPE_F16, L.DTYPE_F16, ws.data_ptr(), 65536,
                            int(torch.cuda.current_stream().cuda_stream))
    assert rc == 0 and _ulps(out, ye, torch.float16) <= 1.0
    assert not bool(ws.any())  # the counters
