"""The fused RMSNorm + GEMM of bf16 rows: every GEMM kernel's epilogue converts its fp16 result to bf16, so
the call equals, bit for bit, the fp16 GEMM of the normalised rows converted afterwards.  The row norm at the
edges of its register form (2048 elements a column, up to 8 columns) against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import awq_oracle as O
from oracle.gen import make_awq_problem

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("M,K,N,G,kw", [
    (1, 1024, 512, 128, {}), (1, 1024, 512, 128, {"decode_layout": "stream"}), (8, 4096, 1024, 128, {"decode_layout": "stream"}),
    (16, 1024, 264, 64, {}), (24, 512, 136, 32, {"decode_layout": "narrow"}), (40, 2048, 264, 128, {}), (100, 4096, 520, 128, {}),
    (300, 256, 65536, 128, {}), (64, 512, 264, 128, {"decode_stream": False}), (130, 512, 264, 128, {"decode_stream": False})])
def test_bf16_rows_equal_converted_fp16_result(M, K, N, G, kw):
    from litevllm_amd import ops
    print(f"rmsnorm bf16 M={M} K={K} N={N} G={G} {kw}", flush=True)
    t = {k: torch.from_numpy(v).to(DEV) for k, v in make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + N).items()
         if isinstance(v, np.ndarray)}
    x = t["x"].to(torch.bfloat16)
    nw = (1 + 0.3 * torch.randn(K, generator=torch.Generator().manual_seed(K))).to(torch.bfloat16).to(DEV)
    w = (t["qweight"], t["scales"], t["qzeros"], G)
    y = ops.rmsnorm_gemm(x, nw, 1e-6, *w, layout="autoawq", **kw)
    # the bf16 call's weight copy: the layout rule sees bf16 activations
    if not kw and M <= 32:
        kw = {"decode_layout": "narrow" if ops._narrow_fits(M, N, K, 0, True) else "stream"}
    xn = ops.rmsnorm(x, nw, 1e-6)
    assert torch.equal(y, ops.gemm(xn, *w, layout="autoawq", **kw).to(torch.bfloat16))


@pytest.mark.parametrize("K", [8, 2048, 2056, 8192, 8200, 16384, 16392])
def test_rows_at_column_edges(K):
    from litevllm_amd import ops
    g = torch.Generator().manual_seed(K)
    x, nw = torch.randn(3, K, generator=g).half(), (1 + 0.3 * torch.randn(K, generator=g)).half()
    got = ops.rmsnorm(x.to(DEV), nw.to(DEV), 1e-6).cpu().numpy()
    assert np.array_equal(got.view(np.uint16), O.rmsnorm_rows(x.float().numpy(), nw.float().numpy(), 1e-6).view(np.uint16))


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,off", [(1, 0), (1, 2048), (8, 0)])
def test_output_over_the_input_rows(M, off, dt):
    """An output that lies over x, wholly or from its middle on: the values of a call whose output lies apart (the
    narrow kernel's blocks read the row while others store, so such a call normalises in a launch of its own)."""
    from litevllm_amd import ops
    K = N = 4096
    print(f"rmsnorm in place M={M} off={off} {dt}", flush=True)
    p = make_awq_problem(M=M, K=K, N=N, group_size=128, seed=5)
    w = tuple(torch.from_numpy(p[k]).to(DEV) for k in ("qweight", "scales", "qzeros")) + (128,)
    nw = (1 + 0.3 * torch.randn(K, generator=torch.Generator().manual_seed(K))).half().to(DEV)
    buf = torch.zeros(M * K + off, dtype=dt, device=DEV)
    x, out = buf[: M * K].view(M, K), buf[off:].view(M, N)
    x.copy_(torch.from_numpy(p["x"]))
    want = ops.rmsnorm_gemm(x, nw, 1e-6, *w, layout="autoawq", decode_layout="narrow")
    assert ops.rmsnorm_gemm(x, nw, 1e-6, *w, layout="autoawq", decode_layout="narrow", out=out).data_ptr() == out.data_ptr()
    # the narrow kernel's own norm and the row-norm launch give the same rows
    assert torch.equal(out, want)


@pytest.mark.parametrize("M", [3, 100])
def test_bf16_call_needs_no_room_for_its_product(M):
    """The workspace of the fp16 call serves the bf16 one, to the byte."""
    from litevllm_amd import _lib as L
    from litevllm_amd import ops
    K, N, G = 512, 264, 128
    t = {k: torch.from_numpy(v).to(DEV) for k, v in make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M).items()
         if isinstance(v, np.ndarray)}
    x, nw = t["x"].to(torch.bfloat16), torch.ones(K, dtype=torch.float16, device=DEV)
    lib, qk = L.load(), ops.pack_decode_stream(t["qweight"])
    need = int(lib.awq_w4a16_rmsnorm_gemm_workspace_bytes(M, N, K, G, 0, L.LAYOUT_DECODE_STREAM, L.DTYPE_F16))
    ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    call = lambda nbytes: lib.awq_w4a16_rmsnorm_gemm(
        x.data_ptr(), K, nw.data_ptr(), 1e-6, qk.data_ptr(), t["scales"].data_ptr(), t["qzeros"].data_ptr(), out.data_ptr(), N, M,
        N, K, G, 0, L.LAYOUT_DECODE_STREAM, L.DTYPE_BF16, L.DTYPE_F16, L.DTYPE_F16, ws.data_ptr(), nbytes,
        int(torch.cuda.current_stream().cuda_stream))
    assert call(need - 1) == L.ERR_WORKSPACE
    assert call(need) == 0
    assert torch.equal(out, ops.rmsnorm_gemm(x, nw, 1e-6, t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq",
                                             decode_layout="stream" if M <= 32 else None))


def test_bf16_rows_past_a_grid_dimension():
    """More rows than a grid's y and z dimensions hold, as fp16 calls always took them."""
    from litevllm_amd import ops
    M, K, N, G = 65536 + 40, 64, 8, 32
    t = {k: torch.from_numpy(v).to(DEV) for k, v in make_awq_problem(M=8, K=K, N=N, group_size=G, seed=1).items()
         if isinstance(v, np.ndarray)}
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).to(DEV)
    nw = torch.ones(K, dtype=torch.float16, device=DEV)
    w = (t["qweight"], t["scales"], t["qzeros"], G)
    y = ops.rmsnorm_gemm(x, nw, 1e-6, *w, layout="autoawq")
    assert torch.equal(y, ops.gemm(ops.rmsnorm(x, nw, 1e-6), *w, layout="autoawq").to(torch.bfloat16))


@pytest.mark.parametrize("N", [8192, 8200, 10248])
def test_one_bf16_row_on_either_side_of_two_tiles_per_cu(N):
    """Up to two 16-column tiles per CU the narrow kernel normalises the row itself; the same bits as the row-norm
    launch and the narrow GEMM on its row."""
    test_bf16_rows_equal_converted_fp16_result(1, 512, N, 128, {"decode_layout": "narrow"})
